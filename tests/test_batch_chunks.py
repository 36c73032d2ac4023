"""CPU tests of the chunk layout of a batched build or update (csrc/batch.h),
compiled as it is."""
import ctypes
import subprocess

import pytest

from radeonrays_sdk_amd import _build

WINDOW = 8  # chunks of 64 leaves in a workgroup of the tree kernel

SHIM = """
#include "batch.h"
extern "C" __attribute__((visibility("default"))) unsigned layout(unsigned before, unsigned tris, int update) {
    return rr::BatchFirstChunk(before, rr::RefitChunks(tris), update != 0);
}
extern "C" __attribute__((visibility("default"))) unsigned chunks(unsigned tris) { return rr::RefitChunks(tris); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("chunks")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run([_build.HIPCC, "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{_build.CSRC}", f"-I{_build.INCLUDE}",
                    str(d / "shim.cpp"), "-o", str(d / "chunks.so")], check=True, capture_output=True)
    return ctypes.CDLL(str(d / "chunks.so"))


@pytest.mark.parametrize("sizes", [(16384, 3000, 1025, 1024, 513, 512, 449, 448, 300, 64, 1), (65536, 16385, 600) * 9,
                                   (330,) * 50, (0, 1, 0, 0)])
def test_updates_pack_chunks_and_builds_align_them(lib, sizes):
    packed = aligned = 0
    for n in sorted(sizes, reverse=True):
        c = lib.chunks(n)
        first = lib.layout(packed, n, 1)
        assert first == packed
        packed = first + c
        first = lib.layout(aligned, n, 0)
        assert aligned <= first < aligned + WINDOW
        if c:
            assert first % WINDOW == 0 or first % WINDOW + c <= WINDOW
        aligned = first + c
    assert packed == sum(-(-n // 64) for n in sizes)
