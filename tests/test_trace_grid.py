"""CPU tests of the rules that size a query's grid and its waves' pieces
(csrc/trace_grid.h), compiled as they are."""
import ctypes
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "radeonrays_sdk_amd" / "csrc"
CUS = 256

SHIM = """
#include "trace_grid.h"
extern "C" unsigned piece(unsigned long long n, unsigned blocks, unsigned tuned) { return rr::PieceRays(n, blocks, tuned); }
"""


@pytest.fixture(scope="module")
def grid(tmp_path_factory):
    d = tmp_path_factory.mktemp("grid")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{CSRC}", str(d / "shim.cpp"), "-o",
                    str(d / "grid.so")], check=True)
    lib = ctypes.CDLL(str(d / "grid.so"))
    lib.piece.argtypes = [ctypes.c_uint64, ctypes.c_uint32, ctypes.c_uint32]
    lib.piece.restype = ctypes.c_uint32
    return lib


@pytest.mark.parametrize("blocks", [1, 769, 4 * CUS, 7 * CUS])
@pytest.mark.parametrize("tuned", [32, 64, 128])
def test_piece_leaves_half_a_share_to_balance(grid, blocks, tuned):
    """No piece is more than half an even share, from a share of 128 rays on; smaller shares go in pieces of 64, and
    every wave has a piece."""
    waves = 4 * blocks
    for share in (1, 31, 32, 33, 63, 64, 65, 96, 127, 128, 129, 150, 191, 192, 193, 255, 256, 257, 1000, 4096):
        for n in (share * waves - 1, share * waves, share * waves + 1):
            piece = grid.piece(n, blocks, tuned)
            assert piece in (32, 64, 96, 128) and piece <= tuned, (share, n)
            if n >= 128 * waves:
                assert 2 * piece * waves <= n, (share, n)
                assert piece == tuned or 2 * (piece + 32) * waves > n, (share, n)  # and no smaller than it has to be
            elif n > 32 * waves:
                assert piece == min(tuned, 64), (share, n)
            else:
                assert piece == 32, (share, n)
