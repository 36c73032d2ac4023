"""CPU test: the tree builder refuses a group that one wave cannot scan."""
import shutil
import subprocess
from pathlib import Path

import pytest

from radeonrays_sdk_amd import _build


@pytest.mark.parametrize("group,compiles", [(63, True), (64, False)])
def test_group_size_is_checked(tmp_path, group, compiles):
    """Lane k writes group_first[k], and group_first[runs] is read as the number of entries: with 64 runs no lane
    would have written it."""
    csrc = tmp_path / "csrc"
    shutil.copytree(_build.CSRC, csrc)
    header = csrc / "tree_device.h"
    text = header.read_text()
    assert "kTreeGroup = 48;" in text
    header.write_text(text.replace("kTreeGroup = 48;", f"kTreeGroup = {group};"))
    (csrc / "probe.hip").write_text('#include "tree_device.h"\n')
    proc = subprocess.run([_build.HIPCC, *_build.DEVICE_FLAGS, f"-I{_build.INCLUDE}", f"-I{csrc}", "-fsyntax-only",
                           str(csrc / "probe.hip")], capture_output=True, text=True)
    assert (proc.returncode == 0) == compiles, proc.stderr
    assert compiles or "static assertion failed" in proc.stderr
