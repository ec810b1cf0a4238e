"""The prefixes that a level's popcount scan stores for bitmap tiles without occupied cells, against the words
that the neighbourhood filters read (tests/prefix_model.cpp): on the CPU, with the arithmetic of the kernels
(csrc/cell_order.h)."""
import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = shutil.which("g++") or shutil.which("clang++")


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("prefix") / "model")
    subprocess.run([CXX, "-std=c++17", "-O2", "-I", os.path.join(REPO, "octree-cuda_amd", "csrc"),
                    os.path.join(REPO, "tests", "prefix_model.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.skipif(CXX is None, reason="no C++ compiler")
@pytest.mark.parametrize("tile", [2048, 64])  # the scan's tiles, and small ones with many more ends inside rows
def test_windows_read_prefixes_that_are_written(model, tile):
    r = subprocess.run([model, str(tile)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
    assert int(r.stdout.split()[-1]) > 0, "no window starts in an empty tile: the case is not met"
