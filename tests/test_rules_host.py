"""CPU checks of the rules that choose a kernel (yrt-pet_amd/csrc/
yrtmi_tiles.hpp), compiled for the host with tests/hostwalk/."""
import ctypes as C
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def hw(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("rules") / "librules.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC",
                    "-I", os.path.join(HERE, "hostwalk"),
                    "-I", os.path.join(REPO, "yrt-pet_amd", "csrc"),
                    os.path.join(HERE, "hostwalk", "rules_host.cpp"), "-o", out],
                   check=True, capture_output=True)
    lib = C.CDLL(out)
    lib.hw_use_bricks.argtypes = [C.c_int64] * 4
    return lib


@pytest.mark.parametrize("dims,frames,want", [
    ((200, 200, 128), 1, True),
    ((96, 96, 48), 1, False),
    # 2^31 voxels and more with the bricks' padding, fewer without
    ((1290, 1290, 1290), 1, False),
    ((1 << 28, 1, 1), 1, False),
    ((1, 1, 1 << 27), 1, False),
    ((1, 1, (1 << 27) - 2), 1, True),
])
def test_bricks_are_indexed_in_32_bits(hw, dims, frames, want):
    assert bool(hw.hw_use_bricks(*dims, frames)) == want
