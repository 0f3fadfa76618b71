"""CPU checks of the rules that choose a kernel (yrt-pet_amd/csrc/
yrtmi_tiles.hpp), compiled for the host with tests/hostwalk/."""
import ctypes as C
import os
import subprocess

import numpy as np
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
    lib.hw_use_bricks.argtypes = [C.c_int64] * 4 + [C.c_int] * 2 + [C.c_int64]
    lib.hw_dd_records.argtypes = [C.c_int64] * 3 + [C.c_float] * 6
    lib.hw_dd_records.restype = C.c_int64
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
    assert bool(hw.hw_use_bricks(*dims, frames, 0, 1, 1000)) == want


@pytest.mark.parametrize("dims,frames,dd,rays,n,want", [
    ((128, 128, 128), 1, 0, 4, 1000, True), ((128, 128, 127), 1, 0, 4, 1 << 30, False),
    ((128, 128, 64), 16, 0, 6, 1 << 30, False),  # a frame at a time
    ((128, 128, 128), 1, 0, 1, 1, True), ((128, 128, 64), 2, 0, 3, 1, True),
    ((64, 64, 64), 1, 0, 1, 1 << 19, True), ((64, 64, 64), 1, 0, 1, (1 << 19) - 1, False),
    ((64, 64, 64), 1, 0, 2, 1 << 18, True), ((64, 64, 63), 1, 0, 3, 1 << 30, False),
    ((128, 128, 64), 1, 1, 1, 1 << 17, True), ((128, 128, 64), 1, 1, 1, (1 << 17) - 1, False),
    ((128, 128, 63), 1, 1, 1, 1 << 30, False), ((96, 96, 48), 16, 1, 1, 1, True),
])
def test_bricks_by_rays_and_length(hw, dims, frames, dd, rays, n, want):
    assert bool(hw.hw_use_bricks(*dims, frames, dd, rays, n)) == want


@pytest.mark.gpu
@pytest.mark.parametrize("oblique", [False, True])
@pytest.mark.parametrize("dims,crystal_z,crystal_t,psf", [
    ((64, 60, 30, 4.0, 4.5, 2.0), 4.0, 4.0, 0.0),
    ((32, 32, 512, 4.0, 4.0, 0.25), 60.0, 4.0, 0.0),   # 30 tiles high
    ((200, 200, 64, 1.0, 1.0, 2.0), 4.0, 80.0, 0.0),   # 3 tiles wide
    ((160, 160, 64, 1.0, 1.0, 0.5), 4.0, 4.0, 30.0),   # wide by its PSF
    ((32, 32, 256, 8.0, 8.0, 1.0), 4.0, 4.0, 0.0),     # tall
    ((160, 40, 16, 1.0, 4.0, 4.0), 4.0, 4.0, 0.0),
], ids=str)
def test_room_for_dd_records(hw, gpu, dims, crystal_z, crystal_t, psf, oblique):
    """The records of DD plans (random LORs, and LORs from the first ring to
    the last) within the room per LOR."""
    import torch
    import yrtmi
    rings = 64 if crystal_z < 10 else 4
    dpr = 128 if crystal_t < 8 else 12
    sc = yrtmi.Scanner("t", crystal_z * rings, crystal_z, crystal_t, 10.0, 180.0, dpr, rings)
    im = yrtmi.ImageParams(*dims)
    n = 20_000
    rng = np.random.default_rng(3)
    d = [rng.integers(0, dpr, n) for _ in range(2)]
    z = [np.zeros(n, np.int64), np.full(n, rings - 1)] if oblique \
        else [rng.integers(0, rings, n) for _ in range(2)]
    t = lambda k: torch.from_numpy((d[k] + dpr * z[k]).astype(np.int32)).to(gpu)
    pp = yrtmi.ProjectorParams(sc, projectorType="DD")
    ext = 0.0
    if psf:
        k, ks = 31, psf / 16
        pp.psf_kernels = np.exp(-0.5 * ((np.arange(k) - 15) / 5.0) ** 2)[None].astype(np.float32)
        pp.psf_s_step, pp.psf_k_spacing = 100.0, ks
        ext = 16 * ks
    ctx = yrtmi.Context(sc, histogram=False)
    p = ctx.projector(pp)
    records = ctx.plan(p, im, yrtmi.LorSet.pairs(t(0), t(1)), tile_shape=3).info()["records"]
    room = hw.hw_dd_records(*dims, crystal_t, crystal_z, ext)
    print(f"{records / n:.1f} records a LOR, room for {room}", flush=True)
    assert 0 < records <= room * n
