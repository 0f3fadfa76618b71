"""CPU check of the plan's tile pieces (sidPieces, yrt-pet_amd/csrc/
yrtmi_rays.hpp): cutting a ray tile by tile gives the pieces that its walk
passes through.

Voxel sizes that are short binary fractions: the same pieces, entered at the
same voxels and alphas.  Others: the walk accumulates its plane positions,
each addition rounding within half an ulp of the position (2^-17 mm below
256 mm), the pieces' planes are start + k v: at most 256 * 2^-17 mm apart,
8e-6 of a 250 mm and longer ray, so entry alphas agree within 1e-5 and only
pieces cut at a corner that the ray passes that closely may differ.  A free
line does so for about 1 piece in 1000 or fewer; the lines at 45 degrees
between crystals of the ring, mirror lines of a grid with vx = vy, run through
voxel corners all along and may all differ."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def hw(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("pieces") / "libpieces.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC",
                    "-I", os.path.join(HERE, "hostwalk"),
                    "-I", os.path.join(REPO, "yrt-pet_amd", "csrc"),
                    os.path.join(HERE, "hostwalk", "pieces_host.cpp"), "-o", out],
                   check=True, capture_output=True)
    lib = C.CDLL(out)
    P = C.c_void_p
    lib.hw_pieces.restype = None
    lib.hw_pieces.argtypes = [P, C.c_int64, P, P, C.c_int, P, P, P, P, P]
    return lib


def lines(n, im, seed):
    """Chords of a ring of 420 mm radius: free ones, crystals of a 512 ring,
    lines on and between voxel planes, lines flat in x, in y and in z."""
    rng = np.random.default_rng(seed)
    nx, ny, nz, vx, vy, vz = im
    a, b = rng.uniform(0, 2 * np.pi, (2, n))
    i = np.arange(n)
    q = 2 * np.pi / 512
    a, b = (np.where(i % 3 == 0, np.floor(t / q) * q, t) for t in (a, b))
    z1, z2 = rng.uniform(-0.5, 0.5, (2, n)) * nz * vz
    z1 = np.where(i % 5 == 0, np.floor(z1 / vz) * vz, z1)
    z2 = np.where((i % 5 == 0) | (i % 7 == 0), z1, z2)
    p1 = np.stack([420 * np.cos(a), 420 * np.sin(a), z1], 1).astype(np.float32)
    p2 = np.stack([420 * np.cos(b), 420 * np.sin(b), z2], 1).astype(np.float32)
    p1[i % 11 == 0, 0] = p2[i % 11 == 0, 0] = vx * np.floor(rng.uniform(-9, 9))
    p1[i % 13 == 0, 1] = p2[i % 13 == 0, 1] = vy * (np.floor(rng.uniform(-9, 9)) + 0.5)
    tof = rng.uniform(-400, 400, n).astype(np.float32)
    return np.ascontiguousarray(p1), np.ascontiguousarray(p2), tof


@pytest.mark.parametrize("tile", [(5, 5, 3), (4, 4, 4), (3, 2, 1)], ids=str)
@pytest.mark.parametrize("im,exact", [((70, 66, 40, 4.0, 4.5, 2.25), True),
                                      ((200, 33, 128, 2.0, 2.0, 2.0), True),
                                      ((61, 57, 35, 5.1, 5.3, 2.7), False),
                                      ((256, 256, 128, 1.6, 1.6, 1.6), False)], ids=str)
@pytest.mark.parametrize("tof", [0, 1])
def test_pieces_are_the_walks(hw, im, exact, tile, tof):
    check(hw, im, exact, tile, tof, lines(12000, im, 7))


@pytest.mark.parametrize("tile", [(5, 5, 3), (3, 2, 1)], ids=str)
@pytest.mark.parametrize("tof", [0, 1])
def test_pieces_of_voxels_below_a_millionth_of_the_scanner(hw, tile, tof):
    """Where a position may be planes off (sidCoarse): voxels of 2^-11 mm (short
    binary fractions: the same pieces) under lines of 840 mm through them."""
    im = (70, 66, 40, 2.0 ** -11, 2.0 ** -11, 2.0 ** -11)
    rng = np.random.default_rng(3)
    n = 12000
    at = rng.uniform(-0.5, 0.5, (n, 3)) * np.array(im[:3]) * im[3]
    a, slope = rng.uniform(0, 2 * np.pi, n), rng.uniform(-1, 1, n)
    slope[::4] = 0.0
    d = 420 * np.stack([np.cos(a), np.sin(a), slope], 1)
    p1, p2 = ((at + q * d).astype(np.float32) for q in (1, -1))
    check(hw, im, True, tile, tof, (np.ascontiguousarray(p1), np.ascontiguousarray(p2),
                                    rng.uniform(-400, 400, n).astype(np.float32)))


def check(hw, im, exact, tile, tof, rays):
    p1, p2, tv = rays
    n = len(p1)
    f = np.float32
    L = [f(im[i]) * f(im[3 + i]) for i in range(3)]
    imp = np.array([*im, *L, max(L[:2]) / 2 - max(im[3:5]) / 1000], f)
    tofc = np.array([16.0, 80.0, 0.02], f)
    out = np.zeros(6, np.int64)
    da = np.zeros(1, f)
    p = lambda a: a.ctypes.data_as(C.c_void_p)
    hw.hw_pieces(p(imp), n, p(p1), p(p2), tof, p(tofc), p(tv), p(np.array(tile, np.int32)),
                 p(out), p(da))
    rays, pieces, counts, voxels, outside, short = (int(v) for v in out)
    print(f"{im} tile 2^{tile} tof {tof}: {rays} rays, {pieces} pieces; other count {counts}, "
          f"other voxel {voxels}, alphas within {da[0]:.1e}")
    assert rays > 1000 and pieces > rays
    assert outside == 0 and short <= voxels
    if exact:
        assert counts == 0 and voxels == 0 and da[0] == 0.0
    else:
        d = np.abs(p2.astype(np.float64) - p1)
        diagonal = int((np.abs(d[:, 0] - d[:, 1]) < 1e-3).sum()) if im[3] == im[4] else 0
        assert counts <= diagonal + rays / 1000
        assert voxels <= pieces / 1000 and da[0] <= 1e-5
