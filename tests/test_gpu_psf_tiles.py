"""The tiled image-space PSF at the edges of its tiles (64 x 32 voxels, 8
outputs a thread, columns of 16 planes) and of its kernels (1 to 63 taps, one
wrap), on the GPU: bitwise the oracle's sums, infinities and NaN reaching the
voxels whose sums hold them and no others."""
import numpy as np
import pytest
import torch

import oracle as O
import yrtmi

pytestmark = pytest.mark.gpu

CASES = [
    # (nz, ny, nx), taps (x, y, z), frames
    ((16, 32, 64), (3, 3, 3), 1),
    ((17, 33, 65), (1, 1, 1), 2),
    ((15, 31, 63), (15, 13, 11), 1),
    ((3, 40, 129), (7, 61, 5), 1),
    ((40, 40, 40), (63, 63, 63), 1),
    ((5, 2, 1), (1, 3, 9), 3),
    ((48, 7, 200), (9, 9, 31), 1),
    # more than 65535 tiles along y, and columns along z
    ((1, 2_200_000, 2), (3, 5, 1), 1),
    ((1_100_000, 2, 1), (1, 3, 5), 1),
]


@pytest.mark.parametrize("shape,ks,nt", CASES, ids=str)
def test_psf_tiles_bitwise(gpu, shape, ks, nt):
    nz, ny, nx = shape
    im = yrtmi.ImageParams(nx, ny, nz, 2.0, 2.5, 3.0, nt=nt)
    ctx = yrtmi.Context(yrtmi.Scanner("t", 96.0, 4.0, 4.0, 10.0, 180.0, 128, 24))
    rng = np.random.default_rng(sum(shape))
    x = rng.random((nt, nz, ny, nx), dtype=np.float32)
    x[:, nz // 2, ny // 2, nx // 2] = np.inf
    x[-1, 0, 0, 0] = np.nan
    k = [rng.random(n).astype(np.float32) for n in ks]
    xg = torch.from_numpy(x).to(gpu)
    out, tmp = torch.empty_like(xg), torch.empty_like(xg)
    for transpose in (False, True):
        ctx.psf(im, xg, out, tmp, *k, transpose=transpose)
        ctx.synchronize()
        with np.errstate(invalid="ignore"):
            want = O.psf_convolve(x, *k, transpose=transpose)
        np.testing.assert_array_equal(out.cpu().numpy(), want)
