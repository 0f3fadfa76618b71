"""Plans of few records (chunks of one record per thread up to 4096) and the
fixed-point scale over value counts around a workgroup, on the GPU: planned
against direct backprojection.

Bars: the tile sum is exact in fixed point, the direct one is summed in FP32
(at most a few thousand terms a voxel, each rounding 6e-8 of the sum): 2e-6
relative L2 with dyadic voxels."""
import numpy as np
import pytest
import torch

import yrtmi
from helpers import rel_l2
from yrtmi import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [1.0, 1e-30, 3e20])
@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 4095, 9000, 70001])
def test_planned_back_small(gpu, n, scale):
    sc = yrtmi.Scanner("small", 64.0, 4.0, 4.0, 10.0, 150.0, 96, 16)
    im = yrtmi.ImageParams(40, 36, 16, 4.0, 4.5, 4.0)
    rng = np.random.default_rng(n)
    ev = synth.random_events(sc, n, rng)
    t = lambda k: torch.from_numpy(ev[k].astype(np.int32)).to(gpu)
    L = yrtmi.LorSet.pairs(t("d1"), t("d2"))
    # values over three binades, one in eight zero
    v = np.where(rng.random(n) < 0.125, 0.0, rng.uniform(0.5, 4.0, n) * scale)
    vg = torch.from_numpy(v.astype(np.float32)).to(gpu)
    ctx = yrtmi.Context(sc)
    p = ctx.projector(yrtmi.ProjectorParams(sc, numRays=2))
    a, b = (torch.zeros(im.shape, device=gpu) for _ in range(2))
    ctx.back(p, im, a, L, vg)
    for shape in (0, 3):
        plan = ctx.plan(p, im, L, tile_shape=shape)
        for _ in range(2):  # the scale's counters are clear again after a launch
            b.zero_()
            ctx.back(p, im, b, L, vg, plan=plan)
            ctx.synchronize()
            r = rel_l2(b.cpu().numpy(), a.cpu().numpy()) if float(a.abs().sum()) else 0.0
            print(f"n {n} scale {scale:g} shape {shape}: planned vs direct {r:.2e}", flush=True)
            assert r <= 2e-6
