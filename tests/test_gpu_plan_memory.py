"""Plan memory kept for reuse, on the GPU: a plan made in the memory of a
dropped one backprojects what a first plan does, while work that used the
dropped plan is still queued (bit for bit: with one chunk per tile each voxel
is one exact fixed-point sum, whatever the records' order); the memory goes
back before free memory is reported."""
import ctypes as C

import numpy as np
import pytest
import torch

import yrtmi
from yrtmi import capi, synth

pytestmark = pytest.mark.gpu


def free_bytes(ctx):
    f = C.c_int64()
    capi.check(capi.lib().yrtmi_mem_info(ctx.h, C.byref(f), None))
    return f.value


def test_plans_in_reused_memory(gpu):
    sc = yrtmi.Scanner("t", 96.0, 4.0, 4.0, 10.0, 180.0, 128, 24)
    im = yrtmi.ImageParams(64, 64, 32, 4.0, 4.0, 4.0)
    ctx = yrtmi.Context(sc)
    p = ctx.projector(yrtmi.ProjectorParams(sc, numRays=3))
    sets = []
    for k, n in enumerate((200_000, 190_000, 1000)):
        ev = synth.random_events(sc, n, np.random.default_rng(k))
        t = lambda q: torch.from_numpy(ev[q].astype(np.int32)).to(gpu)
        L = yrtmi.LorSet.pairs(t("d1"), t("d2"))
        v = torch.rand(n, device=gpu, generator=torch.Generator(gpu).manual_seed(k))
        ref = torch.zeros(im.shape, device=gpu)
        plan = ctx.plan(p, im, L, 1 << 24, tile_shape=3)
        ctx.back(p, im, ref, L, v, plan=plan)
        ctx.synchronize()
        sets.append((L, v, ref))
        del plan
    base = free_bytes(ctx)  # everything given back
    outs = []
    for _ in range(3):
        for L, v, ref in sets:
            plan = ctx.plan(p, im, L, 1 << 24, tile_shape=3)
            out = torch.zeros(im.shape, device=gpu)
            ctx.back(p, im, out, L, v, plan=plan)
            outs.append((out, ref))
            del plan  # its launches are still queued
    ctx.synchronize()
    for out, ref in outs:
        assert torch.equal(out, ref)
    assert abs(free_bytes(ctx) - base) < 64 << 20
