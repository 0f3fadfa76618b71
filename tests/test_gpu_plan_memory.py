"""Plan memory kept for reuse, on the GPU: a plan made in the memory of a
dropped one backprojects what a first plan does, while work that used the
dropped plan is still queued (bit for bit: with one chunk per tile each voxel
is one exact fixed-point sum, whatever the records' order); the memory kept
counts as free, and goes back to the driver when asked for."""
import ctypes as C
import gc

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
    base = free_bytes(ctx)  # (what is kept counts as free)
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


def kept_plan(gpu, n):
    """A context whose pool holds a dropped plan of n LORs."""
    gc.collect()  # (no other test's context goes meanwhile)
    sc = yrtmi.Scanner("t", 96.0, 4.0, 4.0, 10.0, 180.0, 128, 24)
    im = yrtmi.ImageParams(64, 64, 32, 4.0, 4.0, 4.0)
    ctx = yrtmi.Context(sc)
    p = ctx.projector(yrtmi.ProjectorParams(sc, numRays=4))
    ev = synth.random_events(sc, n, np.random.default_rng(1))
    t = lambda q: torch.from_numpy(ev[q].astype(np.int32)).to(gpu)
    L = yrtmi.LorSet.pairs(t("d1"), t("d2"))
    plan = ctx.plan(p, im, L)
    size = plan.info()["bytes"]
    del plan
    return ctx, p, im, L, size


def driver_free():
    return torch.cuda.mem_get_info()[0]


def test_free_memory_is_a_query(gpu):
    """yrtmi_mem_info counts the kept memory as free and leaves it where it
    is, also inside a recording, which stays good; yrtmi_mem_trim gives it
    back and is refused while recording."""
    ctx, p, im, L, size = kept_plan(gpu, 400_000)
    x, u = torch.ones(im.shape, device=gpu), torch.zeros(im.shape, device=gpu)
    ref = torch.zeros(im.shape, device=gpu)
    ctx.set_stream(torch.cuda.Stream())
    ctx.em_subset(p, im, x, ref, L)
    ctx.synchronize()
    held = driver_free()
    free = free_bytes(ctx)
    kept = free - held
    print(f"plan {size >> 20} MiB, kept {kept >> 20} MiB", flush=True)
    assert kept > 64 << 20 and driver_free() == held
    with ctx.graph() as g:
        ctx.fill(u, 0.0)
        ctx.em_subset(p, im, x, u, L)
        inside = free_bytes(ctx)
        with pytest.raises(capi.YrtmiError):
            ctx.mem_trim()
    assert inside == free and driver_free() == held
    for _ in range(2):
        g.launch()
        ctx.synchronize()
        assert float((u - ref).norm() / ref.norm()) <= 1e-5
    ctx.mem_trim()
    # (blocks below the driver's 2 MiB granule may stay in one with live memory)
    assert driver_free() >= held + kept - (16 << 20)


def test_memory_bounds(gpu):
    """A plan within a budget takes no larger kept block than it counts, and the
    scratch of calls without a plan stays within its 1 GiB as it grows."""
    ctx, p, im, L, _ = kept_plan(gpu, 480_000)
    ctx.mem_trim()
    plan = ctx.plan(p, im, L)
    del plan  # kept: every block 1.2 times what the next plan needs
    S = L.slice(0, 400_000)
    free = free_bytes(ctx)
    opt = capi.PlanOptions(0, 0, 0, 1 << 32, 0)
    h, ci, cl, b = C.c_void_p(), im.c(), S.c(), C.c_int64()
    capi.check(capi.lib().yrtmi_plan_create(ctx.h, p.h, C.byref(ci), C.byref(cl), C.byref(opt),
                                            C.byref(h)))
    capi.check(capi.lib().yrtmi_plan_info(h, None, None, C.byref(b)))
    taken = free - free_bytes(ctx)
    capi.lib().yrtmi_plan_destroy(h)
    print(f"plan counts {b.value >> 20} MiB, took {taken >> 20}", flush=True)
    assert b.value > 64 << 20 and taken <= b.value + (16 << 20)  # (five blocks' rounding)

    d1 = torch.randint(0, 128 * 24, (6_000_000,), device=gpu, dtype=torch.int32)
    d2 = d1.flip(0).contiguous()
    v = torch.ones(d1.numel(), device=gpu)
    u = torch.zeros(im.shape, device=gpu)
    torch.cuda.synchronize()
    ctx.mem_trim()
    free = free_bytes(ctx)
    for k in (1_450_000, 1_800_000, 6_000_000):
        ctx.back(p, im, u, yrtmi.LorSet.pairs(d1[:k], d2[:k]), v)
        ctx.synchronize()
        took = free - free_bytes(ctx)
        print(f"{k} LORs: scratch {took >> 20} MiB", flush=True)
        assert 600 << 20 < took <= (1 << 30) + (16 << 20)
