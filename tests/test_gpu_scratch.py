"""The context's scratch (bricked images, tile binning without a plan) under
graphs of the caller's own and graphs launched through another context, on the
GPU.  Bars: forward projections and ratios are the same sums in the same
order, or, where a call reads rows instead of bricks, of the same values: bit
for bit.  Backprojections 1e-5 relative L2, as in test_gpu_stream.py."""
import ctypes as C
import gc
import threading

import pytest
import torch

import yrtmi
from helpers import rel_l2
from test_gpu_stream import setup
from yrtmi import capi

pytestmark = pytest.mark.gpu

BIG = (161, 127, 103, 1.5, 1.75, 1.0)  # 2^21 voxels and more: bricked


def free_bytes(ctx):
    f = C.c_int64()
    capi.check(capi.lib().yrtmi_mem_info(ctx.h, C.byref(f), None))
    return f.value


@pytest.mark.parametrize("kw", [dict(tof=250.0), dict(proj="DD")], ids=str)
def test_captured_by_the_caller(gpu, kw):
    """torch.cuda.graph around the calls, after eager ones on another stream;
    replayed between eager calls on that stream, a larger one among them."""
    im = yrtmi.ImageParams(*BIG)
    n = im.nvox // 4 + 1000
    ctx, p, L, _ = setup(im, n, gpu=gpu, **kw)
    p0 = p if "tof" not in kw else ctx.projector(yrtmi.ProjectorParams(ctx.scanner))
    big = setup(im, 2 * n, gpu=gpu, seed=9, **kw)[2]
    g = torch.Generator(gpu).manual_seed(2)
    x = 0.5 + torch.rand(im.shape, device=gpu, generator=g)
    mu = 0.05 * torch.rand(im.shape, device=gpu, generator=g)
    v = torch.rand(n, device=gpu, generator=g)
    w = torch.rand(big.n, device=gpu, generator=g)
    names = ("fwd", "ratio", "back", "em", "sens")
    L0 = yrtmi.LorSet.pairs(L.d1, L.d2)

    def outputs():
        return [torch.zeros(n if k in ("fwd", "ratio") else im.nvox, device=gpu) for k in names]

    def calls(o):
        ctx.forward(p, im, x, L, o[0])
        ctx.em_ratio(p, im, x, L, o[1])
        for k in (2, 3, 4):
            ctx.fill(o[k], 0.0)
        ctx.back(p, im, o[2].view(im.shape), L, v)
        ctx.em_subset(p, im, x, o[3].view(im.shape), L)
        ctx.sensitivity(p0, im, o[4].view(im.shape), L0, att_im=im, att_img=mu)

    ref, out, eager, more = outputs(), outputs(), outputs(), torch.zeros(im.shape, device=gpu)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    ctx.set_stream(side)
    calls(ref)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ctx.set_stream(torch.cuda.current_stream())
        calls(out)
    ctx.set_stream(side)
    for k in range(3):
        for t in out:
            t.fill_(-1.0)
        torch.cuda.synchronize()
        graph.replay()
        calls(eager)
        ctx.back(p, im, more, big, w)  # (the first grows the scratch)
        torch.cuda.synchronize()
        for name, r, a, b in zip(names, ref, out, eager):
            e = [rel_l2(t.cpu().numpy(), r.cpu().numpy()) for t in (a, b)]
            print(f"replay {k} {name}: captured {e[0]:.2e}, eager {e[1]:.2e}", flush=True)
            assert float(r.abs().sum()) > 0 and max(e) <= 1e-5
            if name in ("fwd", "ratio"):
                assert torch.equal(a, r) and torch.equal(b, r)


def test_graph_launched_through_another_context(gpu):
    """A recorded backprojection replayed through a second context, on that
    one's stream, between eager calls of the first one that use its scratch."""
    im = yrtmi.ImageParams(64, 60, 30, 4.0, 4.5, 2.0)
    ctx, p, L, _ = setup(im, 70_000, rays=2, tof=250.0, gpu=gpu)
    other = setup(im, 200_000, rays=2, tof=250.0, gpu=gpu, seed=9)[2]
    ctx2 = yrtmi.Context(ctx.scanner)
    g = torch.Generator(gpu).manual_seed(5)
    v, w = torch.rand(L.n, device=gpu, generator=g), torch.rand(other.n, device=gpu, generator=g)
    refs = [torch.zeros(im.shape, device=gpu) for _ in range(2)]
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    ctx.set_stream(s1)
    ctx2.set_stream(s2)
    ctx.back(p, im, refs[0], L, v)
    ctx.back(p, im, refs[1], other, w)
    u, u2 = (torch.zeros(im.shape, device=gpu) for _ in range(2))
    torch.cuda.synchronize()
    with ctx.graph() as gr:
        ctx.fill(u, 0.0)
        ctx.back(p, im, u, L, v)
    for k in range(20):
        capi.check(capi.lib().yrtmi_graph_launch(ctx2.h, gr.h))
        ctx.fill(u2, 0.0)
        ctx.back(p, im, u2, other, w)
        if k % 5 == 4:
            torch.cuda.synchronize()
            e = [rel_l2(a.cpu().numpy(), b.cpu().numpy()) for a, b in zip((u, u2), refs)]
            print(f"round {k}: replay {e[0]:.2e}, eager {e[1]:.2e}", flush=True)
            assert max(e) <= 1e-5


def test_graph_and_eager_calls_from_two_threads(gpu):
    """A graph launched through a second context by one thread while another
    makes eager calls on the context that recorded it: each use of the scratch
    waits for the last one, whichever thread it came from."""
    im = yrtmi.ImageParams(64, 60, 30, 4.0, 4.5, 2.0)
    ctx, p, L, _ = setup(im, 70_000, rays=2, tof=250.0, gpu=gpu)
    other = setup(im, 90_000, rays=2, tof=250.0, gpu=gpu, seed=9)[2]
    ctx2 = yrtmi.Context(ctx.scanner)
    g = torch.Generator(gpu).manual_seed(5)
    v, w = torch.rand(L.n, device=gpu, generator=g), torch.rand(other.n, device=gpu, generator=g)
    refs = [torch.zeros(im.shape, device=gpu) for _ in range(2)]
    u, u2 = (torch.zeros(im.shape, device=gpu) for _ in range(2))
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    ctx.set_stream(s1)
    ctx2.set_stream(s2)
    ctx.back(p, im, refs[1], other, w)
    ctx.back(p, im, refs[0], L, v)
    with ctx.graph() as gr:
        ctx.fill(u, 0.0)
        ctx.back(p, im, u, L, v)
    torch.cuda.synchronize()
    errors = []

    def run(call):
        try:
            for _ in range(40):
                call()
        except Exception as e:  # noqa: BLE001 (reported by the test's thread)
            errors.append(e)

    def eager():
        ctx.fill(u2, 0.0)
        ctx.back(p, im, u2, other, w)

    threads = [threading.Thread(target=run, args=(f,)) for f in
               (lambda: capi.check(capi.lib().yrtmi_graph_launch(ctx2.h, gr.h)), eager)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors
    e = [rel_l2(a.cpu().numpy(), b.cpu().numpy()) for a, b in zip((u, u2), refs)]
    print(f"replays {e[0]:.2e}, eager {e[1]:.2e}", flush=True)
    assert max(e) <= 1e-5


def test_scratch_of_a_graph_outlives_its_context(gpu):
    """Scratch that a graph refers to goes back with the graph, not before."""
    gc.collect()  # (no other test's context goes meanwhile)
    im = yrtmi.ImageParams(64, 60, 30, 4.0, 4.5, 2.0)
    ctx, p, L, _ = setup(im, 70_000, rays=2, tof=250.0, gpu=gpu)
    keep = yrtmi.Context(ctx.scanner)
    v = torch.rand(L.n, device=gpu)
    u = torch.zeros(im.shape, device=gpu)
    torch.cuda.synchronize()
    ctx.set_stream(torch.cuda.Stream())
    before = free_bytes(keep)
    ctx.back(p, im, u, L, v)
    with ctx.graph() as gr:
        ctx.back(p, im, u, L, v)
    ctx.synchronize()
    scratch = before - free_bytes(keep)
    assert scratch > 8 << 20
    gr.ctx = None
    del ctx, p
    held = before - free_bytes(keep)
    del gr
    after = before - free_bytes(keep)
    print(f"scratch {scratch >> 20} MiB, held by the graph {held >> 20}, then {after >> 20}",
          flush=True)
    assert held > 8 << 20 and after < 8 << 20
