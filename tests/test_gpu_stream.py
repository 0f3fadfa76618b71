"""Backprojections without a plan on the GPU, of enough rays to be binned by
tiles on the device: against the same calls with direct accumulation (global
atomics, never binned).

Bar 1e-5 relative L2, the projector tests' (dyadic voxels: the tile sums are
FP64, the direct ones sum some 10^4 FP32 terms a voxel, whose rounding grows
as the square root: 100 x 6e-8).  Below and above the
rule's thresholds; one, two and many batches; every LOR source; a batch with more records
than there is room for (it takes the direct kernel)."""
import numpy as np
import pytest
import torch

import yrtmi
from helpers import rel_l2
from yrtmi import synth

pytestmark = pytest.mark.gpu

SC = ("t", 96.0, 4.0, 4.0, 10.0, 180.0, 128, 24)


def setup(im, n, proj="Siddon", rays=1, tof=None, psf=False, fp64=False, frames=0, seed=3,
          sc=SC, gpu=None, motion=0):
    sc = yrtmi.Scanner(*sc)
    rng = np.random.default_rng(seed)
    ev = synth.random_events(sc, n, rng, tof_fwhm_ps=tof)
    t = lambda a, d: torch.from_numpy(np.ascontiguousarray(a).astype(d)).to(gpu)
    ctx = yrtmi.Context(sc)
    mot = None
    if motion:
        ctx.upload_motion(synth.rigid_transforms(rng, motion))
        mot = t(rng.integers(0, motion + 1, n), np.uint8)  # one index past the last: skipped
    fr = t(rng.integers(-1, frames, n), np.int32) if frames else None
    L = yrtmi.LorSet.pairs(t(ev["d1"], np.int32), t(ev["d2"], np.int32),
                           tof=t(ev["tof"], np.float32) if tof else None, frame=fr,
                           motion_frame=mot)
    pp = yrtmi.ProjectorParams(sc, projectorType=proj, numRays=rays, setupFP64=fp64)
    if tof:
        pp.addTOF(tof, 5)
    if psf:
        k, pp.psf_s_step, pp.psf_k_spacing = synth.gaussian_psf_row(2.0, num_s=2, s_step=60.0)
        pp.psf_kernels = k * np.array([[1.0], [1.1]], np.float32)
    return ctx, ctx.projector(pp), L, rng


def pair(gpu, im, proj, call, base=2.0 ** -12):
    """call(img) with per-XCD accumulation (binned) and with direct atomics,
    each into an image that already holds something."""
    out = []
    for xcd in (True, False):
        proj.set_accumulation(xcd)
        img = torch.full(im.shape, base, device=gpu)
        call(img)
        torch.cuda.synchronize()
        out.append((img - base).cpu().numpy())
    r = rel_l2(out[0], out[1])
    print(f"binned vs direct rel L2 {r:.2e}, sum {out[1].sum():.4e}", flush=True)
    assert np.abs(out[1]).sum() > 0
    assert r <= 1e-5
    return out


CASES = [
    # name, image, n, kwargs
    ("below", (64, 60, 30, 4.0, 4.5, 2.0), 131_071, dict()),
    ("above", (64, 60, 30, 4.0, 4.5, 2.0), 131_073, dict()),
    ("above_large_image", (160, 160, 96, 1.5, 1.5, 1.0), 32_769, dict()),
    ("rays4_tof", (64, 60, 30, 4.0, 4.5, 2.0), 60_001, dict(rays=4, tof=250.0)),
    ("rays3_frames", (33, 65, 17, 4.0, 4.0, 4.0), 50_000, dict(rays=3, frames=3)),
    ("motion_tof", (64, 64, 32, 4.0, 4.0, 2.0), 140_000, dict(tof=300.0, motion=4)),
    ("fp64", (64, 60, 30, 4.0, 4.5, 2.0), 70_000, dict(rays=2, tof=250.0, fp64=True)),
    ("dd", (64, 60, 30, 4.0, 4.5, 2.0), 70_000, dict(proj="DD")),
    ("dd_tof_psf", (61, 60, 31, 4.0, 4.5, 2.0), 70_000, dict(proj="DD", tof=300.0, psf=True)),
    ("two_batches", (64, 64, 32, 4.0, 4.0, 2.0), 700_000, dict(rays=16, tof=250.0)),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_back_and_em(gpu, case):
    _, imd, n, kw = case
    im = yrtmi.ImageParams(*imd, nt=max(1, kw.get("frames", 0)))
    ctx, p, L, rng = setup(im, n, gpu=gpu, **kw)
    g = torch.Generator(gpu).manual_seed(5)
    v = torch.rand(n, device=gpu, generator=g) - 0.3
    v[::17] = 0.0
    pair(gpu, im, p, lambda u: ctx.back(p, im, u, L, v))
    x = 0.5 + torch.rand(im.shape, device=gpu, generator=g)
    c = {k: 0.2 + torch.rand(n, device=gpu, generator=g)
         for k in ("meas", "sens", "att", "randoms", "scatter")}
    c["meas"][::5] = 0.0
    pair(gpu, im, p, lambda u: ctx.em_subset(p, im, x, u, L, global_scale=1.5, **c))


@pytest.mark.parametrize("kw", [dict(), dict(tof=250.0, rays=4), dict(fp64=True, rays=2),
                                dict(proj="DD", tof=300.0)], ids=str)
def test_values_of_different_scales(gpu, kw):
    """Each term keeps FP32's 24 bits whatever its size beside the call's other
    values: values over 60 binades in one call and a frame 1e-15 of the
    others, every voxel against the FP32 atomics.  Bar: some 10^3 terms of one
    sign a voxel, each rounding 6e-8 of the sum in FP32: 6e-5 at most."""
    frames = 3
    im = yrtmi.ImageParams(64, 64, 32, 4.0, 4.0, 2.0, nt=frames)
    n = 140_000
    ctx, p, L, rng = setup(im, n, gpu=gpu, frames=frames, **kw)
    v = 2.0 ** rng.uniform(-60.0, 0.0, n)
    v = np.where(L.frame.cpu().numpy() == 1, 1e-15 * rng.uniform(0.5, 1.0, n), v)
    v = torch.from_numpy(v.astype(np.float32)).to(gpu)
    a, b = pair(gpu, im, p, lambda u: ctx.back(p, im, u, L, v), base=0.0)
    a, b = a.astype(np.float64), b.astype(np.float64)
    assert (b.reshape(frames, -1).max(1) > 0).all()
    r = np.abs(a - b)[b > 0] / b[b > 0]
    print(f"largest relative difference of a voxel {r.max():.2e}", flush=True)
    assert ((a > 0) == (b > 0)).all() and r.max() <= 6e-5


@pytest.mark.parametrize("kw", [dict(rays=4, tof=250.0), dict(rays=3, frames=2, fp64=True),
                                dict(proj="DD", tof=300.0)], ids=str)
@pytest.mark.parametrize("keep", [0.0, 3e-5, 0.03, 1.0])
def test_em_subset_of_few_nonzero_lors(gpu, kw, keep):
    """EM subsets that skip most of their LORs (measurement, sensitivity or
    attenuation 0), or all, or none: the others are listed first."""
    im = yrtmi.ImageParams(64, 60, 30, 4.0, 4.5, 2.0, nt=max(1, kw.get("frames", 0)))
    n = 300_001
    ctx, p, L, _ = setup(im, n, gpu=gpu, **kw)
    g = torch.Generator(gpu).manual_seed(5)
    x = 0.5 + torch.rand(im.shape, device=gpu, generator=g)
    c = {k: 0.2 + torch.rand(n, device=gpu, generator=g)
         for k in ("meas", "sens", "att", "randoms", "scatter")}
    for k in ("meas", "sens", "att"):
        c[k][torch.rand(n, device=gpu, generator=g) >= keep ** (1 / 3)] = 0.0
    on = int(((c["meas"] != 0) & (c["sens"] != 0) & (c["att"] != 0)).sum())
    print(f"{on} of {n} LORs", flush=True)
    if on == 0:
        u = torch.zeros(im.shape, device=gpu)
        ctx.em_subset(p, im, x, u, L, **c)
        assert float(u.abs().max()) == 0.0
    else:
        pair(gpu, im, p, lambda u: ctx.em_subset(p, im, x, u, L, **c))
        pair(gpu, im, p, lambda u: ctx.em_subset(p, im, x, u, L, att=c["att"]))


def test_em_subset_listed_in_two_parts(gpu):
    """More LORs than are listed at a time (2^24), batches ending inside both."""
    im = yrtmi.ImageParams(64, 60, 30, 4.0, 4.5, 2.0)
    n = (1 << 24) + 1_234_567
    ctx, p, _, _ = setup(im, 10, gpu=gpu)
    g = torch.Generator(gpu).manual_seed(5)
    d = [torch.randint(0, 128 * 24, (n,), device=gpu, generator=g, dtype=torch.int32)
         for _ in range(2)]
    L = yrtmi.LorSet.pairs(*d)
    meas = torch.rand(n, device=gpu, generator=g)
    meas[::2] = 0.0
    meas[100_000:200_000] = 0.0
    x = 0.5 + torch.rand(im.shape, device=gpu, generator=g)
    pair(gpu, im, p, lambda u: ctx.em_subset(p, im, x, u, L, meas=meas))


@pytest.mark.parametrize("dd", [False, True])
@pytest.mark.parametrize("att", [False, True])
def test_sensitivity_of_histogram_subset(gpu, dd, att):
    im = yrtmi.ImageParams(48, 50, 20, 4.0, 4.0, 4.0)
    ctx, p, _, _ = setup(im, 10, proj="DD" if dd else "Siddon", rays=1 if dd else 2, gpu=gpu)
    L = yrtmi.LorSet.histo_subset(ctx, 5, 3)
    g = torch.Generator(gpu).manual_seed(5)
    s = torch.rand(L.n, device=gpu, generator=g)
    mu = 0.1 * torch.rand(im.shape, device=gpu, generator=g)
    pair(gpu, im, p, lambda u: ctx.sensitivity(p, im, u, L, att_im=im if att else None,
                                               att_img=mu if att else None, sens=s))
    bins = torch.arange(0, 200_000, 3, device=gpu, dtype=torch.int32)
    B = yrtmi.LorSet.bins_(bins)
    v = torch.rand(B.n, device=gpu, generator=g)
    pair(gpu, im, p, lambda u: ctx.back(p, im, u, B, v))


@pytest.mark.parametrize("src", ["histo", "bins", "pairs", "pairs_dd"])
def test_batches_of_every_source(gpu, src):
    """Several batches, the last one ragged, of each LOR source, with frames,
    motion and every per-LOR factor: a batch starts inside each array, and
    inside the subset iterator."""
    dd = src == "pairs_dd"
    frames = 0 if src == "histo" else 2
    im = yrtmi.ImageParams(64, 60, 30, 4.0, 4.5, 2.0, nt=max(1, frames))
    n = 4_400_001 if dd else 800_001
    ctx, p, L, rng = setup(im, n if src[0] == "p" else 10, proj="DD" if dd else "Siddon",
                           rays=1 if dd else 16, tof=250.0, frames=frames if src[0] == "p" else 0,
                           motion=4 if src[0] == "p" else 0, gpu=gpu)
    t = lambda a, d: torch.from_numpy(a.astype(d)).to(gpu)
    if src == "histo":
        L = yrtmi.LorSet.histo_subset(ctx, 3, 1)
        n = L.n
    elif src == "bins":
        total = int(np.prod(ctx.histo_dims))
        L = yrtmi.LorSet.bins_(t(rng.integers(0, total + 10, n), np.int32),
                               tof=t(rng.normal(0.0, 100.0, n), np.float32),
                               frame=t(rng.integers(-1, frames, n), np.int32))
    # bytes a LOR: ray table (64 a ray, DD 128), records (12 a ray and tile, DD 8)
    assert n * (256 if dd else 16 * (64 + 6 * 12)) > 1 << 30
    g = torch.Generator(gpu).manual_seed(5)
    v = torch.rand(n, device=gpu, generator=g)
    pair(gpu, im, p, lambda u: ctx.back(p, im, u, L, v))
    x = 0.5 + torch.rand(im.shape, device=gpu, generator=g)
    c = {k: 0.2 + torch.rand(n, device=gpu, generator=g)
         for k in ("meas", "sens", "att", "randoms", "scatter")}
    pair(gpu, im, p, lambda u: ctx.em_subset(p, im, x, u, L, randoms=c["randoms"],
                                             scatter=c["scatter"]))
    c["meas"][::3] = 0.0
    pair(gpu, im, p, lambda u: ctx.em_subset(p, im, x, u, L, **c))
    if frames == 0:
        mu_im = yrtmi.ImageParams(161, 127, 103, 1.5, 1.75, 1.0)  # bricked
        mu = 0.05 * torch.rand(mu_im.shape, device=gpu, generator=g)
        pair(gpu, im, p, lambda u: ctx.sensitivity(p, im, u, L, att_im=mu_im, att_img=mu, sens=v))


def test_batch_of_high_footprints(gpu):
    """Crystals 240 voxels high over one column of 64 tiles: some 30 records
    for each LOR that meets the image, for which there is room."""
    im = yrtmi.ImageParams(32, 32, 512, 4.0, 4.0, 0.25)
    ctx, p, L, _ = setup(im, 70_000, proj="DD", gpu=gpu,
                         sc=("t", 128.0, 60.0, 4.0, 10.0, 180.0, 128, 2))
    v = torch.rand(L.n, device=gpu, generator=torch.Generator(gpu).manual_seed(1))
    plan = ctx.plan(p, im, L, tile_shape=3)
    assert plan.info()["records"] > 8 * L.n
    pair(gpu, im, p, lambda u: ctx.back(p, im, u, L, v))


@pytest.mark.parametrize("kind", ["back", "em", "em_listed", "sens"])
@pytest.mark.parametrize("kw", [dict(), dict(tof=3000.0), dict(fp64=True)], ids=str)
def test_batch_with_more_records_than_room(gpu, kind, kw):
    """Rays from a tall image's first ring to its last, some 100 tiles each
    (TOF too wide to cut them), where there is room for 64: the batch takes the
    direct kernel (kBackIf)."""
    im = yrtmi.ImageParams(32, 32, 1024, 4.0, 4.0, 0.25)
    n = 140_000
    ctx, p, _, rng = setup(im, 10, gpu=gpu, sc=("t", 256.0, 4.0, 3.4, 10.0, 70.0, 128, 64), **kw)
    i = rng.integers(0, 128, n)
    j = (i + rng.integers(48, 81, n)) % 128
    t = lambda a, d: torch.from_numpy(a.astype(d)).to(gpu)
    tof = t(rng.normal(0.0, 100.0, n), np.float32) if "tof" in kw else None
    L = yrtmi.LorSet.pairs(t(i, np.int32), t(j + 128 * 63, np.int32), tof=tof)
    records = ctx.plan(p, im, L, tile_shape=3).info()["records"]
    print(f"{records / n:.1f} records a ray", flush=True)
    assert records > 64 * n
    g = torch.Generator(gpu).manual_seed(1)
    v = 0.5 + torch.rand(n, device=gpu, generator=g)
    x = 0.5 + torch.rand(im.shape, device=gpu, generator=g)
    mu = 0.01 * torch.rand(im.shape, device=gpu, generator=g)
    pair(gpu, im, p, {
        "back": lambda u: ctx.back(p, im, u, L, v),
        "em": lambda u: ctx.em_subset(p, im, x, u, L),
        "em_listed": lambda u: ctx.em_subset(p, im, x, u, L, meas=v),
        "sens": lambda u: ctx.sensitivity(p, im, u, L, att_im=im, att_img=mu, sens=v)}[kind])


def test_recorded_and_on_other_streams(gpu):
    """Recorded after one eager call and replayed between other calls that
    use (and grow) the same scratch, and on streams in turn."""
    im = yrtmi.ImageParams(64, 60, 30, 4.0, 4.5, 2.0)
    ctx, p, L, _ = setup(im, 70_000, rays=2, tof=250.0, gpu=gpu)
    big = setup(im, 300_000, rays=2, tof=250.0, gpu=gpu, seed=9)[2]
    g = torch.Generator(gpu).manual_seed(5)
    v, w = torch.rand(L.n, device=gpu, generator=g), torch.rand(big.n, device=gpu, generator=g)
    ref, ref2 = (torch.zeros(im.shape, device=gpu) for _ in range(2))
    p.set_accumulation(False)
    ctx.back(p, im, ref, L, v)
    ctx.back(p, im, ref2, big, w)
    torch.cuda.synchronize()
    p.set_accumulation(True)
    streams = [torch.cuda.Stream() for _ in range(2)]
    u, u2 = (torch.zeros(im.shape, device=gpu) for _ in range(2))
    torch.cuda.synchronize()
    ctx.set_stream(streams[0])
    ctx.back(p, im, u, L, v)
    with ctx.graph() as gr:
        ctx.fill(u, 0.0)
        ctx.back(p, im, u, L, v)
    for k in range(4):
        ctx.set_stream(streams[k % 2])
        gr.launch()
        ctx.set_stream(streams[(k + 1) % 2])
        ctx.fill(u2, 0.0)
        ctx.back(p, im, u2, big, w)  # the first grows the scratch
        torch.cuda.synchronize()
        a, b = rel_l2(u.cpu().numpy(), ref.cpu().numpy()), rel_l2(u2.cpu().numpy(),
                                                                  ref2.cpu().numpy())
        print(f"replay {k}: {a:.2e}, other call {b:.2e}", flush=True)
        assert a <= 1e-5 and b <= 1e-5


LARGE = (161, 127, 103, 1.5, 1.75, 1.0)   # 2^21 voxels and more
SMALL = (67, 65, 63, 4.0, 4.0, 4.0)       # 2^18 and more: bricks from 2^19 rays
BRICKED = [(LARGE, dict(rays=1, tof=250.0)), (LARGE, dict(rays=2, tof=250.0)),
           (LARGE, dict(rays=3, frames=2)), (LARGE, dict(rays=5)),
           (LARGE, dict(rays=2, tof=300.0, fp64=True)), (SMALL, dict(rays=1)),
           (SMALL, dict(rays=3, tof=250.0, frames=2))]


@pytest.mark.parametrize("dims,kw", BRICKED, ids=str)
def test_bricked_forward_is_the_forward(gpu, dims, kw):
    """A forward of many rays of a large image gathers from its bricked copy;
    calls of a third of its LORs do not: the same sums, bit for bit, also
    recorded and replayed, and the EM ratio's (1 / A x without measurements)
    against its reciprocal's rounding."""
    nt = max(1, kw.get("frames", 0))
    R = kw["rays"]
    im = yrtmi.ImageParams(*dims, nt=nt)
    step = max(im.nvox * nt // 12, (1 << 19) // 3) // R + 1000
    n = 3 * step
    # bricked all together, rows in thirds, which are above the calls of several
    # lanes a ray
    if dims is LARGE:
        assert im.nvox >= 1 << 21 and 4 * n * R >= im.nvox * nt > 4 * step * R
    else:
        assert im.nvox >= 1 << 18 and n * R >= 1 << 19 > step * R
    assert step * R > 65536
    ctx, p, L, _ = setup(im, n, gpu=gpu, **kw)
    x = torch.rand(im.shape, device=gpu, generator=torch.Generator(gpu).manual_seed(2))
    y, z = torch.zeros(n, device=gpu), torch.zeros(n, device=gpu)
    ctx.forward(p, im, x, L, y)
    for a in range(0, n, step):
        ctx.forward(p, im, x, L.slice(a, a + step), z[a:a + step])
    torch.cuda.synchronize()
    assert float(y.abs().sum()) > 0 and torch.equal(y, z)
    ctx.em_ratio(p, im, x, L, z)
    on = y > 1e-6
    assert float((z * y - 1.0)[on].abs().max()) <= 4e-7
    s = torch.cuda.Stream()
    ctx.set_stream(s)
    with ctx.graph() as g:
        ctx.forward(p, im, x, L, z)
    for _ in range(3):
        z.zero_()
        torch.cuda.synchronize()
        g.launch()
        ctx.forward(p, im, x, L, y)
        torch.cuda.synchronize()
        assert torch.equal(y, z)


@pytest.mark.parametrize("kw", [dict(proj="DD", psf=True), dict(proj="DD", tof=300.0, frames=2),
                                dict(proj="DD", fp64=True)], ids=str)
def test_bricked_dd_ratio_is_the_ratio(gpu, kw):
    """EM ratios of a large image, from its bricked copy, against those of a
    recording made before there is a buffer for it (from rows): the same sums,
    bit for bit; and from two streams in turn."""
    nt = max(1, kw.get("frames", 0))
    im = yrtmi.ImageParams(161, 127, 103, 1.5, 1.75, 1.0, nt=nt)
    ctx, p, L, _ = setup(im, 30_000, gpu=gpu, **kw)
    x = 0.5 + torch.rand(im.shape, device=gpu, generator=torch.Generator(gpu).manual_seed(2))
    x2 = 2.0 * x
    y, z, w = (torch.zeros(L.n, device=gpu) for _ in range(3))
    s, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    ctx.set_stream(s)
    with ctx.graph() as g:
        ctx.em_ratio(p, im, x, L, y)
    g.launch()
    for k in range(3):
        ctx.set_stream(s2)
        ctx.em_ratio(p, im, x2, L, w)
        ctx.set_stream(s)
        ctx.em_ratio(p, im, x, L, z)
        torch.cuda.synchronize()
        assert float(y.abs().sum()) > 0 and torch.equal(y, z)
        assert torch.allclose(w, 0.5 * y, rtol=1e-6, atol=0)


@pytest.mark.parametrize("dims", [(3, 2, 40, 60.0, 60.0, 2.0), (33, 65, 17, 4.0, 4.0, 4.0),
                                  (161, 127, 103, 1.5, 1.75, 1.0)], ids=str)
@pytest.mark.parametrize("kw", [dict(), dict(tof=300.0, psf=True), dict(frames=2, fp64=True)],
                         ids=str)
def test_dd_forward_lanes(gpu, dims, kw):
    """DD projections with four lanes per LOR (calls of up to 196608) against
    one (a call of all; the largest image from bricks), also of 1, 15 and 65 LORs
    and of images of fewer slices than lanes.  Sums of the same positive terms, some
    10^3 to 10^4, in two orders: 100 x 6e-8 of rounding."""
    im = yrtmi.ImageParams(*dims, nt=max(1, kw.get("frames", 0)))
    n = 540_000 if dims[0] > 100 else 196_609
    ctx, p, L, _ = setup(im, n, proj="DD", gpu=gpu, **kw)
    x = 0.5 + torch.rand(im.shape, device=gpu, generator=torch.Generator(gpu).manual_seed(2))
    y, z = torch.full((n,), -1.0, device=gpu), torch.full((n,), -1.0, device=gpu)
    ctx.forward(p, im, x, L, y)
    at = 0
    for k in (1, 15, 65, 196_527, 196_608, n):
        b = min(n, at + k)
        if b > at:
            ctx.forward(p, im, x, L.slice(at, b), z[at:b])
        at = b
    torch.cuda.synchronize()
    y, z = y.cpu().numpy(), z.cpu().numpy()
    print(f"lanes rel L2 {rel_l2(z, y):.2e}", flush=True)
    assert np.abs(y).sum() > 0 and rel_l2(z, y) <= 1e-5
    assert ((y == 0) == (z == 0)).all()


@pytest.mark.parametrize("dims", [(3, 2, 40, 60.0, 60.0, 2.0), (33, 65, 17, 4.0, 4.1, 4.0),
                                  (161, 127, 103, 1.5, 1.75, 1.0), (1, 1, 1, 90.0, 90.0, 90.0)],
                         ids=str)
@pytest.mark.parametrize("kw", [dict(), dict(tof=250.0, rays=3), dict(tof=90.0, frames=2),
                                dict(rays=8, motion=3)], ids=str)
def test_forward_lanes_along_a_ray(gpu, dims, kw):
    """Siddon projections of small calls, four lanes along each ray, against a
    call of all LORs, one lane per ray.  Every segment is in one lane's stretch, so the
    sums differ by rounding, of some 400 positive terms at most: 20 x 6e-8,
    and where voxel sizes are no short binary fractions by planes an ulp of
    the scanner apart, 1e-5 of a voxel."""
    im = yrtmi.ImageParams(*dims, nt=max(1, kw.get("frames", 0)))
    R = kw.get("rays", 1)
    n = 140_000 // R + 1
    ctx, p, L, _ = setup(im, n, gpu=gpu, **kw)
    x = 0.5 + torch.rand(im.shape, device=gpu, generator=torch.Generator(gpu).manual_seed(2))
    y, z = torch.full((n,), -1.0, device=gpu), torch.full((n,), -1.0, device=gpu)
    ctx.forward(p, im, x, L, y)
    at = 0
    for k in (1, 15, 65, 30_000 // R, 30_000 // R, 30_000 // R, 30_000 // R, 30_000 // R):
        b = min(n, at + k)
        ctx.forward(p, im, x, L.slice(at, b), z[at:b])
        at = b
    torch.cuda.synchronize()
    ref, y, z = y.abs().max().item(), y.cpu().numpy()[:at], z.cpu().numpy()[:at]
    print(f"lanes rel L2 {rel_l2(z, y):.2e} max {np.abs(z - y).max() / ref:.2e}", flush=True)
    assert ref > 0 and rel_l2(z, y) <= 1e-5 and np.abs(z - y).max() <= 1e-4 * ref


@pytest.mark.parametrize("dims", [(33, 65, 17, 4.0, 4.0, 4.0), (161, 127, 103, 1.5, 1.75, 1.0)],
                         ids=str)
@pytest.mark.parametrize("kw", [dict(rays=3), dict(proj="DD")], ids=str)
def test_launch_shape_of_forwards(gpu, dims, kw):
    """Forwards with the block and grid that the caller set, by way of small
    calls (several lanes a ray or LOR), bricks, and neither: the same sums.  (A
    grid far too small for the LORs is seen by its time: one block of 64
    threads against the whole chip.)"""
    im = yrtmi.ImageParams(*dims)
    n = 540_000 // kw.get("rays", 1)
    ctx, p, L, _ = setup(im, n, gpu=gpu, **kw)
    x = 0.5 + torch.rand(im.shape, device=gpu, generator=torch.Generator(gpu).manual_seed(2))
    for S in (L, L.slice(0, 10_001)):
        y, z = torch.zeros(S.n, device=gpu), torch.full((S.n,), -1.0, device=gpu)
        ctx.forward(p, im, x, S, y)
        times = []
        for block, grid in ((256, 0), (64, 0), (192, 24), (128, 8)):
            p.set_launch(block=block, grid=grid)
            t = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            t[0].record()
            ctx.forward(p, im, x, S, z.fill_(-1.0))
            t[1].record()
            torch.cuda.synchronize()
            times.append(t[0].elapsed_time(t[1]))
            assert float(y.abs().sum()) > 0 and torch.equal(y, z)
        p.set_launch()
        print("ms:", " ".join(f"{k:.3f}" for k in times), flush=True)
        assert times[3] > 2 * times[1]
