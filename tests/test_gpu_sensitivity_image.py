"""Attenuation images of 2^21 voxels and more in sensitivity calls, on the
GPU: their forward gathers from a bricked copy (kSensValue<.., true>); against
the same call with the per-LOR factors of yrtmi_attenuation_factors, which
reads the image as it is.

Bar 1e-5 relative L2 (the two differ by the order of the backprojection's
sums; with the FP64 set-up also by the line integrals' own set-up, 1e-6).

A dynamic descriptor of the attenuation image stands for its frame 0: the
other frames, NaN here, are not read, and no copy is made of them (they are
there all the same, so that a call that did read them would stay in bounds)."""
import ctypes as C

import numpy as np
import pytest
import torch

import yrtmi
from helpers import rel_l2
from yrtmi import capi

pytestmark = pytest.mark.gpu


def free_bytes(ctx):
    f = C.c_int64()
    capi.check(capi.lib().yrtmi_mem_info(ctx.h, C.byref(f), None))
    return f.value


def sensitivity(ctx, p, im, img, L, mu_im, mu, nt, sens, plan):
    ci, cl, ca = im.c(nt=1), L.c(), mu_im.c(nt=nt)
    args = [ctx.h, p.h, C.byref(ci), img.data_ptr(), C.byref(cl), C.byref(ca), mu.data_ptr(),
            sens.data_ptr()]
    f = capi.lib().yrtmi_sensitivity_planned if plan else capi.lib().yrtmi_sensitivity
    capi.check(f(*args, *([plan.h] if plan else [])))


@pytest.mark.parametrize("proj,fp64", [("Siddon", False), ("Siddon", True), ("DD", False)])
@pytest.mark.parametrize("planned", [False, True])
def test_large_attenuation_image(gpu, proj, fp64, planned):
    sc = yrtmi.Scanner("t", 96.0, 4.0, 4.0, 10.0, 180.0, 128, 24)
    im = yrtmi.ImageParams(48, 50, 20, 4.0, 4.0, 4.0)
    mu_im = yrtmi.ImageParams(161, 127, 103, 1.5, 1.75, 1.0)
    assert mu_im.nvox >= 1 << 21
    ctx = yrtmi.Context(sc)
    p = ctx.projector(yrtmi.ProjectorParams(sc, projectorType=proj, setupFP64=fp64))
    L = yrtmi.LorSet.histo_subset(ctx, 2, 1)
    frames = 2
    assert 4 * L.n >= frames * mu_im.nvox  # (fewer LORs read the image as it is)
    g = torch.Generator(gpu).manual_seed(5)
    s = torch.rand(L.n, device=gpu, generator=g)
    mu = torch.full((frames, mu_im.nz, mu_im.ny, mu_im.nx), float("nan"), device=gpu)
    mu[0] = 0.2 * torch.rand(mu_im.shape, device=gpu, generator=g).reshape(mu[0].shape)
    acf = torch.empty(L.n, device=gpu)
    ctx.attenuation_factors(mu_im, mu[0].reshape(mu_im.shape), L, acf)
    plan = ctx.plan(p, im, L) if planned else None
    ref, one, dyn = (torch.zeros(im.shape, device=gpu) for _ in range(3))
    ctx.sensitivity(p, im, ref, L, sens=s * acf, plan=plan)
    sensitivity(ctx, p, im, one, L, mu_im, mu, 1, s, plan)
    torch.cuda.synchronize()
    free = free_bytes(ctx)
    sensitivity(ctx, p, im, dyn, L, mu_im, mu, frames, s, plan)
    torch.cuda.synchronize()
    assert free_bytes(ctx) == free
    ref, one, dyn = (t.cpu().numpy() for t in (ref, one, dyn))
    print(f"bricked attenuation rel L2 {rel_l2(one, ref):.2e}, dynamic descriptor "
          f"{rel_l2(dyn, ref):.2e}", flush=True)
    assert np.abs(ref).sum() > 0 and float(acf.min()) < 0.5
    assert rel_l2(one, ref) <= 1e-5 and rel_l2(dyn, ref) <= 1e-5
