"""CPU check of the projection-space PSF weights (yrt-pet_amd/csrc/
yrtmi_device.hpp): the form that the tile and ratio kernels take from the
segment table (psfWeightTab) against the 64-bit integral, element by element,
beside the form without it (psfWeight).

Footprints from a thousandth of a tap spacing to all of the kernel, at its
middle, in both tails and over its ends.  A weight is a sum of positive
trapezoids; what it loses beyond their rounding is the place of an end in its
segment, a quotient rounded to 6e-8 of the distance from the centre: an end d
tap spacings inside the kernel's edge, h from the centre, has a value good to
6e-8 h / d.  So the bar is psfWeight's own error: percentiles no more than a
twentieth larger; and where both ends are a tenth of a segment and more inside
the edge and the footprint is no narrower than that, 6e-8 h / 0.1 and some
roundings."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def hw(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("psf") / "libpsf.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC",
                    "-I", os.path.join(HERE, "hostwalk"),
                    "-I", os.path.join(REPO, "yrt-pet_amd", "csrc"),
                    os.path.join(HERE, "hostwalk", "psf_host.cpp"), "-o", out],
                   check=True, capture_output=True)
    lib = C.CDLL(out)
    P = C.c_void_p
    lib.hw_psf.restype = None
    lib.hw_psf.argtypes = [P, C.c_int, C.c_float, C.c_int64, P, P, P]
    return lib


def integral(taps, ks, x0, x1):
    """The integral of the taps' linear interpolant over [x0, x1], in 64 bits."""
    K = len(taps)
    half = (K - 1) // 2
    t = np.concatenate([[0.0, 0.0], taps.astype(np.float64), [0.0, 0.0]])  # from tap -2
    ks = np.float64(ks)
    total = np.zeros(len(x0))
    for j in range(K + 3):  # segment from tap j - 2
        a = (j - 2 - half) * ks
        lo = np.maximum(x0, a)
        hi = np.minimum(x1, a + ks)
        d = np.maximum(hi - lo, 0.0)
        v = lambda x: t[j] + (t[j + 1] - t[j]) * (x - a) / ks
        total += 0.5 * (v(lo) + v(hi)) * d
    return total


@pytest.mark.parametrize("K,ks,sigma", [(29, 0.5, 2.0), (29, 2.0, 8.0), (15, 4.0, 6.0),
                                        (57, 0.3, 1.5), (3, 1.7, 1.0), (1, 2.0, 1.0)])
def test_weights_from_the_segment_table(hw, K, ks, sigma):
    rng = np.random.default_rng(K)
    half = (K - 1) // 2
    f = np.float32
    x = (np.arange(K) - half) * ks
    taps = np.exp(-0.5 * (x / sigma) ** 2).astype(f)
    n = 400_000
    edge = (half + 1) * ks
    c = rng.uniform(-1.1, 1.1, n) * edge
    c[: n // 4] = rng.choice([-1, 1], n // 4) * (edge - ks * rng.uniform(0, 1, n // 4))
    w = ks * 10.0 ** rng.uniform(-3, np.log10(2 * (half + 2)), n)
    x0, x1 = (c - w / 2).astype(f), (c + w / 2).astype(f)
    x0[::97] = np.round(x0[::97] / f(ks)) * f(ks)
    x1[::89] = np.round(x1[::89] / f(ks)) * f(ks)
    out = np.zeros((n, 2), f)
    p = lambda a: a.ctypes.data_as(C.c_void_p)
    hw.hw_psf(p(taps), K, ks, n, p(x0), p(x1), p(out))
    ref = integral(taps, f(ks), x0.astype(np.float64), x1.astype(np.float64))
    assert (out[ref == 0] <= 1e-6 * ks).all()
    on = ref > 0
    e = np.abs(out[on].astype(np.float64) - ref[on, None]) / ref[on, None]
    for q in (50, 90, 99, 99.9):
        a, b = np.percentile(e, q, axis=0)
        print(f"K {K} ks {ks}: percentile {q}: psfWeight {a:.2e}, psfWeightTab {b:.2e}")
        assert b <= 1.05 * a + 6e-8
    l2 = np.sqrt((((out[on] - ref[on, None]) ** 2).sum(0)) / (ref[on] ** 2).sum())
    print(f"rel L2 {l2[0]:.2e} {l2[1]:.2e}")
    assert l2[1] <= 1.05 * l2[0]
    far = np.minimum(edge - np.abs(x0), edge - np.abs(x1))[on]
    wide = (far > 0.1 * ks) & ((x1 - x0)[on] > 0.1 * ks)
    print(f"inside: largest {e[wide].max(0)}")
    assert e[wide, 1].max() <= 2e-6 + 6e-8 * 10 * (half + 1)
