"""The element adjoints' work list at its edges, against the oracle's gradient: one splat, the counts around a 64-bit
mask word, fewer work units than XCDs, a last unit that is partly filled (N no multiple of the unit's 32 samples, pixels
no multiple of 64), a splat that reaches nothing, two frames. Bars of the other parity tests: 1e-9 of the largest entry in
FP64, 1e-3 mixed. Rays whose marched samples differ from the oracle's by more than 1e-10 carry no seed on either side (the
quadratures of a near-critical ray's t can differ by 1e-9, which a gradient of either would show)."""
import math

import numpy as np
import pytest

import kerrsplat_amd as K
from kerrsplat_amd import synthetic as syn

pytestmark = pytest.mark.gpu

A, TH = 0.7, math.radians(55.0)


@pytest.mark.parametrize("ns,size,N,nt", [(1, (5, 4), 32, 1), (5, (8, 8), 34, 2), (64, (8, 7), 66, 1), (65, (10, 9), 48, 2), (130, (6, 8), 40, 1)])
def test_work_list_vs_oracle(oracle, ns, size, N, nt):
    cam = K.Camera((-9.0, 9.0), (-8.0, 8.0), size)
    L = syn.length_unit()
    P = syn.thermal_splats(6, A, ns, single_frame=False)
    P[12] -= math.log(max(ns / 32.0, 1.0))
    if ns > 1:
        P[0:3, ns // 2] = (300.0, 200.0, 100.0)              # outside every ray's samples: no block, a zero column
    times = [3.0 + 9.0 * k for k in range(nt)]
    c = K.GeodesicCache(cam, N, store_samples=True)
    K.regenerate(c, A, TH, marcher=K.Recurrence(64))
    ds = np.random.default_rng(ns).normal(size=size + (nt, 1, 4))
    dev, ora = K.samples(c), oracle.samples(A, TH, cam.alphas, cam.betas, N)
    perm, ok = c.perm_host - 1, (dev["flags"] & 1) > 0
    same = np.zeros(cam.npix, dtype=bool)
    same[perm] = np.all([np.where(ok, np.abs(dev[k] - ora[k][perm]), 0.0).max(axis=1) <= 1e-10 for k in ("t", "r", "theta", "phi")], axis=0)
    assert same.mean() >= 0.7                                 # (a 5-column screen loses its alpha = 0 column)
    ds *= same.reshape(size, order="F")[:, :, None, None, None]
    print(f"{ns} splats, {size}, N = {N}, {nt} frames", flush=True)
    g, _ = K.polarized_gradient(c, P, times, [230e9], L, ds)
    ref = sum(oracle.polarized_gradient(A, TH, cam.alphas, cam.betas, N, P, t, 230e9, L, ds[:, :, k, 0, :].reshape(cam.npix, 4, order="F"))[0]
              for k, t in enumerate(times))
    gmax = np.abs(ref).max()
    assert gmax > 0
    assert np.abs(g - ref).max() <= 1e-9 * gmax
    if ns > 1:
        assert np.all(g[:, ns // 2] == 0.0)
    K.precision(c, "mixed")
    g32, _ = K.polarized_gradient(c, P, times, [230e9], L, ds)
    assert np.abs(g32 - ref).max() <= 1e-3 * gmax
