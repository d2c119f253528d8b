"""The transfer over stored samples at the edges of its packing, against the oracle: one splat, fewer splats than lanes,
the counts around a block of 64 candidates and around the per-tile cull (its smallest count and past its largest, 1024),
samples per ray shorter than a slice and no multiple of it, screens of no multiple of a wavefront. Bars of the other
parity tests: images within 1e-10 of the peak Stokes I in FP64 (both sides sum a sample's contributions in splat order),
1e-4 mixed. Compared on the rays whose marched samples agree with the oracle's to 1e-10: with an odd N the quadrature of
a scattering ray can differ by 1e-8 in t between the two marches (a sample on the turning point), which the transfer of
either would show."""
import math

import numpy as np
import pytest

import kerrsplat_amd as K
from kerrsplat_amd import synthetic as syn

pytestmark = pytest.mark.gpu

A, TH = 0.8, math.radians(50.0)


@pytest.mark.parametrize("ns,size,N", [(1, (6, 5), 3), (9, (10, 7), 33), (63, (8, 9), 41), (64, (8, 8), 64), (65, (12, 11), 90), (1024, (6, 7), 50),
                                       (1025, (6, 7), 50)])
def test_packed_pairs_vs_oracle(oracle, ns, size, N):
    cam = K.Camera((-9.0, 9.0), (-8.0, 8.0), size)
    L = syn.length_unit()
    P = syn.thermal_splats(4, A, ns, single_frame=False)
    P[12] -= math.log(max(ns / 32.0, 1.0))                   # about as thick whatever the count
    c = K.GeodesicCache(cam, N, store_samples=True)
    K.regenerate(c, A, TH, marcher=K.Recurrence(64))
    print(f"{ns} splats, {size}, N = {N}", flush=True)
    img = K.polarized_image(c, P, 7.0, 230e9, L)
    ref = oracle.polarized_image(A, TH, cam.alphas, cam.betas, N, P, 7.0, 230e9, L)[0].reshape(cam.size + (4,), order="F")
    peak = np.abs(ref[..., 0]).max()
    assert peak > 0
    dev, ora = K.samples(c), oracle.samples(A, TH, cam.alphas, cam.betas, N)
    perm = c.perm_host - 1
    ok = (dev["flags"] & 1) > 0
    near = np.all([np.where(ok, np.abs(dev[k] - ora[k][perm]), 0.0).max(axis=1) <= 1e-10 for k in ("t", "r", "theta", "phi")], axis=0)
    same = np.zeros(cam.npix, dtype=bool)
    same[perm] = near
    assert same.mean() >= 0.9
    same = same.reshape(size, order="F")
    assert np.abs(img - ref)[same].max() <= 1e-10 * peak
    K.precision(c, "mixed")
    img32 = K.polarized_image(c, P, 7.0, 230e9, L)
    assert np.abs(img32 - ref).max() <= 1e-4 * peak
