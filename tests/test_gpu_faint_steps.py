"""Gradients on the mixed path over faint samples: weak fields make absorption and rotation coefficients whose squares fall
below FP32's normal range, where the step adjoint's invariants must not divide by them. Every entry is finite wherever the
FP64 path's is, and within the mixed path's bar of it (1e-3 of the largest entry, or FP32's smallest normal number where the whole
gradient is below its range)."""
import math

import numpy as np
import pytest

import kerrsplat_amd as K
from kerrsplat_amd import synthetic as syn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,rows", [("thermal", 14), ("powerlaw", 15), ("kappa", 15)])
@pytest.mark.parametrize("seed", [128, 123, 5])
def test_mixed_gradient_is_finite(kind, rows, seed):
    a = 0.95
    cam = K.Camera((-11.0, 11.0), (-11.0, 11.0), (20, 16))
    c = K.GeodesicCache(cam, 300, store_samples=True)
    K.regenerate(c, a, math.radians(60.0), marcher=K.Recurrence(64))
    gen = {"thermal": syn.thermal_splats, "powerlaw": syn.powerlaw_splats, "kappa": syn.kappa_splats}[kind]
    P = gen(seed, a, 70, single_frame=False)
    P[rows] = np.random.default_rng(seed).uniform(-35.0, -5.0, 70)
    m = K.Model(P, kind=kind)
    ds = np.random.default_rng(seed).normal(size=cam.size + (1, 1, 4))
    L = syn.length_unit()
    g64 = K.polarized_gradient(c, m, [5.0], [230e9], L, ds)[0]
    K.precision(c, "mixed")
    g32 = K.polarized_gradient(c, m, [5.0], [230e9], L, ds)[0]
    ok = np.isfinite(g64)
    assert ok.any() and np.abs(g64[ok]).max() > 0
    assert np.isfinite(g32[ok]).all(), int((~np.isfinite(g32[ok])).sum())
    assert np.abs(g32 - g64)[ok].max() <= max(1e-3 * np.abs(g64[ok]).max(), 1.2e-38)
