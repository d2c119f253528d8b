"""A cache without stored samples marches its pixels in tiles and runs their frames in groups; the result is that of a
cache with stored samples (the same march and transfer, other slices: rounding of the Stokes sums, 1e-12 of the peak).
60 x 40 points x 8000 samples: three tiles, the last one ragged, and five frames in two groups; one tile of one point."""
import math

import numpy as np
import pytest

import kerrsplat_amd as K
from kerrsplat_amd import synthetic as syn

pytestmark = pytest.mark.gpu

A, TH = 0.85, math.radians(35.0)


@pytest.mark.parametrize("size,N,times,nus,nmax", [((60, 40), 8000, [0.0, 4.0, 8.0, 12.0, 16.0], [230e9, 86e9], -1), ((60, 40), 8000, [3.0], [230e9], 1),
                                                   ((1, 1), 70, [0.0], [230e9], -1)])
def test_tiles_equal_stored_samples(size, N, times, nus, nmax):
    cam = K.Camera((-8.0, 8.0), (-6.0, 6.0), size) if size != (1, 1) else K.Camera((4.5, 4.5), (1.2, 1.2), size)
    L = syn.length_unit()
    m = K.Model(syn.thermal_splats(5, A, 6, single_frame=False))
    thin = syn.thin_splats(5, A, 6)
    out = []
    for store, march in ((True, K.Recurrence(64)), (False, K.Fused(64))):
        c = K.GeodesicCache(cam, N, store_samples=store)
        K.regenerate(c, A, TH, marcher=march)
        print(f"{size}, N = {N}, stored {store}", flush=True)
        out.append((K.polarized_cube(c, m, times, nus, L, nmax=nmax, slab=0.5), K.thin_image(c, thin, 2.0)) + K.residuals(c))
    (cube0, thin0, rt0, rp0), (cube1, thin1, rt1, rp1) = out
    peak = np.abs(cube0[..., 0]).max()
    assert peak > 0
    assert np.abs(cube1 - cube0).max() <= 1e-12 * peak
    assert np.abs(thin1 - thin0).max() <= 1e-12 * np.abs(thin0).max()
    assert np.array_equal(rt0, rt1) and np.array_equal(rp0, rp1)
