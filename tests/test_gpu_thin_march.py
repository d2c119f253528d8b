"""Thin images of caches without stored samples: few splats are summed inside the march, more through a tile's samples; on
either side of the rule (2 splats on a screen of one tile, 6 on a larger one) the image is that of a cache with stored samples
(the same march and sums in another order: 1e-12 of the peak) and the anchor residuals are the same. Rays with alpha = 0
exactly (the middle column of an odd screen), whose phi is NaN, are left out."""
import math

import numpy as np
import pytest

import kerrsplat_amd as K
from kerrsplat_amd import synthetic as syn

pytestmark = pytest.mark.gpu

A, TH = 0.85, math.radians(35.0)


@pytest.mark.parametrize("size,N,counts", [((60, 40), 8000, (6, 7)), ((13, 11), 77, (0, 1, 2, 3)), ((1, 1), 70, (2, 3))])
def test_few_splats_equal_stored_samples(size, N, counts):
    cam = K.Camera((-8.0, 8.0), (-6.0, 6.0), size) if size != (1, 1) else K.Camera((4.5, 4.5), (1.2, 1.2), size)
    caches = []
    for store, march in ((True, K.Recurrence(64)), (False, K.Fused(64))):
        c = K.GeodesicCache(cam, N, store_samples=store)
        K.regenerate(c, A, TH, marcher=march)
        caches.append(c)
    for ns in counts:
        P = syn.thin_splats(5, A, max(ns, 1))[:, :ns]
        print(f"{size}, N = {N}, {ns} splats", flush=True)
        ref, got = (np.array(K.thin_image(c, P, 2.0)) for c in caches)
        ref, got = (im[np.abs(np.reshape(cam.alphas, cam.size, order="F")) > 1e-12] for im in (ref, got))
        assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()
        assert ns == 0 or np.abs(ref).max() > 0
        for a, b in zip(K.residuals(caches[0]), K.residuals(caches[1])):
            assert np.array_equal(a, b, equal_nan=True)
