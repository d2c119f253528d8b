"""A captured fit iteration keeps its own order of the work queue: eager renders of other shapes between the replays, which
leave other orders on the cache, change nothing (chi2 and gradients bit for bit those of the first replay)."""
import math

import numpy as np
import pytest

import kerrsplat_amd as K
from kerrsplat_amd import synthetic as syn

pytestmark = pytest.mark.gpu

A, TH = 0.9, math.radians(45.0)
TIMES, NUS = [0.0, 20.0], [230e9, 345e9]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_replay_after_other_shapes(precision):
    cam = K.Camera((-12.0, 12.0), (-12.0, 12.0), (40, 36))
    c = K.GeodesicCache(cam, 160, store_samples=True)
    K.regenerate(c, A, TH, marcher=K.Recurrence(64))
    K.precision(c, precision)
    L = syn.length_unit()
    P = syn.thermal_splats(1, A, 10, single_frame=False)
    m = K.Model(P)
    truth = np.array(K.polarized_cube(c, m, TIMES, NUS, L))
    sigma = [0.05 * np.abs(truth[..., 0]).max()] * 4
    K.tuning(c, queue=True)
    graph = K.FitGraph(c, TIMES, NUS, L, image=(1.1 * truth, sigma))
    chi0, g0 = graph.step(m, P)
    assert chi0 > 0 and np.abs(g0).max() > 0
    for times in ([0.0], [0.0, 5.0], [3.0]):
        print(f"{precision}: {len(times)} frames between the replays", flush=True)
        for _ in range(2):                       # the second launch of a shape has the order of the first
            K.polarized_cube(c, m, times, NUS[:1], L)
        chi, g = graph.step(m, P)
        assert chi == chi0 and np.array_equal(g, g0), times
    assert graph.info()["captures"] == 1
