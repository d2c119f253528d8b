"""A captured fit iteration on the mixed path follows a new march: the element adjoints read an FP32 copy of the samples,
which is made again after the march precision changes (chi2 and gradients bit for bit the eager iteration's)."""
import math

import numpy as np
import pytest

import kerrsplat_amd as K
from kerrsplat_amd import synthetic as syn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_replay_after_a_march(precision):
    a = 0.9
    cam = K.Camera((-9.0, 9.0), (-9.0, 9.0), (40, 36))
    c = K.GeodesicCache(cam, 256, store_samples=True)
    K.regenerate(c, a, math.radians(45.0), marcher=K.Recurrence(64))
    K.precision(c, precision)
    L = syn.length_unit()
    P = syn.thermal_splats(1, a, 10, single_frame=False)
    m = K.Model(P)
    truth = np.array(K.polarized_cube(c, m, [0.0], [230e9], L))
    sigma = [0.05 * np.abs(truth[..., 0]).max()] * 4
    data = 1.1 * truth
    graph = K.FitGraph(c, [0.0], [230e9], L, image=(data, sigma))
    for march in ("fp64", "mixed", "fp64"):
        print(f"{precision}, march {march}", flush=True)
        K.march_precision(c, march)
        K.march(c)
        chi_g, g_g = graph.step(m, P)
        K.gradient_forward(c, m, [0.0], [230e9], L, copy=False)
        chi = K.image_chi2_seed(c, 0, data[:, :, 0, 0, :], sigma)
        g = np.zeros(m.grad_shape, order="F")
        K.gradient_reverse(c, m, g)
        assert np.abs(g).max() > 0
        assert chi_g == chi and np.array_equal(g_g, g), march
