"""The autotuner times what it chooses: the transfer in the two orders of its queue (whole launches of the fastest candidate,
one ratio for every pair of rows), the reverse pass once (the element adjoints have one launch form), and leaves the caller's
adjoint bit and the costs of the cache's last queue launch alone."""
import math

import numpy as np
import pytest

import kerrsplat_amd as K
from kerrsplat_amd import synthetic as syn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_autotune_times_its_choices(precision):
    cam = K.Camera((-12.0, 12.0), (-12.0, 12.0), (72, 56))
    L = syn.length_unit()
    m = K.Model(syn.thermal_splats(70, 0.8, 6, single_frame=False))
    c = K.GeodesicCache(cam, 256, store_samples=True)
    K.regenerate(c, 0.8, math.radians(50.0), marcher=K.Recurrence(64))
    K.precision(c, precision)
    times, nus = [0.0, 10.0], [230e9]
    K.tuning(c, queue=True, adjoint_queue=True)
    base = np.array(K.polarized_cube(c, m, times, nus, L))
    cost = K.queue_costs(c)
    print(precision, flush=True)
    K.autotune(c, m, times, nus, L, records=False, sample_every=2)
    assert np.array_equal(K.queue_costs(c), cost)
    choice, table = K.autotune(c, m, times, nus, L, records=True, sample_every=2, adjoint=True)
    transfer, adjoint = [r for r in table if r[0]], [r for r in table if not r[0]]
    assert len(transfer) == 24 and len(adjoint) == 1
    assert [r[2] & 1 for r in transfer] == [0, 1] * 12 and all(r[2] & 2 for r in table)
    assert all(r[3] > 0 and math.isfinite(r[3]) for r in table)
    ratio = [b[3] / a[3] for a, b in zip(transfer[::2], transfer[1::2])]
    assert max(ratio) - min(ratio) <= 1e-12
    best = min(transfer, key=lambda r: r[3])
    assert (choice["chunk"], choice["patch"], choice["queue"]) == (best[0], best[1], bool(best[2] & 1)) and choice["adjoint_queue"]
    print([f"{a[3]:.3f}" for a in transfer[::2]], ratio[0], flush=True)
    got = np.array(K.polarized_cube(c, m, times, nus, L))
    assert np.abs(got - base).max() <= (1e-12 if precision == "fp64" else 1e-5) * np.abs(base[..., 0]).max()
