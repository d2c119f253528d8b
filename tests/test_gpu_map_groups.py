"""A cube whose segment maps pass their limit (16 GiB) renders its frames in groups: the device memory the call takes stays
within the limit, and every frame is the frame rendered alone, bit for bit. 128 x 128 points x 1024 samples in FP64 take
0.34 GB of maps a frame: 61 frames of one frequency (groups of 31 and 30), 31 frames of two (one group each), in index
order and in the queue's cost order."""
import math

import numpy as np
import pytest
import torch

import kerrsplat_amd as K
from kerrsplat_amd import synthetic as syn

pytestmark = pytest.mark.gpu

A, TH, N, LIMIT = 0.7, math.radians(40.0), 1024, 1 << 34


@pytest.mark.parametrize("nt,nus,nmax", [(61, [230e9], -1), (31, [230e9, 86e9], 1)])
def test_grouped_cube_equals_its_frames(nt, nus, nmax):
    cam = K.Camera((-12.0, 12.0), (-12.0, 12.0), (128, 128))
    L = syn.length_unit()
    m = K.Model(syn.thermal_splats(5, A, 6, single_frame=False))
    c = K.GeodesicCache(cam, N, store_samples=True)
    K.regenerate(c, A, TH, marcher=K.Recurrence(64))
    times = [2.0 * k for k in range(nt)]
    kw = dict(nmax=nmax, slab=0.5)
    alone = {(it, q): np.array(K.polarized_cube(c, m, [times[it]], [nus[q]], L, **kw)).reshape(-1, 4, order="F")
             for it in (0, nt // 2, nt // 2 + 1, nt - 1) for q in range(len(nus))}
    free = torch.cuda.mem_get_info()[0]
    print(f"{nt} frames x {len(nus)}", flush=True)
    cube = np.array(K.polarized_cube(c, m, times, nus, L, **kw))
    took = free - torch.cuda.mem_get_info()[0]
    assert took <= LIMIT + (1 << 29), took           # the maps and the images
    K.tuning(c, queue=True)
    ordered = [np.array(K.polarized_cube(c, m, times, nus, L, **kw)) for _ in range(2)]
    assert np.array_equal(ordered[0], cube) and np.array_equal(ordered[1], cube)
    assert np.abs(cube).max() > 0
    for (it, q), im in alone.items():
        assert np.array_equal(cube[..., it, q, :].reshape(-1, 4, order="F"), im), (it, q)
