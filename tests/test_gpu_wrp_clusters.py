"""GPU checks of WRPStep1's tile sums for crowded tiles: clusters of points, one in each cell of 8 x 8 tiles, so
that a tile collects more points than its work-group has threads before its cell's list ends, in planes whose tiles
take 64, 128 and 256 threads; and one cluster that holds the whole cloud.  Pixels near the points against the FP64
oracle, to the 1e-5 of the other WRP checks."""
import numpy as np
import pytest
import torch

import olref

pytestmark = pytest.mark.gpu
LAM, P = 532e-9, 8e-6


# points a cluster, its side in pixels, the plane, one cluster every `step` pixels
@pytest.mark.parametrize("square", [False, True])
@pytest.mark.parametrize("m,side,n,step", [(150, 10, 4096, 128), (200, 24, 2048, 128), (700, 16, 1024, 128),
                                           (3000, 40, 512, 512), (20000, 50, 2048, 2048)])
def test_clusters(m, side, n, step, square):
    import openol_amd as ol
    rng = np.random.default_rng(m)
    k = n // step
    cy, cx = (c.ravel().repeat(m) for c in np.meshgrid(np.arange(k), np.arange(k), indexing="ij"))
    x = (cx * step + step // 3 + rng.uniform(0, side, cx.size)) * P
    y = (cy * step + step // 3 + rng.uniform(0, side, cy.size)) * P
    z = rng.uniform(0.1501, 0.152, x.size)
    o = rng.permutation(x.size)
    x, y, z = x[o], y[o], z[o]
    U = torch.empty((n, n), dtype=torch.complex64, device="cuda")
    V = torch.empty_like(U)
    obj = ol.Object(x, y, z)
    ol.WRPStep1(obj, U, n, n, P, LAM, 0.15, square=square)
    ol.WRPStep1(obj, V, n, n, P, LAM, 0.15, square=square)
    assert torch.equal(U, V)
    j = rng.integers(0, x.size, 300)
    ph = np.clip((y[j] / P).astype(int) + rng.integers(-6, 7, 300), 0, n - 1)
    pw = np.clip((x[j] / P).astype(int) + rng.integers(-6, 7, 300), 0, n - 1)
    ref = olref.wrp_pixels(x, y, z, ph, pw, P, LAM, 0.15, square=square)
    got = U.cpu().numpy()[ph, pw]
    assert np.linalg.norm(got - ref) < 1e-5 * np.linalg.norm(ref)
