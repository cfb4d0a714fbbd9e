"""GPU checks of the cell lists behind WRPStep1: point counts around the 512 of a binning block, planes
of one cell, of ragged cells, of 64 cells and more (tiles grouped by cell) and of more than 1024
cells of 8 x 8 tiles (cells of 16 x 16).  Pixels near the points against the FP64 oracle, to the 1e-5
of the other WRP checks; the sum over points is one launch of the same order, so two runs are alike."""
import numpy as np
import pytest
import torch

import olref

pytestmark = pytest.mark.gpu
LAM, P = 532e-9, 8e-6


@pytest.mark.parametrize("square", [False, True])
@pytest.mark.parametrize("n,ny,nx", [(1, 16, 16), (511, 100, 2000), (512, 130, 129), (513, 1040, 1048),
                                     (1025, 4112, 4200)])
def test_cells(n, ny, nx, square):
    import openol_amd as ol
    rng = np.random.default_rng(n)
    x, y = rng.uniform(0, nx * P, n), rng.uniform(0, ny * P, n)
    z = rng.uniform(0.151, 0.155, n)
    x[: n // 4] = rng.integers(0, nx // 16 + 1, n // 4) * 16 * P   # on tile and cell borders
    U = torch.empty((ny, nx), dtype=torch.complex64, device="cuda")
    V = torch.empty_like(U)
    obj = ol.Object(x, y, z)
    ol.WRPStep1(obj, U, ny, nx, P, LAM, 0.15, square=square)
    ol.WRPStep1(obj, V, ny, nx, P, LAM, 0.15, square=square)
    assert torch.equal(U, V)
    k = rng.integers(0, n, 800)
    ph = np.clip((y[k] / P).astype(int) + rng.integers(-20, 21, 800), 0, ny - 1)
    pw = np.clip((x[k] / P).astype(int) + rng.integers(-20, 21, 800), 0, nx - 1)
    ref = olref.wrp_pixels(x, y, z, ph, pw, P, LAM, 0.15, square=square)
    got = U.cpu().numpy()[ph, pw]
    assert np.linalg.norm(got - ref) < 1e-5 * np.linalg.norm(ref)
