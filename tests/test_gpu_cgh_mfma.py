"""The direct Fresnel CGH as an FP16 hi + lo split product on the matrix cores.

Bar: each factor is off by at most 2^-24 (split) plus the hardware sine / cosine's
1.3e-7, twice; a chain of n <= 4096 points adds 3 n / 8 rounded times, a random walk of
sqrt(3 n / 8) 2^-24 / 2 = 1.2e-6.  Together below 2e-6; the bar is 3e-6.
"""
import numpy as np
import pytest
import torch

import olref
from openol_amd import synth

pytestmark = pytest.mark.gpu
LAM, P = 532e-9, 8e-6


def ol():
    import openol_amd
    return openol_amd


def cloud(n, seed, ny, nx, amp=1.0):
    pts = synth.random_points(n, seed=seed, xmax=nx * P, ymax=ny * P, zmin=0.05, zmax=0.2)
    pts["amp"] = (pts["amp"] * amp).astype(np.float32)
    return pts


def obj(p, sl=slice(None)):
    return ol().Object(*(p[k][sl] for k in ("x", "y", "z", "amp", "phase")))


def rel(a, b):
    return (torch.linalg.norm(a.to(torch.complex128) - b) / torch.linalg.norm(b)).item()


# one point past and short of a stage (16 points), a tile (256 / 128 rows, 128 columns) and a
# chain (4096 points); few tiles (K slices) and many; one row
@pytest.mark.parametrize("ny,nx,n", [(256, 128, 112), (257, 129, 113), (255, 127, 4097), (1, 300, 500),
                                     (130, 1, 4096), (640, 1000, 10001), (1030, 1300, 300)])
def test_direct_fresnel_matches_fp64(ny, nx, n):
    p = cloud(n, n, ny, nx)
    U = torch.empty((ny, nx), dtype=torch.complex64, device="cuda")
    D = torch.empty((ny, nx), dtype=torch.complex128, device="cuda")
    ol().Cgh(obj(p), U, ny, nx, P, P, LAM)
    ol().CghFP64(obj(p), D, ny, nx, P, P, LAM)
    assert rel(U, D) < 3e-6
    V = torch.empty_like(U)
    ol().Cgh(obj(p), V, ny, nx, P, P, LAM)
    assert torch.equal(U, V)
    ol().Cgh(obj(p), V, ny, nx, P, P, LAM, accumulate=True)
    assert rel(V, 2 * D) < 3e-6


@pytest.mark.parametrize("amp", [-1.0, 1e-30, 3e30, 0.0])
def test_direct_fresnel_amplitude_range(amp):
    """The largest amplitude is divided out before the FP16 split."""
    ny, nx, n = 100, 150, 400
    p = cloud(n, 3, ny, nx)
    U = torch.empty((ny, nx), dtype=torch.complex64, device="cuda")
    ol().Cgh(obj(p), U, ny, nx, P, P, LAM)
    p["amp"] = p["amp"] * np.float32(amp)
    V = torch.empty_like(U)
    ol().Cgh(obj(p), V, ny, nx, P, P, LAM)
    want = U.to(torch.complex128) * float(np.float32(amp))
    assert torch.count_nonzero(V).item() == 0 if amp == 0.0 else rel(V, want) < 3e-6


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_direct_fresnel_nonfinite_amplitude(bad):
    """One infinite or NaN amplitude: every pixel holds what the point's term makes of it."""
    ny, nx, n = 70, 90, 300
    p = cloud(n, 5, ny, nx)
    p["amp"][17] = bad
    U = torch.zeros((ny, nx), dtype=torch.complex64, device="cuda")
    ol().Cgh(obj(p), U, ny, nx, P, P, LAM)
    v = torch.view_as_real(U)
    assert not torch.isfinite(v).any()
    assert torch.isnan(v).all() or not np.isnan(bad)
