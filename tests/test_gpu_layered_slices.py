"""The layered CGH's GEMM at the edges of its tile heights, K slices, chunks and chains.

Bars.  FP16, BF16: as in the parity tests.  Split BF16: two factors rounded to 16 bits,
2^-17 / sqrt 3 each, 6.2e-6; the bar is 1e-5.
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


@pytest.mark.parametrize("prec,bar", [("f16", 1e-3), ("bf16", 6e-3), ("bf16x3", 1e-5)])
@pytest.mark.parametrize("ny,nx,n", [(300, 400, 20011), (65, 64, 33), (2160, 130, 5000)])
def test_layered_slices_and_chains(prec, bar, ny, nx, n):
    p = cloud(n, 70, ny, nx)
    U = torch.empty((ny, nx), dtype=torch.complex64, device="cuda")
    args = (ny, nx, P, P, LAM, 8, 0.05, 0.2)
    ol().CghLayered(obj(p), U, *args, precision=prec)
    V = torch.empty_like(U)
    ol().CghLayered(obj(p), V, *args, precision=prec, tile128=True)
    assert torch.equal(U, V)
    zl = np.array([ol().layer_depth(z, 0.05, 0.2, 8) for z in p["z"]])
    D = torch.empty((ny, nx), dtype=torch.complex128, device="cuda")
    ol().CghFP64(ol().Object(p["x"], p["y"], zl, p["amp"], p["phase"]), D, ny, nx, P, P, LAM)
    assert rel(U, D) < bar
    ol().CghLayered(obj(p), V, *args, precision=prec, accumulate=True)
    assert rel(V, 2 * U.to(torch.complex128)) < 1e-6
