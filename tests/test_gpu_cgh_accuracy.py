"""GPU checks that the matrix-core forms of the direct sums are no further from FP64 than the vector kernels that
they replace, in norm and at the worst pixel: those kernels run when the workspace is bounded to nothing."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture
def limit(monkeypatch):
    """Bounds the workspaces of a library context of the test's own."""
    from openol_amd import _lib
    mine = {}
    monkeypatch.setattr(_lib, "_ctx", mine)
    yield lambda n: _lib.check(_lib.call("olx_ctx_limit_workspace", 0, ctypes.c_size_t(n)))
    torch.cuda.synchronize()
    for c in mine.values():
        _lib.load().olx_ctx_destroy(c)


def errors(limit, o, ny, nx, p, lam, exact):
    """(norm, worst pixel) relative to the field's RMS: matrix-core form, then vector kernel."""
    import openol_amd as ol
    ref = torch.empty(ny, nx, dtype=torch.complex128, device="cuda")
    ol.CghFP64(o, ref, ny, nx, p, p, lam, exact_r=exact)
    rms = ref.abs().square().mean().sqrt()
    out = []
    for bytes_ in (0, 1):
        limit(bytes_)
        U = torch.empty(ny, nx, dtype=torch.complex64, device="cuda")
        ol.Cgh(o, U, ny, nx, p, p, lam, exact_r=exact)
        d = (U.to(torch.complex128) - ref).abs() / rms
        out.append((float(d.square().mean().sqrt()), float(d.max())))
    return out


# small clouds off both axes, whose cross phase lies around the largest that the form takes (0.12 rad; 0.2 here
# where it took more): distance, pitch, wavelength, offset
@pytest.mark.parametrize("z,p,lam,d", [
    (0.01, 1e-6, 405e-9, 4.83e-3), (0.01, 3.74e-6, 405e-9, 7.4e-4), (0.01, 3.74e-6, 405e-9, 9.25e-4),
    (0.01, 3.74e-6, 633e-9, 9.46e-4), (0.03, 3.74e-6, 633e-9, 6.73e-3), (0.03, 8e-6, 633e-9, 2.64e-3),
    (0.1, 8e-6, 405e-9, 0.0147), (0.1, 8e-6, 633e-9, 0.0188)])
def test_exact_off_axis(limit, z, p, lam, d):
    import openol_amd as ol
    n, ny, nx = 600, 128, 128
    got = []
    for seed in range(8):
        r = np.random.default_rng(seed)
        o = ol.Object(r.uniform(0, 64 * p, n) + d, r.uniform(0, 64 * p, n) + d, np.full(n, z),
                      r.uniform(0.2, 3.0, n), r.uniform(0, 6.28, n))
        got.append(errors(limit, o, ny, nx, p, lam, True))
    # one cloud's worst pixel of 16384 scatters by some 20% between two sums of the same error: eight clouds' mean
    # by 7%, their norm (of 4 tiles' points) by less than 2%
    (l2, top), (vl2, vtop) = np.mean(got, axis=0)
    assert l2 <= 1.02 * vl2 and top <= 1.15 * vtop


# far and near-paraxial clouds, where the vector kernels' phases are most exact and the sums' own rounding shows:
# few and many points, small holograms (many slices) and larger ones (several runs a slice)
@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("n,ny,nx,p,z0,z1", [
    (20000, 200, 200, 3.74e-6, 0.1, 0.2), (12000, 500, 800, 3.74e-6, 0.1, 0.2), (20000, 71, 498, 8e-6, 1.5, 1.5),
    (7500, 200, 200, 2e-6, 0.2, 0.2), (7500, 512, 512, 2e-6, 0.4, 0.4), (4000, 71, 498, 3.74e-6, 0.7, 0.7),
    (3000, 1500, 2000, 3.74e-6, 0.1, 0.2)])
def test_sums(limit, n, ny, nx, p, z0, z1, exact):
    import openol_amd as ol
    r = np.random.default_rng(n + ny)
    o = ol.Object(r.uniform(0, nx * p, n), r.uniform(0, ny * p, n), r.uniform(z0, z1, n),
                  r.uniform(0.5, 1.0, n), r.uniform(0, 6.28, n))
    # their sums are over 256 points, then over those; the worst pixel as above, over at least 35,000
    (l2, top), (vl2, vtop) = errors(limit, o, ny, nx, p, 633e-9, exact)
    assert l2 <= 1.02 * vl2 and top <= 1.25 * vtop
