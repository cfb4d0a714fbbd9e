"""GPU checks of the exact-r hologram on the matrix cores, against its FP64 kernel: sides around the 64 x 64
tile, point counts around the 64 of a block and past the 4096 of an accumulator, off-axis clouds,
clouds whose points are all or partly left to the per-pixel kernel, and the other outputs.

Bars: a phase is rounded at most four times at below 2 cycles (6e-8 to 1.2e-7 cycles each, 1.5e-6 rad),
the hardware sine adds about 1e-6, so 5e-6 for far clouds; the per-pixel form of near points carries
phases of hundreds of cycles in FP32, for which the other direct CGH checks allow 1e-4."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
LAM, P = 532e-9, 8e-6


def cloud(n, ny, nx, z0, z1, seed, off=0.0):
    import openol_amd as ol
    r = np.random.default_rng(seed)
    return ol.Object(r.uniform(0, nx * P, n) + off, r.uniform(0, ny * P, n) - off, r.uniform(z0, z1, n),
                     r.uniform(0.2, 3.0, n), r.uniform(0, 6.28, n))


def rel(a, b):
    return float(torch.linalg.vector_norm(a.to(torch.complex128) - b) / torch.linalg.vector_norm(b))


@pytest.mark.parametrize("n,ny,nx,z0,z1,off,bar", [
    (2000, 65, 130, 0.1, 0.2, 0.0, 5e-6), (1025, 63, 64, 0.1, 0.2, 0.0, 5e-6), (1023, 257, 1, 0.15, 0.15, 0.0, 5e-6),
    (8300, 200, 129, 0.1, 0.2, 0.0, 5e-6), (700, 512, 640, 0.1, 0.3, 8e-3, 5e-6),
    (64, 2048, 2048, 0.1, 0.2, 0.0, 5e-6), (3000, 300, 300, 0.002, 0.2, 0.0, 1e-4),
    (1500, 256, 256, 0.001, 0.004, 0.0, 1e-4)])
def test_exact_against_fp64(n, ny, nx, z0, z1, off, bar):
    import openol_amd as ol
    o = cloud(n, ny, nx, z0, z1, n + nx, off)
    ref = torch.empty(ny, nx, dtype=torch.complex128, device="cuda")
    ol.CghFP64(o, ref, ny, nx, P, P, LAM, exact_r=True)
    U = torch.empty(ny, nx, dtype=torch.complex64, device="cuda")
    ol.Cgh(o, U, ny, nx, P, P, LAM, exact_r=True)
    assert rel(U, ref) < bar
    V = U.clone()
    ol.Cgh(o, V, ny, nx, P, P, LAM, exact_r=True, accumulate=True)
    assert rel(V, 2 * ref) < bar
    W, ph, am = torch.empty_like(U), torch.empty(ny, nx, device="cuda"), torch.empty(ny, nx, device="cuda")
    ol.Cgh(o, W, ny, nx, P, P, LAM, exact_r=True, phase_out=ph, amp_out=am)
    assert torch.equal(torch.view_as_real(W), torch.view_as_real(U))
    assert torch.allclose(am, W.abs(), rtol=1e-5) and torch.allclose(ph, W.angle(), atol=1e-5)


def test_amplitudes_beyond_fp16():
    import openol_amd as ol
    r = np.random.default_rng(3)
    n, ny, nx = 1500, 128, 128
    xyz = r.uniform(0, nx * P, n), r.uniform(0, ny * P, n), r.uniform(0.1, 0.2, n)
    a, ph = r.uniform(0.5, 1.0, n), r.uniform(0, 6.28, n)
    U, V = (torch.empty(ny, nx, dtype=torch.complex64, device="cuda") for _ in range(2))
    ol.Cgh(ol.Object(*xyz, a, ph), U, ny, nx, P, P, LAM, exact_r=True)
    for s in (2.0 ** 40, 2.0 ** -40):
        ol.Cgh(ol.Object(*xyz, a * s, ph), V, ny, nx, P, P, LAM, exact_r=True)
        assert torch.equal(torch.view_as_real(V), torch.view_as_real(U) * s)
    a[7] = np.inf
    ol.Cgh(ol.Object(*xyz, a, ph), V, ny, nx, P, P, LAM, exact_r=True)
    assert not torch.isfinite(torch.view_as_real(V)).any()


@pytest.mark.parametrize("exact", [True, False])
def test_under_capture(exact):
    """A captured call takes the kernels without workspace: replays stay right after larger calls."""
    import openol_amd as ol
    n, ny, nx = 1200, 192, 160
    o, big = cloud(n, ny, nx, 0.1, 0.2, 9), cloud(3000, 700, 700, 0.1, 0.2, 10)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        want = torch.empty(ny, nx, dtype=torch.complex64, device="cuda")
        ol.Cgh(o, want, ny, nx, P, P, LAM, exact_r=exact)
        U, W = torch.zeros_like(want), torch.empty(700, 700, dtype=torch.complex64, device="cuda")
        g = torch.cuda.CUDAGraph()
        s.synchronize()
        with torch.cuda.graph(g, stream=s):
            ol.Cgh(o, U, ny, nx, P, P, LAM, exact_r=exact)
        for _ in range(3):
            U.zero_()
            ol.Cgh(big, W, 700, 700, P, P, LAM, exact_r=exact)
            s.synchronize()
            g.replay()
            s.synchronize()
            assert rel(U, want.to(torch.complex128)) < 1e-5
