"""GPU checks that a device allocation which fails leaves no error behind: callers then take a form that needs
no workspace, or report the failure themselves, and the next launch check must not report it again; and that the
forms with a smaller workspace, or none, give the same field."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
HUGE = ctypes.c_size_t(1 << 50)  # more than any device has


def refuse_reserve():
    from openol_amd import _lib
    buf = (ctypes.c_char * 256)()  # a DevBuf that holds nothing
    return getattr(_lib.load(), "_ZN3olx6DevBuf7reserveEm")(buf, HUGE)


def refuse_alloc():
    from openol_amd import _lib
    p = ctypes.c_void_p()
    return _lib.call("olx_dev_alloc", 0, ctypes.byref(p), HUGE)


@pytest.mark.parametrize("refuse", [refuse_reserve, refuse_alloc])
def test_next_call_succeeds(refuse):
    import openol_amd as ol
    from openol_amd import _lib
    u = torch.ones(16, 16, dtype=torch.complex64, device="cuda")
    ol.AsmProp(u, 16, 16, 8e-6, 8e-6, 532e-9, 0.0)
    assert refuse() == _lib.ENOMEM
    ol.AsmProp(u, 16, 16, 8e-6, 8e-6, 532e-9, 0.0)


LAM, P = 532e-9, 8e-6


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


def cloud(n, ny, nx):
    import openol_amd as ol
    r = np.random.default_rng(n)
    return ol.Object(r.uniform(0, nx * P, n), r.uniform(0, ny * P, n), r.uniform(0.1, 0.2, n),
                     r.uniform(0.2, 3.0, n), r.uniform(0, 6.28, n))


@pytest.mark.parametrize("form,n,ny,nx,mib", [("exact", 1000, 700, 700, 1), ("exact", 5000, 192, 160, 0.25),
                                              ("fresnel", 2000, 300, 300, 4), ("fresnel", 5000, 192, 160, 0.25),
                                              ("layered", 2000, 1000, 1000, 20)])
def test_cgh_without_planes(limit, form, n, ny, nx, mib):
    import openol_amd as ol
    o = cloud(n, ny, nx)
    U, V = (torch.empty(ny, nx, dtype=torch.complex64, device="cuda") for _ in range(2))

    def call(out):
        if form == "layered":
            return ol.CghLayered(o, out, ny, nx, P, P, LAM, 8, 0.1, 0.2)
        return ol.Cgh(o, out, ny, nx, P, P, LAM, exact_r=form == "exact")

    limit(int(mib * 2 ** 20))
    call(U)
    limit(0)
    call(V)
    assert not bool((U == V).all())  # another form
    assert float(torch.linalg.vector_norm(U - V) / torch.linalg.vector_norm(V)) < 1e-5
    limit(int(mib * 2 ** 20))  # frees what passes the bound
    V.zero_()
    call(V)
    assert torch.equal(torch.view_as_real(U), torch.view_as_real(V))


@pytest.mark.parametrize("ny,nx", [(512, 512), (300, 250), (1024, 1024)])
def test_stack_field_by_field(limit, ny, nx):
    import openol_amd as ol
    from openol_amd import _lib, ops
    g = torch.Generator().manual_seed(nx)
    u = torch.randn(5, ny, nx, dtype=torch.complex64, generator=g).cuda()
    a, b = torch.empty_like(u), torch.empty_like(u)
    ops.asm_batch(u, a, P, P, LAM, 0.03, True)
    limit(int(16 * ny * nx * 1.2))  # one field's intermediate, with the padding of its columns
    ops.asm_batch(u, b, P, P, LAM, 0.03, True)
    assert torch.equal(torch.view_as_real(a), torch.view_as_real(b))
    limit(16 * ny * nx // 2)
    with pytest.raises(_lib.OlxError):
        ops.asm_batch(u, b, P, P, LAM, 0.03, True)
