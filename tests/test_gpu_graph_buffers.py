"""GPU checks that a captured graph keeps the buffers it was captured with: its replays stay right after eager
calls that need larger ones, and a captured call finds room that the same call before it made."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
LAM, P = 532e-9, 8e-6


@pytest.fixture
def fresh(monkeypatch):
    """A library context whose buffers hold nothing yet."""
    from openol_amd import _lib
    mine = {}
    monkeypatch.setattr(_lib, "_ctx", mine)
    yield
    torch.cuda.synchronize()
    for c in mine.values():
        _lib.load().olx_ctx_destroy(c)


def cloud(n, ny, nx, seed):
    import openol_amd as ol
    r = np.random.default_rng(seed)
    return ol.Object(r.uniform(0, nx * P, n), r.uniform(0, ny * P, n), r.uniform(0.1, 0.2, n),
                     r.uniform(0.2, 3.0, n), r.uniform(0, 6.28, n))


def field(*shape):
    return torch.empty(shape, dtype=torch.complex64, device="cuda")


def check(call, out, later, bar=1e-5, warm=True):
    """call fills out; replays of its graph stay the same while later runs between them."""
    from openol_amd import _lib
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        _lib.ctx()  # bound to s before the capture
        if warm:
            call()
            want = out.clone()
        g = torch.cuda.CUDAGraph()
        s.synchronize()
        with torch.cuda.graph(g, stream=s):
            call()
        first = None
        for _ in range(3):
            out.zero_()
            s.synchronize()
            g.replay()
            s.synchronize()
            first = out.clone() if first is None else first
            assert torch.equal(torch.view_as_real(out), torch.view_as_real(first))
            later()
        if not warm:
            call()
            want = out
        d = torch.linalg.vector_norm(first - want) / torch.linalg.vector_norm(want)
        assert float(d) < bar


def large_calls():
    import openol_amd as ol
    o, U = cloud(20000, 900, 1100, 2), field(900, 1100)
    for ex in (True, False):
        ol.Cgh(o, U, 900, 1100, P, P, LAM, exact_r=ex)
    ol.CghLayered(o, U, 900, 1100, P, P, LAM, 8, 0.1, 0.2)


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("warm", [True, False])
def test_direct_cgh_of_sliced_points(fresh, exact, warm):
    import openol_amd as ol
    o, U = cloud(5000, 192, 160, 1), field(192, 160)
    check(lambda: ol.Cgh(o, U, 192, 160, P, P, LAM, exact_r=exact), U, large_calls, warm=warm)


@pytest.mark.parametrize("precision", ["f16", "bf16x3"])
def test_layered_cgh(fresh, precision):
    import openol_amd as ol
    o, U = cloud(3000, 300, 400, 3), field(300, 400)
    check(lambda: ol.CghLayered(o, U, 300, 400, P, P, LAM, 8, 0.1, 0.2, precision=precision), U, large_calls)


@pytest.mark.parametrize("ny,nx", [(256, 256), (1024, 1024), (300, 250)])
@pytest.mark.parametrize("nb", [1, 3])
def test_propagation(fresh, ny, nx, nb):
    import openol_amd as ol
    from openol_amd import ops
    r = torch.Generator().manual_seed(4)
    u, out = torch.randn(nb, ny, nx, dtype=torch.complex64, generator=r).cuda(), field(nb, ny, nx)
    big, to = field(8, ny, nx).zero_(), field(8, ny, nx)
    check(lambda: ops.asm_batch(u, out, P, P, LAM, 0.03, True), out,
          lambda: ops.asm_batch(big, to, P, P, LAM, 0.03, True), bar=1e-9)


def test_tables_of_a_graph_are_not_evicted(fresh):
    import openol_amd as ol
    r = torch.Generator().manual_seed(6)
    src, u = torch.randn(96, 120, dtype=torch.complex64, generator=r).cuda(), field(96, 120)
    w = field(16, 16).zero_()

    def call():
        u.copy_(src)
        ol.FresnelProp(u, 96, 120, P, P, LAM, 0.03)

    def later():  # more tables than a context keeps
        for k in range(80):
            ol.FresnelProp(w, 16, 16, P, P, LAM, 0.01 + 1e-4 * k)

    check(call, u, later, bar=1e-9)
