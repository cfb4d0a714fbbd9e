"""GPU checks of the stacked angular-spectrum propagation behind autograd's asm_prop: every field of a
stack comes out bit for bit as its own call gives it, for stacks held in one part and for strided,
conjugated and single-field inputs, and the source is left alone."""
import pytest
import torch

pytestmark = pytest.mark.gpu
LAM, P = 532e-9, 8e-6


@pytest.mark.parametrize("nb,ny,nx", [(1, 256, 256), (3, 1024, 1024), (5, 96, 140), (7, 4, 8), (2, 1024, 2048)])
@pytest.mark.parametrize("adjoint", [False, True])
def test_stack_equals_single_calls(nb, ny, nx, adjoint):
    import openol_amd as ol
    from openol_amd import ops
    g = torch.Generator().manual_seed(nb * ny + nx)
    u = torch.randn(nb, ny, nx, dtype=torch.complex64, generator=g).cuda()
    keep, out = u.clone(), torch.empty_like(u)
    ops.asm_batch(u, out, P, P, LAM, 0.03, True, adjoint)
    assert torch.equal(u, keep)
    for k in range(nb):
        one = u[k].clone()
        ol.AsmProp(one, ny, nx, P, P, LAM, 0.03, bandlimit=True, adjoint=adjoint)
        assert torch.equal(torch.view_as_real(one), torch.view_as_real(out[k]))


def test_strided_and_conjugated_stacks():
    from openol_amd import autograd as ag
    g = torch.Generator().manual_seed(5)
    u = torch.randn(2, 3, 128, 64, dtype=torch.complex64, generator=g).cuda()
    want = ag.asm_prop(u.conj().resolve_conj().transpose(-1, -2).contiguous(), P, P, LAM, 0.01)
    got = ag.asm_prop(u.conj().transpose(-1, -2), P, P, LAM, 0.01)
    assert got.shape == (2, 3, 64, 128) and torch.equal(got.resolve_conj(), want.resolve_conj())
