"""The mixed-radix propagation's transforms: every radix, one to five stages, lengths whose halves
take several butterflies a thread, padded intermediate columns, large batches in parts.

Bar: complex64 transforms round to 2^-24 a few tens of times on the way (4e-7 measured against FP64
on every path), and the transfer function's sine and cosine add 1.3e-7; 1e-6 leaves a factor two.
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


# single stages; prime powers; 5-smooth and 13-smooth products; odd lengths; 4394 and 7436 (both
# halves need more than 1024 threads at one butterfly each)
@pytest.mark.parametrize("ny,nx", [(2, 3), (5, 6), (9, 10), (11, 12), (13, 14), (15, 16), (7, 32), (121, 169),
                                   (49, 81), (125, 128), (343, 22), (26, 1001), (2187, 4), (1155, 40),
                                   (4394, 12), (12, 7436), (8190, 3), (6591, 2), (3, 4096)])
@pytest.mark.parametrize("adj", [False, True])
def test_asm_lengths(ny, nx, adj):
    u0 = synth.random_field(ny, nx, 5)
    u = torch.from_numpy(u0).cuda()
    ol().AsmProp(u, ny, nx, P, P, LAM, 0.01, bandlimit=True, adjoint=adj)
    ref = olref.asm_prop(u0.astype(np.complex128), P, P, LAM, 0.01,
                         olref.BANDLIMIT | (olref.ADJOINT if adj else 0))
    assert olref.rel_l2(u.cpu().numpy(), ref) < 1e-6


def test_batch_in_parts():
    """A batch whose padded intermediate passes 2 GiB (13 columns pad to 52 a half)."""
    nb, ny, nx = 6000, 1000, 13
    g = torch.Generator(device="cuda").manual_seed(3)
    u = torch.randn(nb, ny, nx, 2, device="cuda", generator=g)
    u = torch.view_as_complex(u)
    at = [0, 1, 1999, 2500, 2581, 4000, 5162, 5999]
    one = [u[k].clone() for k in at]
    ol().prop_batch(u, P, P, LAM, 0.01)
    for k, f in zip(at, one):
        ol().AsmProp(f, ny, nx, P, P, LAM, 0.01)
        assert torch.equal(u[k], f), k


# every radix; 3146 and 3718 (a radix-2 stage); 4096 (the longest); one to four transforms a work-group
@pytest.mark.parametrize("ny,nx", [(2, 3), (9, 10), (13, 14), (15, 16), (22, 143), (3146, 4), (3, 3718), (4096, 6),
                                   (5, 4056), (1500, 20), (512, 64), (1024, 30)])
def test_c128_lengths(ny, nx):
    """FP64 throughout; phases of up to 1e5 cycles leave 1e-11 of a cycle, hence 1e-9."""
    u0 = synth.random_field(ny, nx, 6, np.complex128)
    u = torch.from_numpy(u0).cuda()
    ol().AsmProp(u, ny, nx, P, P, LAM, 0.01, bandlimit=True)
    assert olref.rel_l2(u.cpu().numpy(), olref.asm_prop(u0, P, P, LAM, 0.01, olref.BANDLIMIT)) < 1e-9
