"""The mixed-radix propagation's launch shapes, in rows and in columns: two work-groups a CU with twice the
butterflies a thread (3380, 3920, 4000, 4160), one alone with all its threads (4732, 5292, 6000, 8100), waves
rounded up to whole rounds of the SIMDs (2420, 3528), three to six butterflies of radix 2, 3, 4 and 5 a thread
(3388, 3564, 3718, 3861, 3900, 4004), and row passes whose halves take another shape than their pairs.

Bar: as the other complex64 lengths, 1e-6 (4e-7 measured against FP64 on every path)."""
import numpy as np
import pytest
import torch

import olref
from openol_amd import synth

pytestmark = pytest.mark.gpu
LAM, P = 532e-9, 8e-6


@pytest.mark.parametrize("n", [2420, 3380, 3388, 3528, 3564, 3718, 3861, 3900, 3920, 4000, 4004, 4160, 4732, 5000, 5292,
                               6000, 7260, 8100])
@pytest.mark.parametrize("col", [False, True])
def test_shapes(n, col):
    import openol_amd as ol
    ny, nx = (n, 12) if col else (9, n)
    u0 = synth.random_field(ny, nx, n)
    u = torch.from_numpy(u0).cuda()
    ol.AsmProp(u, ny, nx, P, P, LAM, 0.01, bandlimit=True)
    ref = olref.asm_prop(u0.astype(np.complex128), P, P, LAM, 0.01, olref.BANDLIMIT)
    assert olref.rel_l2(u.cpu().numpy(), ref) < 1e-6
