"""GPU checks of the power-of-two passes with a side below 1024, whose work-groups are sized by the
number of columns: every count of columns a work-group from 16 down to 4, one row to eight a row pass's
wave, and stacks, which count all fields' columns, bit for bit as single fields.  Against the FP64 oracle
to 1e-6: FP32 transforms of up to 16384 points are about 3e-7 off."""
import numpy as np
import pytest
import torch

import olref
from openol_amd import synth

pytestmark = pytest.mark.gpu
LAM, P = 532e-9, 8e-6


@pytest.mark.parametrize("ny,nx", [(4, 4), (8, 512), (64, 1024), (256, 256), (512, 64), (512, 2048), (2048, 128),
                                   (8192, 16)])
def test_small_fields(ny, nx):
    import openol_amd as ol
    from openol_amd import ops
    u = np.stack([synth.random_field(ny, nx, seed=ny + nx + k) for k in range(3)]).astype(np.complex64)
    d = torch.from_numpy(u).cuda()
    out = torch.empty_like(d)
    ops.asm_batch(d, out, P, P, LAM, 0.02, True)
    for k in range(3):
        one = d[k].clone()
        ol.AsmProp(one, ny, nx, P, P, LAM, 0.02, bandlimit=True)
        assert torch.equal(torch.view_as_real(one), torch.view_as_real(out[k]))
    ref = olref.asm_prop(u[0].astype(np.complex128), P, P, LAM, 0.02, olref.BANDLIMIT)
    got = out[0].cpu().numpy()
    assert np.linalg.norm(got - ref) < 1e-6 * np.linalg.norm(ref)
