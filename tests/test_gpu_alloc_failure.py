"""GPU checks that a device allocation which fails leaves no error behind: callers then take a form that needs
no workspace, or report the failure themselves, and the next launch check must not report it again."""
import ctypes

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
