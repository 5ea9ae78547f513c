"""Operands that the kernels read as 16-byte vectors are refused on the host when
they are not aligned for it, before anything is launched (no GPU needed: the
pointers are never read)."""

import pytest

from metal_liger_amd import _hip


@pytest.mark.parametrize("fn", ["ml_flce_fwd_grad", "ml_flce_fwd_grad_masked"])
@pytest.mark.parametrize("hidden,ldh,weight,ldw", [(4098, 64, 8192, 64), (4096, 65, 8192, 64),
                                                   (4096, 64, 8194, 64), (4096, 64, 8192, 68)])
def test_one_pass_loss(fn, hidden, ldh, weight, ldw):
    for dh, dw in ((0x8000, 0x9000), (0x8000, None), (None, 0x9000)):
        rc = getattr(_hip.lib(), fn)(hidden, ldh, weight, ldw, None, 0, 0x4000, 8, 64, 64, -100, 8,
                                     0x5000, 0x6000, 0x7000, dh, dw, 0x10000, 1 << 40, None)
        assert rc == 1 and b"row strides in multiples of 8" in _hip.lib().ml_last_error()
