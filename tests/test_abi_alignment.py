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


WS = (0x100000, 1 << 40)


def _refused(fn, args, match):
    rc = getattr(_hip.lib(), fn)(*args)
    assert rc == 1 and match in _hip.lib().ml_last_error(), _hip.lib().ml_last_error()


# (rank 16 reads B and X A^T in single elements: any alignment)
@pytest.mark.parametrize("rank,operands", [(16, "X dY"), (32, "X dY B XA"), (48, "X dY B XA"),
                                           (64, "X dY B XA"), (24, "X dY B XA")])
def test_lora_backwards_of_shared_inputs(rank, operands):
    for at in operands.split():
        p = dict(X=0x1000, dY=0x2000, B=0x3000, XA=0x4000)
        p[at] += 2
        for k in range(3):   # the one adapter whose operand is off; k = 0 too for X, XA
            dy = _hip.ptrs([p["dY"] if i == k else 0x2000 for i in range(3)])
            b = _hip.ptrs([p["B"] if i == k else 0x3000 for i in range(3)])
            w, db = _hip.ptrs([0x5000] * 3), _hip.ptrs([0x6000] * 3)
            _refused("ml_lora_qkv_bwd",
                     (p["X"], 4, 64, dy, _hip.geom([64] * 3), w, 0x7000, b, _hip.floats([1.0] * 3),
                      p["XA"], rank, 0x8000, 0x9000, db, *WS, None), b"must be 16-byte aligned")
        _refused("ml_lora_linear_bwd",
                 (p["X"], 4, 64, p["dY"], 64, 0x5000, 0x7000, p["B"], 1.0, p["XA"], rank, 0x8000,
                  0x9000, 0x6000, *WS, None), b"must be 16-byte aligned")


@pytest.mark.parametrize("rank,operands", [(16, "X dY h"), (32, "X dY h BG BU BD XA hA"),
                                           (64, "X dY h BG BU BD XA hA")])
def test_lora_mlp_backward(rank, operands):
    for at in operands.split():
        p = {n: 0x1000 * (i + 1) for i, n in enumerate("X dY h BG BU BD XA hA".split())}
        p[at] += 2
        _refused("ml_lora_mlp_bwd",
                 (p["X"], 4, 64, 128, 0x10000, 0x11000, p["h"], p["dY"], 0x12000, 0x13000, 0x14000,
                  0x15000, 0x16000, p["BG"], p["BU"], p["BD"], _hip.floats([1.0] * 3), p["XA"],
                  p["hA"], rank, 0x17000, 0x18000, 0x19000, 0x1a000, 0x1b000, 0x1c000, *WS, None),
                 b"must be 16-byte aligned")
