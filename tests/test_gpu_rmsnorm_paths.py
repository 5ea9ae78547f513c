"""RMSNorm forward / backward at the edges of its launch plans: the widest
row of each path, the one after it, a single row, and row counts that leave
the last batch of rows partly filled; with and without a residual and a saved
rrms. Against the oracle at the bars of tests/parity.py (fp32 1e-5 of the
tensor's scale; 16-bit rtol 2e-2 / atol 1e-2 and 2e-2 in the norm)."""

import pytest
import torch

from oracle import reference_ops as ref
from tests.parity import assert_close, seeded

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32

CASES = [
    # rows, cols, dtype, weight dtype
    (1, 513, BF16, BF16),      # one element per access: first width past a wave
    (1030, 511, F32, F32),     # ... and the last within one
    (259, 1025, F16, F32),
    (1027, 2051, BF16, F32),
    (300, 4097, F32, F32),
    (258, 8191, BF16, BF16),
    (3, 8193, F32, F32),       # past the block path: generic
    (257, 2056, BF16, BF16),   # vectors: first width past the wave backward
    (1281, 4096, BF16, BF16),
    (513, 4104, F16, F16),
    (515, 2052, F32, F32),
    (259, 8192, F32, F32),
    (260, 16384, BF16, F32),   # widest vector row
    (2, 16392, BF16, BF16),    # past it: generic
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{c[1]}-{str(c[2])[6:]}-{str(c[3])[6:]}")
def test_rmsnorm_launch_plans(dev, case):
    from metal_liger_amd import hip_ops
    rows, cols, dtype, wdtype = case
    x, res, dy, ds = (seeded((rows, cols), i, dtype) for i in range(4))
    w = seeded((cols,), 9, wdtype, 0.1, 1.0)
    gx, gr, gdy, gds, gw = (t.to(dev) for t in (x, res, dy, ds, w))

    y, rrms = hip_ops.rms_norm_fwd(gx, gw, 1e-6)
    ry, rr = ref.rms_norm_forward(x, w, 1e-6)
    assert_close(y, ry, "y", dtype)
    assert_close(rrms, rr.squeeze(-1), "rrms", F32)
    rdx, rdw = ref.rms_norm_backward(x, w, rr, dy)
    for r in (rrms, None):
        dx, dw = hip_ops.rms_norm_bwd(gx, gw, gdy, r, 1e-6)
        assert_close(dx, rdx, "dx", dtype)
        assert_close(dw, rdw, "dw", wdtype)

    y, total, rrms = hip_ops.rms_norm_add_fwd(gx, gr, gw, 1e-6)
    ry, rtotal, rr = ref.add_rms_norm_forward(x, res, w, 1e-6)
    assert torch.equal(total.cpu(), rtotal)
    assert_close(y, ry, "add y", dtype)
    rdx, rdw = ref.add_rms_norm_backward(rtotal, w, rr, dy, ds)
    for r in (rrms, None):
        dx, dw = hip_ops.rms_norm_bwd(total, gw, gdy, r, 1e-6, dsum=gds)
        assert_close(dx, rdx, "add dx", dtype)
        assert_close(dw, rdw, "add dw", wdtype)
