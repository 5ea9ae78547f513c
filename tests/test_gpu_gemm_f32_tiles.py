"""fp32 GEMM at the edges of its tile and split-K choice: one LoRA rank on
either side, odd leading dimensions, remainders of the 64 / 128 tiles and of
the k-tiles, the smallest split, a split over several K segments. Against
float64 at the fp32 bar (1e-5 of the tensor's scale); the split result is
the same from call to call, and without a workspace the call computes the
same product unsplit."""

import pytest
import torch

from tests.parity import assert_close, seeded

pytestmark = pytest.mark.gpu

SHAPES = [(1000, 16, 2048), (16, 2048, 1000), (200, 2048, 2064), (63, 65, 4101), (129, 67, 256),
          (65, 63, 255), (2945, 2943, 37), (1, 1, 5000), (999, 8, 777)]


@pytest.mark.parametrize("a_t,b_t", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_gemm_f32_tiles(dev, a_t, b_t, M, N, K):
    from metal_liger_amd import hip_ops
    a = seeded((K, M) if a_t else (M, K), 1).to(dev)
    b = seeded((N, K) if b_t else (K, N), 2).to(dev)
    out = hip_ops.gemm_f32([a], [b], a_t, b_t, 0.5)
    want = 0.5 * ((a.t() if a_t else a).double() @ (b.t() if b_t else b).double())
    assert_close(out, want.float(), f"{M}x{N}x{K}")
    assert torch.equal(out, hip_ops.gemm_f32([a], [b], a_t, b_t, 0.5))


def test_gemm_f32_split_segments_beta_and_no_workspace(dev):
    from metal_liger_amd import _hip
    M, N, ks = 120, 70, [300, 0, 17, 515]
    As = [seeded((M, k + 3), 3 + i).to(dev)[:, 1:1 + k] for i, k in enumerate(ks)]
    Bs = [seeded((k, N), 13 + i).to(dev) for i, k in enumerate(ks)]
    c0 = seeded((M, N + 5), 23).to(dev)
    want = 2.0 * sum(a.double() @ b.double() for a, b in zip(As, Bs)) - 0.5 * c0[:, :N].double()
    need = _hip.query("ml_gemm_f32_workspace_bytes", M, N, sum(ks))
    assert need >= 2 * M * N * 4
    ws = torch.empty(need // 4, device=dev)
    for w, size in ((ws, need), (ws, need - 1), (None, 0)):
        c = c0.clone()
        _hip.call("ml_gemm_f32_segments_ws", M, N, len(ks), _hip.geom(ks),
                  _hip.ptrs([t.data_ptr() for t in As]), _hip.geom([t.stride(0) for t in As]),
                  _hip.ptrs([t.data_ptr() for t in Bs]), _hip.geom([t.stride(0) for t in Bs]),
                  0, 1, c.data_ptr(), N + 5, 2.0, -0.5, _hip.ptr(w), size, _hip.stream_of(c))
        assert_close(c[:, :N], want.float(), f"workspace {size}")
        assert torch.equal(c[:, N:], c0[:, N:])
