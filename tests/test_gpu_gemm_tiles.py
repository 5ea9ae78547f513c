"""The two tiles of the K-major GEMM engine, with and without K split over
workgroups (also through segments), at the edges of tiles and k-tiles."""

import pytest
import torch

from metal_liger_amd import _hip, hip_ops

pytestmark = pytest.mark.gpu


def _check(got, ref64, k):
    # fp32 sums of k products: sqrt(k) roundings of 2^-24 is far below the
    # bound; a bf16 result is rounded once (8 significant bits: 2^-8 at most)
    bound = 2 ** -8 if got.dtype == torch.bfloat16 else 2 ** -22 * max(4, k ** 0.5)
    err = (got.double() - ref64).norm() / ref64.norm()
    assert err <= bound, (float(err), bound)


@pytest.mark.parametrize("tile_cfg", [3, 4])
@pytest.mark.parametrize("ksplit", [1, 3])
@pytest.mark.parametrize("m,n,k", [(1, 8, 8), (127, 136, 72), (129, 128, 264), (257, 264, 1000)])
def test_tiles(m, n, k, ksplit, tile_cfg):
    g = torch.Generator().manual_seed(m + n + k)
    a = torch.randn(m, k, generator=g).bfloat16().cuda()
    for b_t in (True, False):
        b = torch.randn(*((n, k) if b_t else (k, n)), generator=g).bfloat16().cuda()
        ref = a.double() @ (b.double().t() if b_t else b.double())
        for dt in (torch.float32, torch.bfloat16):
            _check(hip_ops.matmul(a, b, b_t=b_t, out_dtype=dt, tile_cfg=tile_cfg, ksplit=ksplit),
                   ref, k)


@pytest.mark.parametrize("tile_cfg", [3, 4])
@pytest.mark.parametrize("ksplit", [1, 3])
@pytest.mark.parametrize("m,n,k", [(127, 136, 200), (257, 264, 1000)])
def test_tiles_add_to_c(m, n, k, ksplit, tile_cfg):
    """alpha A B + beta C, in every store of the tiles and of the split's
    reduction, at an N that no tile divides; columns past N stay."""
    g = torch.Generator().manual_seed(m + k)
    a = torch.randn(m, k, generator=g).bfloat16().cuda()
    b = torch.randn(n, k, generator=g).bfloat16().cuda()
    for dt in (torch.float32, torch.bfloat16):
        wide = torch.randn(m, n + 8, generator=g).to(dt).cuda()
        c = wide[:, :n]
        ref = 0.5 * (a.double() @ b.double().t()) - 1.5 * c.double()
        rest = wide[:, n:].clone()
        hip_ops.matmul(a, b, b_t=True, out=c, alpha=0.5, beta=-1.5, tile_cfg=tile_cfg,
                       ksplit=ksplit)
        # the product's error bound, and C's own share: exact in the products,
        # one more rounding of the sum (fp32) or the same one (bf16)
        _check(c, ref, k)
        assert torch.equal(wide[:, n:], rest)


@pytest.mark.parametrize("b_layout", [0, 1])
@pytest.mark.parametrize("m,n,ks", [(16, 1024, (2048, 8)), (200, 2048, (1000, 72, 3000, 24)),
                                    (513, 136, (72, 4104)), (1, 8, (64, 64))])
def test_segments_split_over_workgroups(m, n, ks, b_layout):
    g = torch.Generator().manual_seed(m + n)
    a = [torch.randn(m, k, generator=g).bfloat16().cuda() for k in ks]
    b = [torch.randn(*((k, n) if b_layout else (n, k)), generator=g).bfloat16().cuda() for k in ks]
    ref = sum(x.double() @ (y.double() if b_layout else y.double().t()) for x, y in zip(a, b))
    lens = _hip.geom(ks)
    wsb = _hip.query("ml_gemm_bf16_segments_workspace_bytes", m, n, len(ks), lens)
    ws = torch.empty(max(wsb, 4), dtype=torch.uint8, device="cuda")
    for size in {0, wsb}:   # no workspace: not split
        out = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
        _hip.call("ml_gemm_bf16_segments_ws", m, n, len(ks), lens,
                  _hip.ptrs([t.data_ptr() for t in a]), _hip.geom([t.stride(0) for t in a]),
                  _hip.ptrs([t.data_ptr() for t in b]), _hip.geom([t.stride(0) for t in b]), 0,
                  b_layout, out.data_ptr(), n, _hip.BF16, 1.0, 0.0,
                  ws.data_ptr() if size else None, size, _hip.stream_of(out))
        _check(out, ref, sum(ks))


def test_split_is_chosen_where_tiles_are_few():
    def splits(m, n, *ks):
        b = _hip.query("ml_gemm_bf16_segments_workspace_bytes", m, n, len(ks), _hip.geom(ks))
        assert b % (m * n * 4) == 0 and b <= 96 << 20
        return b // (m * n * 4)

    assert splits(1777, 2048, 6144, 6144, 64) > 1   # 56 tiles of 256 x 256
    assert splits(8192, 2048, 6144, 6144, 64) == 0  # 256 tiles: one per CU
    assert splits(8192, 6144, 2048, 16) == 0
    assert splits(16, 1024, 64) == 0                # one k-tile cannot be split
