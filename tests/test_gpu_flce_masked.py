"""The one-pass loss and gradients without the ignored tokens: live rows at the
edges of row tiles and token chunks, against the unmasked form and the fp32
oracle."""

import pytest
import torch

from metal_liger_amd import hip_ops
from oracle import reference_ops as ref
from tests.parity import rel_fro, seeded

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _case(n, n_live, V=1000, H=136, seed=0):
    h = seeded((n, H), seed, BF)
    w = seeded((V, H), seed + 1, BF, scale=0.3)
    g = torch.Generator().manual_seed(seed + 2)
    lab = torch.randint(0, V, (n,), generator=g)
    lab[torch.randperm(n, generator=g)[n_live:]] = -100
    return h, w, lab


@pytest.mark.parametrize("chunk", [None, 256, 512])
@pytest.mark.parametrize("n,n_live", [(1, 1), (1, 0), (700, 0), (700, 1), (700, 255), (700, 256),
                                      (700, 257), (1024, 513), (1030, 1030), (9000, 8191)])
def test_masked_matches_oracle(n, n_live, chunk):
    if n > 8000 and chunk == 256:
        pytest.skip("the same rows in more chunks")
    h, w, lab = _case(n, n_live)
    # what an ignored token holds must not reach any output
    h[lab == -100] = float("nan")
    clean = torch.where(torch.isnan(h), torch.zeros_like(h), h)
    d = [t.cuda() for t in (h, w, lab)]
    for need_w in (True, False):
        loss, lse, nv, dh, dw = hip_ops.flce_fwd_grad(*d, None, -100, True, need_w,
                                                      token_chunk=chunk, masked=True)
        rl, rlse, mask = ref.flce_forward(clean, w, lab, None, -100, 384)
        rdh, rdw = ref.flce_backward(clean, w, lab, rlse, mask, torch.tensor(1.0), None, 384)
        live = lab != -100
        assert nv.item() == n_live
        assert abs(loss.item() - rl.item()) <= 1e-3 * max(abs(rl.item()), 1e-6)
        assert torch.equal(dh.cpu()[~live], torch.zeros_like(h[~live]))
        assert torch.isinf(lse.cpu()[~live]).all()
        if n_live:
            assert rel_fro(lse.cpu()[live], rlse[live]) <= 1e-5
            assert rel_fro(dh, rdh) <= 2e-2
        if need_w:
            assert rel_fro(dw, rdw) <= 2e-2 if n_live else not dw.any()


def test_masked_equals_unmasked_without_ignored_tokens():
    h, w, lab = (t.cuda() for t in _case(1500, 1500, V=2056, H=264, seed=5))
    a = hip_ops.flce_fwd_grad(h, w, lab, None, -100, token_chunk=512)
    b = hip_ops.flce_fwd_grad(h, w, lab, None, -100, token_chunk=512, masked=True)
    for x, y in zip(a, b):
        assert torch.equal(x, y)


def test_repeated_backward_with_ignored_tokens():
    from metal_liger_amd.ops.fused_linear_cross_entropy import _FusedLinearCrossEntropyFunction
    h, w, lab = (t.cuda() for t in _case(300, 170, seed=9))
    h.requires_grad_()
    w.requires_grad_()
    loss = _FusedLinearCrossEntropyFunction.apply(h, w, lab, None, -100, 384)
    first = torch.autograd.grad(loss, [h, w], retain_graph=True)
    again = torch.autograd.grad(loss, [h, w])
    for x, y in zip(first, again):
        # the same sums from bf16 dlogits of 2^-8 rounding
        assert rel_fro(x, y) <= 1e-2


@pytest.mark.parametrize("big", [50.0, 400.0])
def test_masked_recomputes_flagged_rows(big):
    """Rows whose loss leaves the shift window are recomputed among gathered
    rows too."""
    h, w, lab = _case(600, 300, seed=11)
    live = (lab != -100).nonzero().flatten()
    rows = live[[0, 100, 255, 256, 299]]
    h[rows] = h[rows] * big
    loss, lse, nv, dh, dw = hip_ops.flce_fwd_grad(h.cuda(), w.cuda(), lab.cuda(), None, -100,
                                                  masked=True)
    rl, rlse, mask = ref.flce_forward(h, w, lab, None, -100, 8192)
    rdh, rdw = ref.flce_backward(h, w, lab, rlse, mask, torch.tensor(1.0), None, 8192)
    assert abs(loss.item() - rl.item()) <= 1e-3 * abs(rl.item())
    assert rel_fro(dh, rdh) <= 2e-2 and rel_fro(dw, rdw) <= 2e-2


@pytest.mark.parametrize("chunk", [None, 256])
def test_unmasked_reads_strided_rows_in_place(chunk):
    """Without the mask nothing is gathered: rows of a wider tensor, ignored
    tokens among them (their lse is computed, their gradients are zero)."""
    h, w, lab = _case(700, 500, seed=13)
    wide = torch.full((700, 160), float("nan"), dtype=BF)
    wide[:, 8:144] = h
    d = wide.cuda()[:, 8:144]
    assert d.stride(0) == 160
    loss, lse, nv, dh, dw = hip_ops.flce_fwd_grad(d, w.cuda(), lab.cuda(), None, -100,
                                                  token_chunk=chunk)
    rl, rlse, mask = ref.flce_forward(h, w, lab, None, -100, 384)
    rdh, rdw = ref.flce_backward(h, w, lab, rlse, mask, torch.tensor(1.0), None, 384)
    assert nv.item() == 500
    assert abs(loss.item() - rl.item()) <= 1e-3 * abs(rl.item())
    assert rel_fro(lse, rlse) <= 1e-5
    assert rel_fro(dh, rdh) <= 2e-2 and rel_fro(dw, rdw) <= 2e-2
    assert not dh[(lab == -100).cuda()].any()
