"""Repeated key / value heads and their gradients against torch's expand."""

import pytest
import torch

from metal_liger_amd.ops import gqa_attention as ga
from tests.parity import seeded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("b,h,s,d,groups", [(1, 1, 1, 8, 2), (2, 3, 37, 64, 4), (1, 2, 5, 24, 3),
                                            (2, 8, 300, 128, 2), (1, 2, 9, 12, 2)])
@pytest.mark.parametrize("layout", ["bshd", "bhsd", "slice"])
def test_repeat_kv(b, h, s, d, groups, dtype, layout):
    def make(seed, width=d):
        if layout == "bshd":     # the projections' layout
            return seeded((b, s, h, width), seed, dtype).cuda().transpose(1, 2)
        if layout == "bhsd":
            return seeded((b, h, s, width), seed, dtype).cuda()
        return seeded((b, h, s + 3, width + 3), seed, dtype).cuda()[:, :, 1:s + 1, 1:width + 1]

    k, v = make(1).requires_grad_(), make(2, 2 * d).requires_grad_()
    ko, vo = ga._repeat_kv(k, v, groups)
    kr, vr = ga._repeat_heads(k, groups), ga._repeat_heads(v, groups)
    assert torch.equal(ko, kr) and torch.equal(vo, vr) and ko.is_contiguous()
    dk = seeded((b, s, h * groups, d), 3, dtype).cuda().transpose(1, 2)
    dv = seeded((b, h * groups, s, 2 * d), 4, dtype).cuda()
    got = torch.autograd.grad([ko, vo], [k, v], [dk, dv])
    want = torch.autograd.grad([kr, vr], [k, v], [dk, dv])
    for g, w in zip(got, want):
        # fp32 sums of up to 4 values in another order, then one rounding
        tol = {torch.bfloat16: 2 ** -8, torch.float16: 2 ** -10, torch.float32: 2 ** -21}[dtype]
        assert torch.allclose(g.float(), w.float(), rtol=tol, atol=4 * tol)


def test_transforms_take_the_torch_path():
    k = seeded((2, 1, 2, 5, 16), 1).cuda()
    out = torch.vmap(lambda t: ga._repeat_kv(t, t, 2)[0])(k)
    assert torch.equal(out, k.repeat_interleave(2, 2))
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(k[0], k[1])
        out = ga._repeat_kv(dual, dual, 2)[1]
        assert torch.equal(torch.autograd.forward_ad.unpack_dual(out).tangent,
                           k[1].repeat_interleave(2, 1))
    g = torch.compile(lambda t: ga._repeat_kv(t, t, 2)[0], fullgraph=True, backend="aot_eager")(k[0])
    assert torch.equal(g, k[0].repeat_interleave(2, 1))
