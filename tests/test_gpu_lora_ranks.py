"""The adapters' parameters and gradients in one launch each (packing, casting,
rank padding), and the backward passes at every kind of rank and few tokens."""

import pytest
import torch

from metal_liger_amd import hip_ops
from tests.parity import rel_fro, seeded

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("dtype", [torch.float32, BF, torch.float16, torch.float64])
@pytest.mark.parametrize("r,rank", [(16, 16), (5, 16), (17, 32)])
def test_pack_and_unpack(r, rank, dtype):
    ins, outs, scales = (24, 24, 136), (8, 48, 520), (2.0, 1.0, 0.3)
    As = [seeded((r, i), k, dtype).cuda() for k, i in enumerate(ins)]
    # B as a column slice: rows neither dense nor 16-byte aligned
    Bs = [seeded((o, r + 3), 9 + k, dtype).cuda()[:, 1:1 + r] for k, o in enumerate(outs)]
    flat = hip_ops.lora_pack(As, Bs, scales, rank)
    a = [torch.nn.functional.pad(t.to(BF), (0, 0, 0, rank - r)) for t in As]
    b = [torch.nn.functional.pad(t.to(BF), (0, rank - r)) for t in Bs]
    want = torch.cat([t.reshape(-1) for t in (*a, *b, *(t * s for t, s in zip(b, scales)))])
    assert torch.equal(flat, want)
    if dtype == torch.float64:
        return
    src = seeded((3000,), 4).cuda()
    spec = [0, 7, 20, 24, 512, 33, r, rank]
    out = hip_ops.lora_unpack(src, spec, dtype)
    offs, _ = hip_ops.unpack_layout(spec)
    for k, o in enumerate(offs):
        at, rows, cols, ld = spec[4 * k:4 * k + 4]
        assert torch.equal(out[o:o + rows * cols].view(rows, cols),
                           src.as_strided((rows, cols), (ld, 1), at).to(dtype))


@pytest.mark.parametrize("n", [1, 31, 300, 1025])
@pytest.mark.parametrize("rank", [1, 8, 24, 32, 48, 64, 72])
@pytest.mark.parametrize("adapter", [BF, torch.float32])
def test_backward_at_every_rank(n, rank, adapter):
    from metal_liger_amd.ops.fused_lora import _LoRA_QKV, _LoRA_MLP
    H, inter, outs = 264, 520, (272, 136, 136)

    def adapters(dims):
        flat = []
        for k, (o, i) in enumerate(dims):
            flat += [seeded((o, i), 3 * k, BF, scale=i ** -0.5).cuda(),
                     seeded((rank, i), 3 * k + 1, adapter, scale=i ** -0.5).cuda().requires_grad_(),
                     seeded((o, rank), 3 * k + 2, adapter, scale=rank ** -0.5).cuda().requires_grad_(),
                     2.0]
        return flat

    def ref_linear(x, w, a, b, s):
        return x @ w.double().t() + s * ((x @ a.t()) @ b.t())

    x = seeded((n, H), 50, BF).cuda().requires_grad_()
    for fn, dims in ((_LoRA_QKV, [(o, H) for o in outs]), (_LoRA_MLP, [(inter, H), (inter, H), (H, inter)])):
        args = adapters(dims)
        got = fn.apply(x, *args)
        got = list(got) if isinstance(got, tuple) else [got]
        dys = [seeded(tuple(t.shape), 60 + k, BF).cuda() for k, t in enumerate(got)]
        leaves = [x, *(t for t in args if torch.is_tensor(t) and t.requires_grad)]
        grads = torch.autograd.grad(got, leaves, dys)
        # the adapters are cast to the activation dtype before they are used
        l64 = [t.detach().to(BF).double().requires_grad_() for t in leaves]
        it, ps = iter(l64[1:]), []
        for k in range(3):
            ps.append((args[4 * k], next(it), next(it), 2.0))
        if fn is _LoRA_QKV:
            want = [ref_linear(l64[0], *p) for p in ps]
        else:
            h = torch.nn.functional.silu(ref_linear(l64[0], *ps[0])) * ref_linear(l64[0], *ps[1])
            want = [ref_linear(h, *ps[2])]
        wgrads = torch.autograd.grad(want, l64, [d.double() for d in dys])
        for g, w in zip([*got, *grads], [*want, *wgrads]):
            assert g.shape == w.shape
            # bf16 intermediates: up to five roundings (2^-8 at most each), in sums
            # that cancel where one token or one rank leaves a single dot product
            assert rel_fro(g, w) <= 2e-2, (fn.__name__, tuple(g.shape), float(rel_fro(g, w)))
        for g, leaf in zip(grads, leaves):
            assert g.dtype == leaf.dtype and g.is_contiguous()


def test_fake_kernels_match():
    import metal_liger_amd._custom_ops  # noqa: F401
    ops = torch.ops.metal_liger_amd
    check = ("test_schema", "test_faketensor")
    x = seeded((40, 64), 1, BF).cuda()
    Ws = [seeded((o, 64), 2 + o, BF).cuda() for o in (48, 24, 24)]
    As = [seeded((5, 64), 3 + k, torch.float32).cuda() for k in range(3)]
    Bs = [seeded((o, 5), 6 + o, torch.float32).cuda() for o in (48, 24, 24)]
    scales, rank = [2.0, 2.0, 2.0], 16
    torch.library.opcheck(ops.lora_pack.default, (As, Bs, scales, rank), test_utils=check)
    torch.library.opcheck(ops.lora_qkv_fwd.default, (x, Ws, As, Bs, scales, rank), test_utils=check)
    q, k, v, xa, packed = ops.lora_qkv_fwd(x, Ws, As, Bs, scales, rank)
    spec = [0, 5, 64, 64, 3072, 48, 5, 16]
    for sp in (spec, []):
        torch.library.opcheck(ops.lora_qkv_bwd_packed.default,
                              (x, [q, k, v], Ws, packed, scales, xa, rank, sp, torch.float32),
                              test_utils=check)
    torch.library.opcheck(ops.lora_unpack.default, (seeded((4000,), 7).cuda(), spec, BF),
                          test_utils=check)
    kv = [seeded((2, 4, 5, 16), 8 + i, BF).cuda() for i in range(2)]
    torch.library.opcheck(ops.kv_expand.default, (*kv, 2), test_utils=check)
    torch.library.opcheck(ops.kv_reduce.default, (*kv, 2), test_utils=check)
