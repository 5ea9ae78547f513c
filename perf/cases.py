"""The work whose speed is measured: forward + backward passes through the
fused ops' public entry points, from one small call to a whole LoRA training
step.

The sizes are those of the workloads this repository is built around (a
Qwen3-style text model: hidden 2048, 16 / 8 heads of 128, MLP 6144, vocabulary
151936, rank-16 adapters, 4 x 2048 tokens) and of what users of the same entry
points bring besides: other hidden sizes and LoRA ranks, ragged token counts,
fp32 activations, short sequences.

A case is a dict of plain values. ``kind`` names the entry point:

  norm    MetalLigerRMSNorm, or fused_add_rms_norm with ``residual``
  swiglu  fused_swiglu
  rope    apply_fused_rotary_inline (cos / sin from positions)
  qkv     apply_fused_lora_qkv
  mlp     apply_fused_lora_mlp
  linear  apply_fused_lora_linear (o_proj and other single projections)
  flce    MetalLigerFusedLinearCrossEntropy
  step    decoder layers built from all of these, and the loss: one training
          step of the adapters
"""

import math

import torch
import torch.nn as nn
import torch.nn.functional as F

from metal_liger_amd.ops.fused_add_rms_norm import fused_add_rms_norm
from metal_liger_amd.ops.fused_linear_cross_entropy import MetalLigerFusedLinearCrossEntropy
from metal_liger_amd.ops.fused_lora import (apply_fused_lora_linear, apply_fused_lora_mlp,
                                            apply_fused_lora_qkv)
from metal_liger_amd.ops.fused_qk_norm_rope import apply_fused_qk_norm_rope
from metal_liger_amd.ops.fused_rms_norm import MetalLigerRMSNorm
from metal_liger_amd.ops.fused_rope import apply_fused_rotary_inline
from metal_liger_amd.ops.fused_swiglu import fused_swiglu
from metal_liger_amd.ops.gqa_attention import expanded_kv_attention_forward

DEV = "cuda"
EPS = 1e-6
THETA = 1e6
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # a decoder layer's norm in an fp32 model, 4 x 2048 tokens
        dict(name="norm_fp32", kind="norm", rows=8192, cols=2048, dtype="fp32", residual=False),
        # the residual add and post-attention norm of a wider model, ragged batch
        dict(name="add_norm_bf16_wide", kind="norm", rows=3333, cols=4096, dtype="bf16",
             residual=True),
        # the MLP activation of a model whose projections are not LoRA-patched
        dict(name="swiglu_bf16", kind="swiglu", rows=8192, cols=6144, dtype="bf16"),
        # the rotation of one short sequence: launches and host time count
        dict(name="rope_bf16_short", kind="rope", batch=1, seq=37, heads=16, kv_heads=8, dim=128,
             dtype="bf16"),
        # the q, k, v projections of a short prompt, PEFT's default rank
        dict(name="lora_qkv_r8_short", kind="qkv", tokens=200, hidden=2048, q_out=2048,
             kv_out=1024, rank=8, dtype="bf16", adapter="bf16"),
        # the same block over a full training batch
        dict(name="lora_qkv_r16", kind="qkv", tokens=8192, hidden=2048, q_out=2048, kv_out=1024,
             rank=16, dtype="bf16", adapter="bf16"),
        # the MLP block over a ragged batch, a larger rank, fp32 adapters (as
        # PEFT keeps them unless told otherwise)
        dict(name="lora_mlp_r32_ragged", kind="mlp", tokens=1777, hidden=2048, inter=6144, rank=32,
             dtype="bf16", adapter="fp32"),
        # the MLP block over a full training batch
        dict(name="lora_mlp_r16", kind="mlp", tokens=8192, hidden=2048, inter=6144, rank=16,
             dtype="bf16", adapter="bf16"),
        # an output projection of a model kept in fp32
        dict(name="lora_linear_fp32", kind="linear", tokens=1000, hidden=2048, out=2048, rank=16,
             dtype="fp32", adapter="fp32"),
        # the loss of a LoRA run (frozen head) on one ragged batch with its
        # prompt tokens masked
        dict(name="flce_frozen_ragged", kind="flce", tokens=1000, hidden=2048, vocab=151936,
             train_head=False, ignored=0.3, dtype="bf16"),
        # the loss of a full fine-tuning run, head trained, every token labelled
        dict(name="flce_full", kind="flce", tokens=8192, hidden=2048, vocab=151936,
             train_head=True, ignored=0.0, dtype="bf16"),
        # the whole training step: 4 layers, every projection with an adapter
        dict(name="train_step", kind="step", layers=4, batch=4, seq=2048, hidden=2048, heads=16,
             kv_heads=8, dim=128, inter=6144, vocab=151936, rank=16, dtype="bf16",
             adapter="bf16"),
    ]


def _log_int(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi, step=64):
    """A feature size: a multiple of `step`, spread over the logarithm."""
    return step * _log_int(rng, max(1, lo // step), hi // step)


def draw(rng):
    kind = rng.choice(["norm", "swiglu", "rope", "qkv", "mlp", "linear", "flce", "step"])
    if kind == "norm":
        cols = _width(rng, 64, 5120) if rng.random() < 0.75 else _log_int(rng, 7, 5120)
        return dict(kind=kind, rows=_log_int(rng, 1, 8192), cols=cols,
                    dtype=rng.choice(["fp32", "bf16", "bf16", "fp16"]),
                    residual=rng.random() < 0.5)
    if kind == "swiglu":
        cols = _width(rng, 64, 6144) if rng.random() < 0.75 else _log_int(rng, 37, 6144)
        return dict(kind=kind, rows=_log_int(rng, 1, 8192), cols=cols,
                    dtype=rng.choice(["bf16", "bf16", "fp16"]))
    if kind == "rope":
        kv = rng.choice([1, 2, 4, 8])
        return dict(kind=kind, batch=rng.randint(1, 4), seq=_log_int(rng, 1, 2048),
                    heads=kv * rng.choice([1, 2]), kv_heads=kv, dim=rng.choice([32, 64, 128]),
                    dtype=rng.choice(["bf16", "fp32"]))
    tokens = _log_int(rng, 16, 8192)
    if kind in ("qkv", "mlp"):
        base = dict(kind=kind, tokens=tokens, hidden=_width(rng, 256, 2048),
                    rank=rng.choice([4, 8, 16, 32, 64]), dtype="bf16",
                    adapter=rng.choice(["bf16", "fp32"]))
        if kind == "qkv":
            kv = _width(rng, 128, 1024)
            return dict(base, q_out=kv * rng.choice([1, 2]), kv_out=kv)
        return dict(base, inter=_width(rng, 512, 6144))
    if kind == "linear":
        dtype = rng.choice(["fp32", "bf16"])
        step = 64 if rng.random() < 0.75 else 1
        return dict(kind=kind, tokens=tokens if dtype == "bf16" else min(tokens, 2048),
                    hidden=_width(rng, 72, 2048, step), out=_width(rng, 72, 2048, step),
                    rank=rng.choice([4, 8, 12, 16, 32]), dtype=dtype, adapter=dtype)
    if kind == "flce":
        vocab = _width(rng, 1024, 151936) if rng.random() < 0.5 else _log_int(rng, 1000, 151936)
        return dict(kind=kind, tokens=tokens, hidden=_width(rng, 256, 2048), vocab=vocab,
                    train_head=rng.random() < 0.5, ignored=rng.choice([0.0, 0.3, 0.6]), dtype="bf16")
    return dict(kind=kind, layers=rng.randint(1, 4), batch=rng.randint(1, 4),
                seq=_log_int(rng, 32, 2048), hidden=2048, heads=16, kv_heads=8, dim=128, inter=6144,
                vocab=_log_int(rng, 8192, 151936), rank=rng.choice([8, 16, 32]), dtype="bf16",
                adapter="bf16")


# ------------------------------------------------------------------ the inputs

class _Rng:
    """Tensors drawn on the GPU from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(self, shape, dtype, std=1.0, mean=0.0):
        t = torch.empty(shape, dtype=torch.float32, device=DEV).normal_(mean, std, generator=self.g)
        return t.to(dtype)

    def uniform(self, shape, dtype, bound):
        t = torch.empty(shape, dtype=torch.float32, device=DEV)
        return t.uniform_(-bound, bound, generator=self.g).to(dtype)

    def integers(self, shape, high):
        return torch.randint(0, high, shape, generator=self.g, device=DEV)


class _LoraLinear(nn.Module):
    """A frozen linear layer with one adapter, laid out as PEFT lays it out:
    A uniform as nn.Linear's default, B as after some training, alpha = 2 r."""

    def __init__(self, rng, in_f, out_f, rank, dtype, adapter):
        super().__init__()
        self.base_layer = nn.Module()
        self.base_layer.weight = nn.Parameter(rng.normal((out_f, in_f), dtype, 0.02), False)
        a, b = nn.Module(), nn.Module()
        a.weight = nn.Parameter(rng.uniform((rank, in_f), adapter, in_f ** -0.5))
        b.weight = nn.Parameter(rng.normal((out_f, rank), adapter, 0.02))
        self.lora_A, self.lora_B = nn.ModuleDict({"default": a}), nn.ModuleDict({"default": b})
        self.scaling = {"default": 2.0}

    def adapters(self):
        return [self.lora_A["default"].weight, self.lora_B["default"].weight]


class _Block(nn.Module):
    """Named children, as the attention and MLP modules of a model hold them."""

    def __init__(self, **parts):
        super().__init__()
        for name, part in parts.items():
            setattr(self, name, part)

    def adapters(self):
        return [p for m in self.children() if isinstance(m, _LoraLinear) for p in m.adapters()]


def _lora_types(case):
    return case["rank"], DTYPES[case["dtype"]], DTYPES[case["adapter"]]


def _qkv_block(rng, case, hidden, q_out, kv_out):
    t = _lora_types(case)
    return _Block(q_proj=_LoraLinear(rng, hidden, q_out, *t),
                  k_proj=_LoraLinear(rng, hidden, kv_out, *t),
                  v_proj=_LoraLinear(rng, hidden, kv_out, *t))


def _mlp_block(rng, case, hidden, inter):
    t = _lora_types(case)
    return _Block(gate_proj=_LoraLinear(rng, hidden, inter, *t),
                  up_proj=_LoraLinear(rng, hidden, inter, *t),
                  down_proj=_LoraLinear(rng, inter, hidden, *t))


def _norm(rng, cols, dtype):
    return MetalLigerRMSNorm(cols, EPS, rng.normal((cols,), dtype, 0.1, 1.0))


def _labels(rng, n, vocab, ignored):
    labels = rng.integers((n,), vocab)
    if ignored > 0:
        labels[: int(ignored * n)] = -100  # the prompt's tokens
    return labels


def prepare(case, seed):
    rng, kind = _Rng(seed), case["kind"]
    dtype = DTYPES[case["dtype"]]
    s = dict(case=case)
    if kind == "norm":
        shape = (case["rows"], case["cols"])
        s["x"] = rng.normal(shape, dtype).requires_grad_()
        s["norm"] = _norm(rng, case["cols"], dtype)
        s["dy"] = rng.normal(shape, dtype)
        if case["residual"]:
            s["res"] = rng.normal(shape, dtype).requires_grad_()
            s["dsum"] = rng.normal(shape, dtype)
    elif kind == "swiglu":
        shape = (case["rows"], case["cols"])
        s["gate"] = rng.normal(shape, dtype).requires_grad_()
        s["up"] = rng.normal(shape, dtype).requires_grad_()
        s["dy"] = rng.normal(shape, dtype)
    elif kind == "rope":
        b, n, d = case["batch"], case["seq"], case["dim"]
        hq, hk = case["heads"], case["kv_heads"]
        # [B, H, S, D] views of [B, S, H, D] projections, as attention has them
        s["q"] = rng.normal((b, n, hq, d), dtype).transpose(1, 2).requires_grad_()
        s["k"] = rng.normal((b, n, hk, d), dtype).transpose(1, 2).requires_grad_()
        s["dq"] = rng.normal((b, hq, n, d), dtype)
        s["dk"] = rng.normal((b, hk, n, d), dtype)
        s["pos"] = torch.arange(n, device=DEV).unsqueeze(0).expand(b, n)
    elif kind == "qkv":
        s["x"] = rng.normal((case["tokens"], case["hidden"]), dtype).requires_grad_()
        s["block"] = _qkv_block(rng, case, case["hidden"], case["q_out"], case["kv_out"])
        s["dy"] = [rng.normal((case["tokens"], o), dtype)
                   for o in (case["q_out"], case["kv_out"], case["kv_out"])]
    elif kind == "mlp":
        shape = (case["tokens"], case["hidden"])
        s["x"] = rng.normal(shape, dtype).requires_grad_()
        s["block"] = _mlp_block(rng, case, case["hidden"], case["inter"])
        s["dy"] = rng.normal(shape, dtype)
    elif kind == "linear":
        s["x"] = rng.normal((case["tokens"], case["hidden"]), dtype).requires_grad_()
        s["linear"] = _LoraLinear(rng, case["hidden"], case["out"], *_lora_types(case))
        s["dy"] = rng.normal((case["tokens"], case["out"]), dtype)
    elif kind == "flce":
        s["x"] = rng.normal((case["tokens"], case["hidden"]), dtype).requires_grad_()
        head = nn.Module()
        head.weight = nn.Parameter(rng.normal((case["vocab"], case["hidden"]), dtype, 0.02),
                                   case["train_head"])
        head.bias = None
        s["loss"] = MetalLigerFusedLinearCrossEntropy(head)
        s["labels"] = _labels(rng, case["tokens"], case["vocab"], case["ignored"])
    else:
        s.update(_prepare_step(case, rng, dtype))
    return s


def _rope_tables(batch, seq, dim, dtype):
    inv = 1.0 / (THETA ** (torch.arange(0, dim, 2, device=DEV).float() / dim))
    ang = torch.arange(seq, device=DEV).float()[:, None] * inv
    ang = torch.cat((ang, ang), -1).expand(batch, seq, dim)
    return ang.cos().to(dtype), ang.sin().to(dtype)


def _prepare_step(case, rng, dtype):
    h, d = case["hidden"], case["dim"]
    q_out, kv_out = case["heads"] * d, case["kv_heads"] * d
    layers = []
    for _ in range(case["layers"]):
        attn = _qkv_block(rng, case, h, q_out, kv_out)
        attn.o_proj = _LoraLinear(rng, q_out, h, *_lora_types(case))
        attn.q_norm, attn.k_norm = _norm(rng, d, dtype), _norm(rng, d, dtype)
        attn.num_key_value_groups, attn.is_causal = case["heads"] // case["kv_heads"], True
        layers.append(_Block(input_layernorm=_norm(rng, h, dtype), self_attn=attn,
                             post_attention_layernorm=_norm(rng, h, dtype),
                             mlp=_mlp_block(rng, case, h, case["inter"])))
    norm = _norm(rng, h, dtype)
    for m in [norm, *(m for layer in layers for m in layer.modules())]:
        if isinstance(m, MetalLigerRMSNorm):
            m.requires_grad_(False)  # only the adapters train
    head = nn.Module()
    head.weight = nn.Parameter(rng.normal((case["vocab"], h), dtype, 0.02), False)
    head.bias = None
    ids = rng.integers((case["batch"], case["seq"]), case["vocab"])
    labels = F.pad(ids, (0, 1), value=-100)[:, 1:].reshape(-1)
    cos, sin = _rope_tables(case["batch"], case["seq"], d, dtype)
    params = [p for la in layers for b in (la.self_attn, la.mlp) for p in b.adapters()]
    return dict(layers=layers, norm=norm, head=head,
                loss=MetalLigerFusedLinearCrossEntropy(head), ids=ids, labels=labels, cos=cos,
                sin=sin, params=params)


# ------------------------------------------------------------------- one pass

def run(s):
    kind = s["case"]["kind"]
    grad = torch.autograd.grad
    if kind == "norm":
        if s["case"]["residual"]:
            y, total = fused_add_rms_norm(s["x"], s["res"], s["norm"])
            return [y, total, *grad([y, total], [s["x"], s["res"], s["norm"].weight],
                                    [s["dy"], s["dsum"]])]
        y = s["norm"](s["x"])
        return [y, *grad(y, [s["x"], s["norm"].weight], s["dy"])]
    if kind == "swiglu":
        y = fused_swiglu(s["gate"], s["up"])
        return [y, *grad(y, [s["gate"], s["up"]], s["dy"])]
    if kind == "rope":
        q, k = apply_fused_rotary_inline(s["q"], s["k"], s["pos"], THETA)
        return [q, k, *grad([q, k], [s["q"], s["k"]], [s["dq"], s["dk"]])]
    if kind == "qkv":
        out = apply_fused_lora_qkv(s["block"], s["x"])
        return [*out, *grad(list(out), [s["x"], *s["block"].adapters()], s["dy"])]
    if kind == "mlp":
        y = apply_fused_lora_mlp(s["block"], s["x"])
        return [y, *grad(y, [s["x"], *s["block"].adapters()], s["dy"])]
    if kind == "linear":
        y = apply_fused_lora_linear(s["linear"], s["x"])
        return [y, *grad(y, [s["x"], *s["linear"].adapters()], s["dy"])]
    if kind == "flce":
        loss = s["loss"](s["x"], s["labels"])
        wrt = [s["x"], s["loss"].weight] if s["case"]["train_head"] else [s["x"]]
        return [loss, *grad(loss, wrt)]
    return _run_step(s)


def _run_step(s):
    c = s["case"]
    b, n, d = c["batch"], c["seq"], c["dim"]
    x = F.embedding(s["ids"], s["head"].weight)
    for layer in s["layers"]:
        attn = layer.self_attn
        q, k, v = apply_fused_lora_qkv(attn, layer.input_layernorm(x))
        q, k, v = (t.view(b, n, -1, d).transpose(1, 2) for t in (q, k, v))
        q, k = apply_fused_qk_norm_rope(q, k, attn.q_norm, attn.k_norm, s["cos"], s["sin"])
        o, _ = expanded_kv_attention_forward(attn, q, k, v, None, scaling=d ** -0.5)
        o = apply_fused_lora_linear(attn.o_proj, o.reshape(b, n, -1))
        y, x = fused_add_rms_norm(o, x, layer.post_attention_layernorm)
        x = x + apply_fused_lora_mlp(layer.mlp, y)
    x = s["norm"](x)
    loss = s["loss"](x, s["labels"])
    return [loss, x, *torch.autograd.grad(loss, s["params"])]


# ------------------------------------------------- what a pass cannot do without

def _lora_flops(n, i, o, r):
    """One projection: x W^T and dy W, and the adapter's six rank-r products."""
    return 2 * n * (2 * i * o + 3 * r * (i + o))


def work(case):
    kind, es = case["kind"], DTYPES[case["dtype"]].itemsize
    if kind == "norm":
        n, c = case["rows"], case["cols"]
        # x (and the residual) read, y (and the sum) written; then x or the
        # sum, dy (and the sum's gradient) read and dx written
        return {"bytes": (8 if case["residual"] else 5) * n * c * es + 2 * c * es,
                "flops": 12 * n * c}
    if kind == "swiglu":
        n = case["rows"] * case["cols"]
        return {"bytes": 8 * n * es, "flops": 20 * n}
    if kind == "rope":
        n = case["batch"] * case["seq"] * (case["heads"] + case["kv_heads"]) * case["dim"]
        return {"bytes": 4 * n * es, "flops": 6 * n}
    if kind in ("qkv", "mlp", "linear"):
        n, h, r, ae = case["tokens"], case["hidden"], case["rank"], DTYPES[case["adapter"]].itemsize
        if kind == "qkv":
            pairs = [(h, case["q_out"]), (h, case["kv_out"]), (h, case["kv_out"])]
            acts = 2 * n * h + 2 * n * sum(o for _, o in pairs)
        elif kind == "mlp":
            pairs = [(h, case["inter"]), (h, case["inter"]), (case["inter"], h)]
            acts = 4 * n * h + 4 * n * case["inter"]   # gate and up are kept for the backward
        else:
            pairs = [(h, case["out"])]
            acts = 2 * n * h + 2 * n * case["out"]
        return {"bytes": es * (acts + sum(i * o for i, o in pairs)) +
                2 * ae * sum(r * (i + o) for i, o in pairs),
                "flops": sum(_lora_flops(n, i, o, r) for i, o in pairs)}
    if kind == "flce":
        n, h, v = case["tokens"], case["hidden"], case["vocab"]
        # logits and dH, and dW when the head trains (the weight read, dW written)
        products = 3 if case["train_head"] else 2
        return {"bytes": es * (2 * n * h + (products - 1) * v * h) + 8 * n,
                "flops": products * 2 * n * v * h}
    n, h, r, i = case["batch"] * case["seq"], case["hidden"], case["rank"], case["inter"]
    qo, kv = case["heads"] * case["dim"], case["kv_heads"] * case["dim"]
    pairs = [(h, qo), (h, kv), (h, kv), (qo, h), (h, i), (h, i), (i, h)]
    # causal attention: two products over half the square forward, five backward
    attn = 7 * case["batch"] * case["seq"] ** 2 * qo
    layer = sum(_lora_flops(n, a, o, r) for a, o in pairs) + attn
    per_layer = sum(a * o + 2 * r * (a + o) for a, o in pairs) + n * (4 * h + 4 * qo + 4 * kv + 4 * i)
    return {"bytes": es * (case["layers"] * per_layer + case["vocab"] * h + 4 * n * h),
            "flops": case["layers"] * layer + 4 * n * h * case["vocab"]}


# ------------------------------------------------------------------- tolerances

def tolerance(case):
    """About four times the distance from the 64-bit result that is seen."""
    kind = case["kind"]
    low = case["dtype"] != "fp32"
    if kind in ("norm", "swiglu", "rope"):
        # one rounding of each result (bf16: 1.7e-3); fp32: a sum over a row
        # or over all rows
        return {"rel": 7e-3, "max": 1.6e-2} if low else {"rel": 2e-6, "max": 2e-5}
    if kind == "linear" and not low:
        return {"rel": 5e-6, "max": 5e-5}   # 9.9e-7: fp32 products over 2048 terms
    if kind == "step":
        # 2.6e-2: every layer's bf16 roundings travel through those behind it
        return {"rel": 8e-2}
    if kind == "mlp":
        return {"rel": 1.6e-2}   # 3.9e-3: gate, up, h and their gradients in bf16
    return {"rel": 1.2e-2}       # 2.4e-3 to 2.9e-3: products of bf16 operands


# ----------------------------------------------------------------- in 64 bits

def _lora64(m, x):
    w, (a, b) = m.base_layer.weight.double(), m.p64
    return x @ w.t() + m.scaling["default"] * ((x @ a.t()) @ b.t())


def _to64(module):
    """Every projection's adapters as 64-bit leaves, in adapters() order."""
    leaves = []
    for m in module.modules():
        if isinstance(m, _LoraLinear):
            m.p64 = [p.detach().double().requires_grad_() for p in m.adapters()]
            leaves += m.p64
    return leaves


def _norm64(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w


def _rotate64(x, cos, sin):
    a, b = x.chunk(2, -1)
    return x * cos + torch.cat((-b, a), -1) * sin


def _mlp64(block, x):
    return _lora64(block.down_proj, F.silu(_lora64(block.gate_proj, x)) * _lora64(block.up_proj, x))


def _loss64(h, weight, labels, need_dw):
    """(loss, d loss / d h, d loss / d weight) over slices of the tokens."""
    w = weight.double()
    keep = labels != -100
    scale = 1.0 / max(1, int(keep.sum()))
    loss, dh = h.new_zeros(()), torch.empty_like(h)
    dw = torch.zeros_like(w) if need_dw else None
    for i in range(0, h.shape[0], 1024):
        hc, yc, kc = h[i:i + 1024], labels[i:i + 1024].clamp(min=0), keep[i:i + 1024, None]
        z = hc @ w.t()
        lse = z.logsumexp(-1, keepdim=True)
        loss = loss + ((lse - z.gather(1, yc[:, None])) * kc).sum() * scale
        z = (z - lse).exp_()
        z.scatter_add_(1, yc[:, None], -torch.ones_like(lse))
        z.mul_(kc * scale)
        dh[i:i + 1024] = z @ w
        if need_dw:
            dw += z.t() @ hc
    return loss, dh, dw


def exact(case, seed):
    s, kind = prepare(case, seed), case["kind"]
    grad = torch.autograd.grad

    def leaf(name):
        return s[name].detach().double().requires_grad_()

    if kind == "norm":
        x, w = leaf("x"), s["norm"].weight.detach().double().requires_grad_()
        if case["residual"]:
            res = leaf("res")
            # the sum is a result of its own and is normalised as it is kept
            total = (s["x"] + s["res"]).detach().double().requires_grad_()
            y = _norm64(total, w)
            dt, dw = grad(y, [total, w], s["dy"].double())
            dt = dt + s["dsum"].double()
            return [y.detach(), (x + res).detach(), dt, dt, dw]
        y = _norm64(x, w)
        return [y.detach(), *grad(y, [x, w], s["dy"].double())]
    if kind == "swiglu":
        g, u = leaf("gate"), leaf("up")
        y = F.silu(g) * u
        return [y.detach(), *grad(y, [g, u], s["dy"].double())]
    if kind == "rope":
        q, k = leaf("q"), leaf("k")
        d = case["dim"]
        # the angles are fp32 values: frequencies and products rounded as given
        inv = 1.0 / (THETA ** (torch.arange(0, d, 2, dtype=torch.int64).float() / d))
        ang = s["pos"].float()[..., None] * inv.to(DEV)
        ang = torch.cat((ang, ang), -1).double()[:, None]
        oq, ok = (_rotate64(t, ang.cos(), ang.sin()) for t in (q, k))
        return [oq.detach(), ok.detach(),
                *grad([oq, ok], [q, k], [s["dq"].double(), s["dk"].double()])]
    if kind == "qkv":
        x, p = leaf("x"), _to64(s["block"])
        out = [_lora64(m, x) for m in s["block"].children()]
        return [*(o.detach() for o in out), *grad(out, [x, *p], [t.double() for t in s["dy"]])]
    if kind == "mlp":
        x, p = leaf("x"), _to64(s["block"])
        y = _mlp64(s["block"], x)
        return [y.detach(), *grad(y, [x, *p], s["dy"].double())]
    if kind == "linear":
        x, p = leaf("x"), _to64(s["linear"])
        y = _lora64(s["linear"], x)
        return [y.detach(), *grad(y, [x, *p], s["dy"].double())]
    if kind == "flce":
        loss, dh, dw = _loss64(s["x"].detach().double(), s["loss"].weight.detach(), s["labels"],
                               case["train_head"])
        return [loss, dh, dw] if case["train_head"] else [loss, dh]
    return _exact_step(s)


def _exact_step(s):
    c = s["case"]
    b, n, d = c["batch"], c["seq"], c["dim"]
    leaves = [p for la in s["layers"] for blk in (la.self_attn, la.mlp) for p in _to64(blk)]
    cos, sin = s["cos"].double()[:, None], s["sin"].double()[:, None]
    mask = torch.full((n, n), float("-inf"), dtype=torch.float64, device=DEV).triu(1)
    x = F.embedding(s["ids"], s["head"].weight.detach()).double()
    for layer in s["layers"]:
        attn = layer.self_attn
        y = _norm64(x, layer.input_layernorm.weight.double())
        q, k, v = (_lora64(m, y).view(b, n, -1, d).transpose(1, 2)
                   for m in (attn.q_proj, attn.k_proj, attn.v_proj))
        q = _rotate64(_norm64(q, attn.q_norm.weight.double()), cos, sin)
        k = _rotate64(_norm64(k, attn.k_norm.weight.double()), cos, sin)
        k, v = (t.repeat_interleave(attn.num_key_value_groups, 1) for t in (k, v))
        p = ((q @ k.transpose(2, 3).contiguous()) * d ** -0.5 + mask).softmax(-1)
        o = (p @ v).transpose(1, 2).reshape(b, n, -1)
        x = x + _lora64(attn.o_proj, o)
        x = x + _mlp64(layer.mlp, _norm64(x, layer.post_attention_layernorm.weight.double()))
    x = _norm64(x, s["norm"].weight.double())
    loss, dh, _ = _loss64(x.detach().reshape(b * n, -1), s["head"].weight.detach(), s["labels"],
                          False)
    return [loss, x.detach(), *torch.autograd.grad(x, leaves, dh.view_as(x))]
