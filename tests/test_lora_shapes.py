"""Adapters whose sizes do not fit their projection are refused before anything
is launched (the packed buffer is read at offsets that follow from the weights'
sizes)."""

import pytest
import torch

from metal_liger_amd import hip_ops
from metal_liger_amd.ops.fused_lora import _LoRA_MLP, _LoRA_QKV, _LoRA_W, _lora_linear

BF = torch.bfloat16


def _projection(i, o, r=8, a=None, b=None):
    """(W, A, B, scale); a / b: sizes of A / B that differ from the right ones."""
    return [torch.zeros(o, i, dtype=BF), torch.zeros(a or (r, i), dtype=BF),
            torch.zeros(b or (o, r), dtype=BF), 2.0]


# what is wrong with the one adapter: A narrower, A wider, B shorter, B longer,
# a B of more or less than A's rank (within the rank that the kernels pad to)
WRONG = [dict(a=(8, 56)), dict(a=(8, 72)), dict(b=(24, 8)), dict(b=(40, 8)), dict(b=(32, 12)),
         dict(b=(32, 4))]


def _args(projections, wrong, at):
    return [v for k, io in enumerate(projections)
            for v in _projection(*io, **(wrong if k == at else {}))]


@pytest.mark.parametrize("wrong", WRONG, ids=str)
@pytest.mark.parametrize("at", [0, 1, 2])
def test_blocks_refuse_adapters_that_do_not_fit(at, wrong):
    x = torch.zeros(4, 64, dtype=BF)
    with pytest.raises(ValueError, match="do not fit 64 input features"):
        _LoRA_QKV.apply(x, *_args([(64, 32)] * 3, wrong, at))
    inter = [(64, 32), (64, 32), (32, 64)]
    if at == 2:   # the down projection's sizes are the other way round
        wrong = {k: (8, v[1] - 32) if k == "a" else (v[0] + 32, v[1]) for k, v in wrong.items()}
    with pytest.raises(ValueError, match="do not fit (64|32) input features"):
        _LoRA_MLP.apply(x, *_args(inter, wrong, at))


@pytest.mark.parametrize("wrong", WRONG, ids=str)
def test_one_projection_refuses_an_adapter_that_does_not_fit(wrong):
    x = torch.zeros(4, 64, dtype=BF)
    args = _projection(64, 32, **wrong)
    with pytest.raises(ValueError, match="do not fit 64 input features"):
        _LoRA_W.apply(x, *args)
    with pytest.raises(ValueError, match="do not fit 64 input features"):
        _lora_linear(x, *args)


def test_weights_that_do_not_fit_the_input_are_refused():
    x = torch.zeros(4, 64, dtype=BF)
    with pytest.raises(ValueError, match="do not fit 64 input features"):
        _LoRA_QKV.apply(x, *_args([(72, 32)] * 3, {}, 0))


@pytest.mark.parametrize("rows", [16, 96, 192, 256])
def test_stacked_adapters_of_another_width_are_refused(rows):
    with pytest.raises(ValueError, match="does not fit 64 input features"):
        hip_ops.lora_xa(torch.zeros(4, 64, dtype=BF), torch.zeros(rows, 72, dtype=BF))


def _seen_by_the_device_check(monkeypatch, fn, *args):
    """The tensors that fn checks for being on one GPU before it launches."""
    class Checked(Exception):
        pass

    def check(*tensors):
        raise Checked(tensors)

    monkeypatch.setattr(hip_ops, "ensure_rocm_device", check)
    with pytest.raises(Checked) as e:
        fn(*args)
    return {id(t) for t in e.value.args[0]}


def test_every_operand_of_the_products_is_checked_for_its_device(monkeypatch):
    """An adapter left on the CPU beside an input on the GPU must not reach a
    kernel as a host pointer."""
    x, w, a, xa, sb = (torch.zeros(s, dtype=BF)
                       for s in ((4, 64), (32, 64), (16, 64), (4, 16), (32, 16)))
    seen = _seen_by_the_device_check(monkeypatch, hip_ops.lora_xa, x, a)
    assert {id(x), id(a)} <= seen
    seen = _seen_by_the_device_check(monkeypatch, hip_ops.lora_linear_out, x, w, xa, sb)
    assert {id(t) for t in (x, w, xa, sb)} <= seen
    seen = _seen_by_the_device_check(monkeypatch, hip_ops.lora_qkv_out, x, [w] * 3, xa, [sb] * 3)
    assert {id(t) for t in (x, w, xa, sb)} <= seen


@pytest.mark.gpu
def test_adapters_on_another_device_are_refused(dev):
    x = torch.zeros(4, 64, dtype=BF, device=dev)
    one = _projection(64, 32)
    for fn in (_LoRA_W.apply, _lora_linear):
        for on_gpu in range(7):   # every subset of the weight, A and B but all of them
            args = [t.to(dev) if on_gpu >> k & 1 else t for k, t in enumerate(one[:3])]
            with pytest.raises((ValueError, RuntimeError), match="ROCm GPU|device"):
                fn(x, *args, 2.0)


def test_plain_projection_does_not_ask_for_adapter_gradients():
    """_lora_linear records nothing for its adapters (the Functions do): its
    result must not require a gradient that cannot be formed."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        x, w, a, b = (torch.empty(s, dtype=BF, device="cuda:0")
                      for s in ((4, 64), (32, 64), (8, 64), (32, 8)))
        out = _lora_linear(x, w, a.requires_grad_(), b.requires_grad_(), 2.0)
    assert out.shape == (4, 32) and not out.requires_grad
