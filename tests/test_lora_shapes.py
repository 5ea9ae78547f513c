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
