"""The packing ops of the LoRA adapters, registered without custom_op's wrapper,
keep what it gave them: schema, fake kernels, the refusal of tensors that are
not on a GPU and of gradients that no formula forms (no GPU needed)."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from metal_liger_amd import _custom_ops as cops

BF = torch.bfloat16


def test_schemas():
    assert str(cops.lora_pack._schema) == (
        "metal_liger_amd::lora_pack(Tensor[] As, Tensor[] Bs, float[] scales, SymInt rank) -> Tensor")
    assert str(cops.lora_unpack._schema) == (
        "metal_liger_amd::lora_unpack(Tensor flat, SymInt[] spec, ScalarType dtype) -> Tensor")


def test_fakes():
    with FakeTensorMode():
        a, b, flat = (torch.empty(s, device="cuda") for s in ((5, 64), (48, 5), (4000,)))
        packed = cops.lora_pack([a, a], [b, b], [2.0, 2.0], 16)
        assert packed.shape == (16 * (2 * 64 + 4 * 48),) and packed.dtype == BF
        out = cops.lora_unpack(flat, [0, 5, 64, 64, 1024, 48, 5, 16], BF)
        assert out.shape == (320 + 256,) and out.dtype == BF


def test_refusals():
    a, b = torch.zeros(8, 16), torch.zeros(32, 8)
    with pytest.raises(ValueError, match="ROCm GPU"):
        cops.lora_pack([a], [b], [1.0], 16)
    with pytest.raises(ValueError, match="ROCm GPU"):
        cops.lora_unpack(a, [0, 1, 1, 1], BF)
    for x, y in ((a.clone().requires_grad_(), b), (a, b.clone().requires_grad_())):
        with pytest.raises(RuntimeError, match="no autograd formula"):
            cops.lora_pack([x], [y], [1.0], 16)
        with torch.no_grad(), pytest.raises(ValueError, match="ROCm GPU"):
            cops.lora_pack([x], [y], [1.0], 16)
