"""The private torch names that save host time have public ways round them (no
GPU needed)."""

import types

import torch
from torch.autograd import forward_ad

from metal_liger_amd import _hip
from metal_liger_amd.ops import gqa_attention as ga


def test_stream_without_the_raw_handle(monkeypatch):
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    monkeypatch.setattr(torch.cuda, "current_stream",
                        lambda device: types.SimpleNamespace(cuda_stream=(7, device)))
    t = types.SimpleNamespace(is_cuda=True, device="cuda:1", get_device=lambda: 1)
    assert _hip.stream_of(t) == (7, "cuda:1")


def test_repeated_heads_without_the_transform_queries(monkeypatch):
    assert ga._plain_eager()
    with forward_ad.dual_level():
        assert not ga._plain_eager()
    for owner, name in ((torch._C, "_are_functorch_transforms_active"),
                        (forward_ad, "_current_level")):
        with monkeypatch.context() as m:
            m.delattr(owner, name)
            assert not ga._plain_eager()
