"""Entry points that take device tensors as they come refuse host tensors
before anything is launched (runs without a GPU)."""

from __future__ import annotations

import pytest
import torch

from ccut import _dev


@pytest.mark.parametrize("device", ["cpu", "meta"])
def test_stream_of_a_host_device(device):
    with pytest.raises(ValueError):
        _dev.stream_ptr(torch.device(device))


@pytest.mark.parametrize("shape", [(1, 128), (4, 128), (2, 3, 128), (40, 128)])
def test_awq_gemm_refuses_host_activations(shape):
    from ccut.quant import awq

    w = awq.AwqWeights(torch.zeros(128 * 16 // 8, dtype=torch.int32), torch.zeros((16, 4), dtype=torch.int32),
                       torch.float16, 128, 16, 128)
    with pytest.raises(ValueError, match="cpu"):
        awq.gemm(torch.zeros(shape, dtype=torch.float16), w)


def test_moe_ffn_fp8_refuses_host_activations():
    from ccut.blocks import moe

    u8, f32 = lambda *s: torch.zeros(s, dtype=torch.uint8), lambda *s: torch.zeros(s)  # noqa: E731
    ex = moe.Fp8Experts(u8(2, 128, 128), f32(2, 1, 1), u8(2, 128, 128), f32(2, 1, 1), u8(2, 128, 128), f32(2, 1, 1),
                        num_experts=2, hidden=128, inter=128)
    with pytest.raises(ValueError, match="cpu"):
        moe.moe_ffn_fp8(torch.zeros((3, 128)), torch.zeros((3, 1), dtype=torch.int64), torch.ones((3, 1)), ex)


@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("forward", [False, True])
def test_moe_w4_refuses_host_activations(monkeypatch, forward, shared):
    """(Only x is on the host here; to_device stands in for the GPU's copies of
    the other operands.)"""
    from ccut.blocks import moe

    monkeypatch.setattr(_dev, "to_device", lambda a, dtype=None: a if dtype is None else a.to(dtype))
    i32 = lambda *s: torch.zeros(s, dtype=torch.int32)  # noqa: E731
    w, sz = i32(2 + shared, 128 * 128 // 8), i32(2 + shared, 128, 4)
    ex = moe.W4Experts(w, sz, w, sz, w, sz, torch.float16, num_experts=2 + shared, hidden=128, inter=128,
                       group_size=128, shared_expert=shared)
    x = torch.zeros((3, 128), dtype=torch.float16)
    with pytest.raises(ValueError, match="cpu"):
        if forward:
            moe.moe_forward_w4(x, torch.zeros((3, 2)), ex, 1)
        else:
            moe.moe_ffn_w4(x, torch.zeros((3, 1), dtype=torch.int64), torch.ones((3, 1)), ex)
