"""The two-map combine (csrc/mixers/stream_ops.hip), which takes four vectors at a time from some number on: on both sides
of that number and with a last group that is not full."""
from __future__ import annotations

import pytest
import torch

from dynamo_exp_amd.ops import mixers as mx


@pytest.mark.gpu
@pytest.mark.parametrize("T,H", [(5, 3), (2731, 3), (4099, 2)])
@pytest.mark.parametrize("dv", [2, 64, 252, 256, 260])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_diff_combine(T, H, dv, dtype):
    torch.manual_seed(dv)
    for gate in (None, torch.randn(T, H + 2).to(dtype)[:, :H]):
        for skew in (0, 1):  # (a start that is not 16-byte aligned: the general form)
            a = torch.randn(T * H * 2 * dv + skew)[skew:].view(T, H, 2, dv)
            o = a[:, :, 0].double() - 0.6 * a[:, :, 1].double()
            inv = torch.rsqrt((o * o).mean(-1, keepdim=True) + 1e-5) * 0.8
            want = o * inv
            if gate is not None:
                want = want * torch.sigmoid(gate.double())[:, :, None]
            dev = torch.empty(a.numel() + skew, device="cuda")[skew:].view(a.shape).copy_(a)
            got = mx.diff_combine(dev, 0.6, 0.8, 1e-5, dtype, None if gate is None else gate.cuda()).cpu().double()
            # one rounding to the result's type; the difference of two values below 6 is rounded at their size (2^-21)
            tol = 2 ** -8 if dtype == torch.bfloat16 else 2 ** -20
            assert ((got.view(want.shape) - want).abs() <= tol * want.abs() + 2 ** -20 * inv).all()
