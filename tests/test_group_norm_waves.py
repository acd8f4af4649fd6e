"""Norms of groups and heads by lanes of a wave (gate_group_norm_wave_kernel and head_norm_gate_vec_kernel in
csrc/mixers/recurrent.hip) against float64."""
from __future__ import annotations

import pytest
import torch

from dynamo_exp_amd.ops import recurrent as rc


@pytest.mark.gpu
@pytest.mark.parametrize("n", [8, 504, 512, 520, 1024, 1032, 2048, 2056])
@pytest.mark.parametrize("groups,dtype,shift", [(1, torch.bfloat16, 0), (3, torch.bfloat16, 0), (3, torch.bfloat16, 1),
                                                (5, torch.float32, 0)])
def test_group_norm_waves(n, groups, dtype, shift):
    """Groups around the lengths that a wave holds; weights that are not on 16 bytes."""
    torch.manual_seed(n)
    y, z = torch.randn(7, groups * n) * 3, torch.randn(7, groups * n + 16).to(dtype)
    w = torch.randn(groups * n + 4).cuda()[shift:shift + groups * n]
    got = rc.gate_group_norm(y.cuda(), z.cuda()[:, 16:], w, groups, 1e-5, dtype)
    x = (y.double() * torch.nn.functional.silu(z[:, 16:].double())).view(7, groups, n)
    want = (x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5)).flatten(1) * w.cpu().double()
    # half an ulp of bf16, or fp32 with the gate from the hardware's exp2 and reciprocal
    assert torch.allclose(got.cpu().double(), want, rtol=2.0 ** -8 if dtype == torch.bfloat16 else 1e-5, atol=1e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("gate_act", ["sigmoid", "silu"])
@pytest.mark.parametrize("dv,shift", [(4, 0), (8, 0), (24, 1), (36, 1), (64, 0), (128, 1), (136, 0), (256, 0), (256, 1), (520, 0),
                                      (1024, 0), (2048, 1)])
def test_head_norm_by_runs(dv, shift, gate_act):
    """Heads of whole runs of eight and of four, up to and beyond the width that lanes share; weights not on 16 bytes."""
    torch.manual_seed(dv)
    o, z, w = torch.randn(5, 2 * dv), torch.randn(5, 2 * dv).bfloat16(), torch.randn(2 * dv)
    x = o.double().view(5, 2, dv)
    x = (x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5)).flatten(1) * w.double()
    for gate in (z, None):
        got = rc.head_norm_gate(o.cuda(), 2, torch.cat([w[:shift], w]).cuda()[shift:], gate.cuda() if gate is not None else None, 1e-5, torch.bfloat16, gate_act)
        g = 1.0 if gate is None else torch.sigmoid(z.double()) * (z.double() if gate_act == "silu" else 1.0)
        assert torch.allclose(got.cpu().double(), x * g, rtol=2.0 ** -8, atol=1e-6)
