"""The join of attention parts (merge_parts_kernel, csrc/mixers/row_attention.hip): batches of eight parts, more parts than
lanes, parts without keys, and value widths on every path of its column loads."""
from __future__ import annotations

import pytest
import torch

from dynamo_exp_amd.ops import mixers as mx


@pytest.mark.gpu
@pytest.mark.parametrize("parts", [2, 8, 9, 17, 70])
@pytest.mark.parametrize("dv", [2, 64, 130, 255, 256, 320])
@pytest.mark.parametrize("weights", ["softmax", "sigmoid"])
def test_join(parts, dv, weights):
    torch.manual_seed(parts + dv)
    ctx, bs, n_qh, d = [1, 20, 333], 16, 3, 64
    nb = [-(-c // bs) for c in ctx]
    table = torch.zeros(len(ctx), max(nb), dtype=torch.int32)
    ids = torch.randperm(sum(nb)).to(torch.int32)
    for i, n in enumerate(nb):
        table[i, :n] = ids[sum(nb[:i]):sum(nb[:i]) + n]
    kc, vc = torch.randn(sum(nb) * bs, n_qh * d), torch.randn(sum(nb) * bs, n_qh * dv)
    q, pos, gate = torch.randn(len(ctx), n_qh * d), torch.tensor([c - 1 for c in ctx]), torch.randn(len(ctx), n_qh)
    args = (table, bs, n_qh, 1, 1, d, dv, d ** -0.5)
    want = mx.row_attention(q, kc, vc, pos, None, *args, weights=weights, head_gate=gate)
    got = mx.row_attention(q.cuda(), kc.cuda(), vc.cuda(), pos.cuda(), None, args[0].cuda(), *args[1:], parts=parts, out_f32=True,
                           weights=weights, head_gate=gate.cuda()).cpu()
    # fp32 sums of at most 333 weighted values on both sides
    assert float((got - want).abs().max()) < 2 ** -18 * max(1.0, float(want.abs().max())) * 333 ** 0.5
