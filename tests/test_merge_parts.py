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


@pytest.mark.gpu
@pytest.mark.parametrize("parts", [1, 2, 9, 70])
@pytest.mark.parametrize("dv", [64, 255, 320])
@pytest.mark.parametrize("at", [0, 2000, 4250])
@pytest.mark.parametrize("with_sink", [False, True])
def test_join_of_a_nan(parts, dv, at, with_sink):
    """A key that holds a NaN, in one of the first parts, a middle one and (of 70) one behind the 64th, and one whose value does
    and whose weight is 0: the heads that see it are NaN as in one part."""
    torch.manual_seed(parts + dv)
    ctx, bs, n_qh, d = [4300, 1500], 16, 3, 64
    nb = [-(-c // bs) for c in ctx]
    table = torch.arange(2 * max(nb)).view(2, -1).to(torch.int32)
    kc, vc = torch.randn(2 * max(nb) * bs, n_qh * d), torch.randn(2 * max(nb) * bs, n_qh * dv)
    q, pos = torch.randn(2, n_qh * d), torch.tensor([c - 1 for c in ctx])
    kc[at, d] = float("nan")                                # head 1
    vc[at, 2 * dv:], kc[at, 2 * d:] = float("nan"), -1e4 * q[0, 2 * d:]  # head 2
    sink = torch.randn(n_qh) if with_sink else None
    got = mx.row_attention(q.cuda(), kc.cuda(), vc.cuda(), pos.cuda(), None, table.cuda(), bs, n_qh, 1, 1, d, dv, d ** -0.5,
                           parts=parts, out_f32=True, sink=None if sink is None else sink.cuda()).cpu().view(2, n_qh, dv)
    want = mx.row_attention(q, kc, vc, pos, None, table, bs, n_qh, 1, 1, d, dv, d ** -0.5, sink=sink).view(2, n_qh, dv)
    assert bool(got[0, 1:].isnan().all()) and not bool(got[0, 0].isnan().any()) and not bool(got[1].isnan().any())
    for i, h in ((0, 0), (1, 0), (1, 1), (1, 2)):  # (bound of test_join, of 4300 values)
        assert float((got[i, h] - want[i, h]).abs().max()) < 2 ** -18 * max(1.0, float(want[i, h].abs().max())) * 4300 ** 0.5
