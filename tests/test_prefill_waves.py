"""Prefill attention (csrc/kernels/attn_prefill.hip) with workgroups of four waves (few of them) and of eight: ragged
sequences whose last rows fill a part of a workgroup, one to four heads per key / value head, cached prefixes."""
from __future__ import annotations

import math

import pytest
import torch

from dynamo_exp_amd import ops
from dynamo_exp_amd.ops import reference as ref


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv", [(4, 4), (8, 4), (16, 4)])
@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("bs", [16, 64])
def test_rows(hq, hkv, many, bs):
    torch.manual_seed(hq + many)
    rows, past = [1, 31, 32, 33, 64, 65, 97, 129], [0, 40, 64, 3, 0, 65, 0, 20]
    reps = 16 if many else 1  # 4 x 16 x 8 workgroups and up: eight waves
    rows, past = rows * reps, past * reps
    n = len(rows)
    ctx = [r + p for r, p in zip(rows, past)]
    nb = [-(-c // bs) for c in ctx]
    table = torch.zeros(n, max(nb), dtype=torch.int32)
    ids = torch.randperm(sum(nb)).to(torch.int32)
    for i, k in enumerate(nb):
        table[i, :k] = ids[sum(nb[:i]):sum(nb[:i]) + k]
    kc, vc = (torch.randn(sum(nb), hkv, bs, 128).bfloat16() for _ in range(2))
    q = torch.randn(sum(rows), hq, 128).bfloat16()
    cu = torch.tensor([0] + rows).cumsum(0).to(torch.int32)
    lens, scale = torch.tensor(ctx, dtype=torch.int32), 1 / math.sqrt(128)
    out = torch.full_like(q, float("nan")).cuda()
    ops.prefill_attention(q.cuda(), kc.cuda(), vc.cuda(), table.cuda(), cu.cuda(), lens.cuda(), scale, out)
    want = ref.paged_attention(q, kc, vc, table, cu, lens, scale, bs)
    # bf16 weights (2^-9 each, of values of order one) and one rounding of the result
    err = (out.cpu().float() - want.float()).abs().max()
    assert float(err) < 2 ** -7 * max(1.0, float(want.float().abs().max())), float(err)


@pytest.mark.gpu
@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("bs,ctx", [(16, [1101, 2187, 1030]), (4, [301, 517, 258]), (32, [2600, 2049, 2113]), (64, [4200, 4163, 4500])])
def test_more_pages_than_lanes(bs, ctx, many):
    """The block table is read 64 entries at a time: contexts whose tables are read again in the middle, with tiles of one
    entry and of several, in workgroups of four waves and (many sequences of the same three contexts) of eight."""
    torch.manual_seed(bs + many)
    hq, hkv = (32, 8) if many else (4, 4)
    rows = [(5 + 29 * i) % 71 + 1 for i in range(66)] if many else [70, 33, 129]  # 8 x 66 workgroups and up: eight waves
    nb = [-(-c // bs) for c in ctx]
    table = torch.zeros(len(ctx), max(nb), dtype=torch.int32)
    ids = torch.randperm(sum(nb)).to(torch.int32)
    for i, k in enumerate(nb):
        table[i, :k] = ids[sum(nb[:i]):sum(nb[:i]) + k]
    kc, vc = (torch.randn(sum(nb), hkv, bs, 128).bfloat16() for _ in range(2))
    for i, (c, k) in enumerate(zip(ctx, nb)):  # rows behind the context's end are nobody's
        kc[table[i, k - 1], :, c - (k - 1) * bs:] = vc[table[i, k - 1], :, c - (k - 1) * bs:] = float("nan")
    table, lens = (x.repeat(len(rows) // 3, *[1] * (x.dim() - 1)) for x in (table, torch.tensor(ctx, dtype=torch.int32)))
    q, cu = torch.randn(sum(rows), hq, 128).bfloat16(), torch.tensor([0] + rows).cumsum(0).to(torch.int32)
    out = torch.full_like(q, float("nan")).cuda()
    ops.prefill_attention(q.cuda(), kc.cuda(), vc.cuda(), table.cuda(), cu.cuda(), lens.cuda(), 1 / math.sqrt(128), out)
    want = ref.paged_attention(q, kc, vc, table, cu, lens, 1 / math.sqrt(128), bs)
    err = (out.cpu().float() - want.float()).abs().max()  # (bound of test_rows)
    assert float(err) < 2 ** -7 * max(1.0, float(want.float().abs().max())), float(err)
