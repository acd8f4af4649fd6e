"""Decode attention's join of partitions and its block-table prefetch (csrc/kernels/attn_decode.hip): numbers of parts
around the 16 rows and the 64 lanes that the join asks for at once, workspaces full of NaN, rows and workspaces with
their elements' alignment only, and tables of fewer and of more than the 64 columns that are asked for early."""
from __future__ import annotations

import math

import pytest
import torch

from dynamo_exp_amd import ops
from dynamo_exp_amd.ops import reference as ref


@pytest.mark.gpu
@pytest.mark.parametrize("ctx", [[1, 17, 130], [2100, 3, 0, 1024], [20000, 129]])
@pytest.mark.parametrize("n_parts", [2, 15, 16, 17, 64, 65, 150])
def test_parts(ctx, n_parts):
    torch.manual_seed(n_parts)
    B, hq, hkv, bs = len(ctx), 8, 2, 16
    need = [-(-c // bs) for c in ctx]
    wide = max(need) + 5
    table = torch.zeros(B, wide, dtype=torch.int32)
    ids = torch.randperm(sum(need)).to(torch.int32)
    for b, n in enumerate(need):
        table[b, :n] = ids[sum(need[:b]):sum(need[:b]) + n]
    kc, vc = (torch.randn(sum(need), hkv, bs, 128).bfloat16() for _ in range(2))
    q, lens, scale = torch.randn(B, hq, 128).bfloat16(), torch.tensor(ctx, dtype=torch.int32), 1 / math.sqrt(128)
    live = [b for b in range(B) if ctx[b]]
    want = ref.paged_attention(q[live], kc, vc, table[live], torch.arange(len(live) + 1, dtype=torch.int32), lens[live], scale, bs)
    bt = table.cuda()[:, :max(need)]  # rows farther apart than the columns that may be read
    nan = float("nan")
    out = torch.full((B * hq * 128 + 1,), nan, dtype=torch.bfloat16, device="cuda")[1:].view(B, hq, 128)
    ws = (torch.full((B * hq * n_parts * 128 + 1,), nan, device="cuda")[1:].view(B, hq, n_parts, 128),
          torch.full((B * hq * n_parts * 2 + 1,), nan, device="cuda")[1:].view(B, hq, n_parts, 2))
    ops.decode_attention(q.cuda(), kc.cuda(), vc.cuda(), bt, lens.cuda(), scale, out, n_parts, workspace=ws)
    got = out.cpu()
    assert bool((got[[b for b in range(B) if not ctx[b]]] == 0).all())
    # bf16 weights (2^-9 each, of values of order one) and one rounding of the result
    err = (got[live].float() - want.float()).abs().max()
    assert float(err) < 2 ** -7 * max(1.0, float(want.float().abs().max())), float(err)


@pytest.mark.gpu
@pytest.mark.parametrize("at", [0, 700, 1999])
@pytest.mark.parametrize("n_parts", [1, 2, 16, 70])
@pytest.mark.parametrize("mfma", ["0", "1"])
def test_rows_that_see_a_nan(monkeypatch, mfma, n_parts, at):
    """A key that holds a NaN, in the first, a middle and the last part: the query heads of its key head are NaN, not 0."""
    monkeypatch.setenv("DX_DECODE_MFMA", mfma)
    torch.manual_seed(n_parts)
    hq, hkv, bs, lens = 8, 2, 16, torch.tensor([2000, 300], dtype=torch.int32)
    table = torch.arange(2 * 125, dtype=torch.int32).view(2, 125)
    kc, vc = (torch.randn(250, hkv, bs, 128).bfloat16() for _ in range(2))
    q, scale = torch.randn(2, hq, 128).bfloat16(), 1 / math.sqrt(128)
    want = ref.paged_attention(q, kc, vc, table, torch.arange(3, dtype=torch.int32), lens, scale, bs)
    kc[at // bs, 1, at % bs, 3] = float("nan")
    out = torch.empty(2, hq, 128, dtype=torch.bfloat16, device="cuda")
    got = ops.decode_attention(q.cuda(), kc.cuda(), vc.cuda(), table.cuda(), lens.cuda(), scale, out, n_parts).cpu()
    assert bool(got[0, 4:].isnan().all())
    for g, w in ((got[0, :4], want[0, :4]), (got[1], want[1])):  # (bound of test_parts)
        assert float((g.float() - w.float()).abs().max()) < 2 ** -7 * max(1.0, float(want.float().abs().max()))


@pytest.mark.gpu
@pytest.mark.parametrize("n_parts", [3, 17, 33])
@pytest.mark.parametrize("mfma,bs", [("1", 16), ("1", 48), ("1", 64), ("0", 64)])
def test_part_lengths(monkeypatch, mfma, bs, n_parts):
    """Shares of a context around a quarter, a half and the whole of a workgroup's stride, so around the lengths at which
    parts get coarser; blocks of one, of a ragged number and of a whole number of a wave's 32 tokens."""
    monkeypatch.setenv("DX_DECODE_MFMA", mfma)
    torch.manual_seed(n_parts)
    hq, hkv = 8, 2
    ctx = [n_parts * k + e for k in (16, 32, 64, 128) for e in (-1, 0, 1)]
    need = [-(-c // bs) for c in ctx]
    table = torch.zeros(len(ctx), max(need), dtype=torch.int32)
    ids = torch.randperm(sum(need)).to(torch.int32)
    for b, n in enumerate(need):
        table[b, :n] = ids[sum(need[:b]):sum(need[:b]) + n]
    kc, vc = (torch.randn(sum(need), hkv, bs, 128).bfloat16() for _ in range(2))
    q, lens, scale = torch.randn(len(ctx), hq, 128).bfloat16(), torch.tensor(ctx, dtype=torch.int32), 1 / math.sqrt(128)
    want = ref.paged_attention(q, kc, vc, table, torch.arange(len(ctx) + 1, dtype=torch.int32), lens, scale, bs)
    out = torch.empty(len(ctx), hq, 128, dtype=torch.bfloat16, device="cuda")
    got = ops.decode_attention(q.cuda(), kc.cuda(), vc.cuda(), table.cuda(), lens.cuda(), scale, out, n_parts).cpu()
    err = (got.float() - want.float()).abs().max()  # (bound of test_parts)
    assert float(err) < 2 ** -7 * max(1.0, float(want.float().abs().max())), float(err)
