"""Prompt rows on csrc/mixers/prompt_attention.hip and decode rows on csrc/mixers/decode_attention.hip: pages of whole
64-key tiles, heads of 128 columns (values of 128 or 256) or one shared row of 256 columns, every score form, against
dense float64 arithmetic over the bf16 inputs.  The pages' unused rows hold NaN."""
from __future__ import annotations

import re
from pathlib import Path

import numpy as np
import pytest
import torch

from dynamo_exp_amd.ops import mixers as mx

# n_qh, maps, group, d, dv, form; group 2 takes two heads a workgroup, 4 and 8 four; "shared": one row is key and value
FORMS = {
    "plain": (8, 1, 4, 128, 128), "plain pair": (6, 1, 2, 128, 128), "fine": (8, 1, 8, 128, 128),
    "capped": (4, 1, 2, 128, 128), "penalty": (8, 1, 4, 128, 128), "both": (8, 1, 4, 128, 128),
    "sigmoid": (8, 1, 4, 128, 128), "sigmoid capped": (4, 1, 2, 128, 128), "diff": (16, 2, 4, 128, 256),
    "diff pair": (8, 2, 2, 128, 256), "shared": (16, 1, 16, 256, 192),
    "shared wide": (8, 1, 8, 256, 256), "shared pair": (6, 1, 6, 256, 192), "gated": (8, 1, 4, 128, 128),
}
MASKS = [("causal", 0, 0), ("window", 70, 0), ("window", 1, 0), ("window", 100, 5), ("window", 66, 64), ("window", 40, 130),
         ("chunk", 50, 0), ("chunk", 256, 0)]


def dense(q, k, v, pos, scale, mask, size, keep, cap, db, sink, sig, hb):
    """q [R, n_qh, d], k [n, n_qh, d], v [n, n_qh, dv] float64 -> [R, n_qh, dv]."""
    s = torch.einsum("ihd,jhd->hij", q, k) * scale
    p, j = pos[:, None], torch.arange(k.shape[0])[None, :]
    if cap:
        s = cap * torch.tanh(s / cap)
    if db is not None:
        s = s - db[0].double()[:, None, None] * torch.log1p(db[1].double()[:, None, None] * (p - j).clamp_min(0)[None])
    vis = (j <= p) & ((j >= mx.first_visible(p, mask, size)) | (j < keep))
    if sig:
        w = torch.sigmoid(s + hb.double()[:, None, None]) * vis
    else:
        s = s.masked_fill(~vis, float("-inf"))
        if sink is not None:
            s = torch.cat([s, sink.double()[:, None, None].expand(-1, s.shape[1], 1)], -1)
        w = torch.softmax(s, -1)[..., :k.shape[0]]
    return torch.einsum("hij,jhd->ihd", w, v)



def terms(form, n_qh):
    """(cap, distance penalty, sigmoid weights, bias, sink) of a form."""
    cap = 2.0 if form in ("capped", "both", "sigmoid capped") else 0.0
    db = (torch.rand(n_qh), torch.rand(n_qh) + 0.1) if form in ("penalty", "both") else None
    sig = form.startswith("sigmoid")
    hb = torch.randn(n_qh) - 2.0 if sig else None
    sink = torch.randn(n_qh) if form in ("shared", "shared wide", "plain") else None
    return cap, db, sig, hb, sink


def pages(form, lengths, bs):
    """Caches of sequences of these lengths over shuffled pages: (kc, vc, table, [(K, V) float64 per query vector])."""
    n_qh, maps, group, d, dv = FORMS[form]
    shared, G = form.startswith("shared"), n_qh // maps // group
    heads = torch.arange(n_qh) // maps
    kh, vh = heads // group * maps + torch.arange(n_qh) % maps, heads // group
    nb = [-(-n // bs) for n in lengths]
    perm = torch.randperm(sum(nb)).to(torch.int32)
    table = torch.zeros(len(lengths), max(nb), dtype=torch.int32)
    kc = torch.full((sum(nb) * bs, d if shared else G * maps * d), float("nan"), dtype=torch.bfloat16)
    vc = kc if shared else torch.full((sum(nb) * bs, G * dv), float("nan"), dtype=torch.bfloat16)
    at, kv = 0, []
    for i, n in enumerate(lengths):
        table[i, :nb[i]] = perm[at:at + nb[i]]
        at += nb[i]
        sl = table[i].long()[torch.arange(n) // bs] * bs + torch.arange(n) % bs
        kc[sl] = (torch.randn(n, kc.shape[1]) * 1.5).bfloat16()
        if shared:
            K = kc[sl].double()[:, None].expand(n, n_qh, d)
            kv.append((K, K[:, :, :dv]))
        else:
            vc[sl] = torch.randn(n, vc.shape[1]).bfloat16()
            kv.append((kc[sl].double().view(n, -1, d)[:, kh], vc[sl].double().view(n, -1, dv)[:, vh]))
    kd = kc.cuda()
    return kd, kd if shared else vc.cuda(), table.cuda(), kv


def cuda(t):
    return None if t is None else t.cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("mask,size,keep", MASKS)
@pytest.mark.parametrize("form", FORMS)
def test_prompt_rows(form, mask, size, keep):
    """Portions of 257, 33 and 1 rows that start at 0 and inside a cached prefix; the second sequence's last tile holds a
    single key."""
    n_qh, maps, group, d, dv = FORMS[form]
    torch.manual_seed(11)
    scale = 0.7 * d ** -0.5
    starts, rows = [43, 32, 0], [257, 33, 1]
    cap, db, sig, hb, sink = terms(form, n_qh)
    gate = torch.randn(sum(rows), n_qh // maps + 3).bfloat16()[:, :n_qh // maps] if form == "gated" else None
    for bs in (64, 128):
        kd, vd, table, kv = pages(form, [s + r for s, r in zip(starts, rows)], bs)
        q = torch.randn(sum(rows), n_qh * d + 8).bfloat16()[:, :n_qh * d]  # rows wider than the heads
        want = []
        for i, (s, r) in enumerate(zip(starts, rows)):
            r0 = sum(rows[:i])
            want.append(dense(q[r0:r0 + r].double().reshape(r, n_qh, d), *kv[i], torch.arange(s, s + r), scale, mask, size,
                              keep, cap, db, sink, sig, hb))
        want = torch.cat(want)
        if gate is not None:
            want = want * torch.sigmoid(gate.double()).repeat_interleave(maps, 1)[:, :, None]
        pos = torch.cat([torch.arange(s, s + r) for s, r in zip(starts, rows)]).cuda()
        seq = torch.tensor([i for i, r in enumerate(rows) for _ in range(r)], dtype=torch.int32).cuda()
        tiles = torch.tensor([t for i in range(3) for t in mx.tile_list(sum(rows[:i]), rows[i])], dtype=torch.int32).cuda()
        out_f32 = form.startswith("diff")
        got = mx.attention(q.cuda(), kd, vd, pos, seq, table, bs, n_qh, maps, group, d, dv, scale, mask, size, 1, out_f32,
                           tiles, sum(rows), softcap=cap, dist_bias=None if db is None else tuple(map(cuda, db)),
                           weights="sigmoid" if sig else "softmax", head_bias=cuda(hb), head_gate=cuda(gate),
                           keep_first=keep, sink=cuda(sink), fine_weights=form == "fine").cpu().double()
        err = float((got - want).abs().max())
        # a bf16 result: its rounding (2^-9 of it) and one rounding of every weight (2^-9 of sum w |v|, |v| < 5 here
        # and weights that sum to 1, or for sigmoid weights to their sum); fp32: two bf16 numbers per weight, 2^-17,
        # and the hardware's exp2, logarithm and reciprocal in the scores
        top = float(want.abs().max())
        assert err < (3e-4 if out_f32 else 2.0 ** -8 * (top + (top if sig else 5.0))), err


@pytest.mark.gpu
@pytest.mark.parametrize("mask,size,keep", MASKS)
@pytest.mark.parametrize("form", FORMS)
def test_decode_rows(form, mask, size, keep):
    """Contexts that end at, in front of and behind the edges of 32-key tiles and pages, in one, three and nine parts
    (some of them, and some waves, without a key), as row i = sequence i and by sequence numbers."""
    n_qh, maps, group, d, dv = FORMS[form]
    torch.manual_seed(13)
    scale = 0.7 * d ** -0.5
    ctx = [1, 31, 32, 33, 64, 65, 300, 129]
    B = len(ctx)
    cap, db, sig, hb, sink = terms(form, n_qh)
    gate = torch.randn(B, n_qh // maps + 3).bfloat16()[:, :n_qh // maps] if form == "gated" else None
    for bs, parts, out_f32, by_seq in ((64, 1, True, False), (128, 3, True, True), (64, 9, True, False), (64, 3, False, False),
                                       (64, 1, False, True)):
        kd, vd, table, kv = pages(form, ctx, bs)
        q = torch.randn(B, n_qh * d + 8).bfloat16()[:, :n_qh * d]
        want = torch.cat([dense(q[i:i + 1].double().reshape(1, n_qh, d), *kv[i], torch.tensor([c - 1]), scale, mask, size, keep,
                                cap, db, sink, sig, hb) for i, c in enumerate(ctx)])
        if gate is not None:
            want = want * torch.sigmoid(gate.double()).repeat_interleave(maps, 1)[:, :, None]
        pos = torch.tensor([c - 1 for c in ctx]).cuda()
        order = torch.randperm(B) if by_seq else torch.arange(B)
        seq = order.to(torch.int32).cuda() if by_seq else None
        got = mx.attention(q[order].cuda(), kd, vd, pos[order.cuda()], seq, table, bs, n_qh, maps, group, d, dv, scale, mask,
                           size, parts, out_f32, softcap=cap, dist_bias=None if db is None else tuple(map(cuda, db)),
                           weights="sigmoid" if sig else "softmax", head_bias=cuda(hb),
                           head_gate=None if gate is None else gate[order].cuda(), keep_first=keep,
                           sink=cuda(sink)).cpu().double()
        err = float((got - want[order]).abs().max())
        # fp32: weights as two bf16 numbers, 2^-17 of sum w |v|; bf16: one rounding of the result on top
        top = float(want.abs().max())
        assert err < (3e-4 if not sig else 3e-4 * max(top, 1.0)) + (0.0 if out_f32 else 2.0 ** -8 * top), (bs, parts, err)


@pytest.mark.gpu
@pytest.mark.parametrize("rate", [0.1, 1.0, 100.0, 1e4, 6.3e5, 1e7, 1e12])
@pytest.mark.parametrize("form", ["penalty", "both"])
def test_penalty_of_any_rate(form, rate):
    """The log-distance penalty from slow rates to ones whose product with a distance leaves no bit of the 1 beside it,
    where a row's own key (distance 0) still pays nothing: prompt rows at every place of a key tile and a decode row."""
    n_qh, maps, group, d, dv = FORMS[form]
    torch.manual_seed(17)
    scale, starts, rows = 0.7 * d ** -0.5, [43, 0, 199], [70, 97, 1]
    cap = terms(form, n_qh)[0]
    db = (torch.rand(n_qh) + 0.2, rate * (torch.rand(n_qh) + 0.5))
    kd, vd, table, kv = pages(form, [s + r for s, r in zip(starts, rows)], 64)
    q, T, Tp = torch.randn(sum(rows), n_qh * d).bfloat16(), sum(rows), sum(rows[:2])
    want = []
    for i, (s, r) in enumerate(zip(starts, rows)):
        r0 = sum(rows[:i])
        want.append(dense(q[r0:r0 + r].double().reshape(r, n_qh, d), *kv[i], torch.arange(s, s + r), scale, "window", 100, 0,
                          cap, db, None, False, None))
    want = torch.cat(want)
    pos = torch.cat([torch.arange(s, s + r) for s, r in zip(starts, rows)]).cuda()
    seq = torch.tensor([i for i, r in enumerate(rows) for _ in range(r)], dtype=torch.int32).cuda()
    tiles = torch.tensor([t for i in range(2) for t in mx.tile_list(sum(rows[:i]), rows[i])], dtype=torch.int32).cuda()
    got = mx.attention(q.cuda(), kd, vd, pos, seq, table, 64, n_qh, maps, group, d, dv, scale, "window", 100, 3, False, tiles, Tp,
                       softcap=cap, dist_bias=tuple(map(cuda, db))).cpu().double()
    # as test_prompt_rows: the result's rounding to bf16 and one rounding of every weight
    err, top = float((got - want).abs().max()), float(want.abs().max())
    assert err < 2.0 ** -8 * (top + 5.0), err


# heads of the long contexts: shared rows for 20, 32 and 40 heads take blocks of 32 query vectors, 40 of them two workgroups
LONG = {"plain": FORMS["plain"], "both": FORMS["both"], "sigmoid": FORMS["sigmoid"], "diff": FORMS["diff"],
        **{f"shared {H} / {dv}": (H, 1, H, 256, dv) for H in (16, 20, 32, 40) for dv in (192, 256)}}


@pytest.mark.gpu
@pytest.mark.parametrize("mask,size,keep", [("causal", 0, 0), ("window", 1500, 0), ("window", 1000, 64), ("chunk", 2048, 0)])
@pytest.mark.parametrize("form", LONG)
def test_decode_rows_of_long_contexts(form, mask, size, keep):
    """Contexts of 11 to 188 tiles in three to nine parts that hold keys, up to 21 tiles each (an even and an odd number a
    wave), on pages of one, two and four tiles; float64 on the GPU."""
    n_qh, maps, group, d, dv = LONG[form]
    kind = form.split()[0]
    torch.manual_seed(31)
    scale, ctx = 0.7 * d ** -0.5, [700, 3500, 6000, 351]
    G, heads, B = n_qh // maps // group, torch.arange(n_qh, device="cuda") // maps, len(ctx)
    kh, vh = heads // group * maps + torch.arange(n_qh, device="cuda") % maps, heads // group
    cap, db, sig, hb, sink = terms("shared" if kind == "shared" else kind, n_qh)
    for bs, parts in ((32, 3), (64, 5), (128, 9)):
        nb = [-(-n // bs) for n in ctx]
        perm = torch.randperm(sum(nb), device="cuda").to(torch.int32)
        table = torch.zeros(B, max(nb), dtype=torch.int32, device="cuda")
        kc = torch.full((sum(nb) * bs, d if kind == "shared" else G * maps * d), float("nan"), device="cuda").bfloat16()
        vc = kc if kind == "shared" else torch.full((sum(nb) * bs, G * dv), float("nan"), device="cuda").bfloat16()
        q, at, want = torch.randn(B, n_qh * d, device="cuda").bfloat16(), 0, []
        for i, n in enumerate(ctx):
            table[i, :nb[i]] = perm[at:at + nb[i]]
            at += nb[i]
            j = torch.arange(n, device="cuda")
            sl = table[i].long()[j // bs] * bs + j % bs
            kc[sl] = (torch.randn(n, kc.shape[1], device="cuda") * 1.5).bfloat16()
            if kind == "shared":
                K = kc[sl].double()[:, None].expand(n, n_qh, d)
                V = K[:, :, :dv]
            else:
                vc[sl] = torch.randn(n, vc.shape[1], device="cuda").bfloat16()
                K, V = kc[sl].double().view(n, -1, d)[:, kh], vc[sl].double().view(n, -1, dv)[:, vh]
            # (float64 scores as sums, not as a batched product)
            s = torch.stack([K[:, h] @ q[i, h * d:(h + 1) * d].double() for h in range(n_qh)]) * scale
            p = n - 1
            if cap:
                s = cap * torch.tanh(s / cap)
            if db is not None:
                s = s - cuda(db[0]).double()[:, None] * torch.log1p(cuda(db[1]).double()[:, None] * (p - j)[None])
            vis = (j >= int(mx.first_visible(torch.tensor([p]), mask, size))) | (j < keep)
            if sig:
                w = torch.sigmoid(s + cuda(hb).double()[:, None]) * vis
            else:
                s = s.masked_fill(~vis, float("-inf"))
                if sink is not None:
                    s = torch.cat([s, cuda(sink).double()[:, None]], -1)
                w = torch.softmax(s, -1)[:, :n]
            want.append(torch.stack([w[h] @ V[:, h] for h in range(n_qh)]))
        want = torch.stack(want)
        got = mx.attention(q, kc, vc, torch.tensor([c - 1 for c in ctx]).cuda(), None, table, bs, n_qh, maps, group, d, dv, scale,
                           mask, size, parts, True, softcap=cap, dist_bias=None if db is None else tuple(map(cuda, db)),
                           weights="sigmoid" if sig else "softmax", head_bias=cuda(hb), keep_first=keep, sink=cuda(sink)).double()
        err, top = float((got - want).abs().max()), float(want.abs().max())
        # as test_decode_rows: weights as two bf16 numbers, 2^-17 of sum w |v|
        assert err < 3e-4 * (max(top, 1.0) if sig else 1.0), (bs, parts, err, top)


@pytest.mark.gpu
@pytest.mark.parametrize("form,mask,size,keep", [("plain", "causal", 0, 0), ("fine", "window", 4500, 70),
                                                 ("diff", "window", 4300, 64), ("shared", "chunk", 4200, 0),
                                                 ("both", "window", 130, 4100)])
def test_prompt_rows_behind_many_pages(form, mask, size, keep):
    """More pages than lanes of a wave, tables that are read a second time in the middle of a row's keys (and, with
    kept keys, go back to the front)."""
    n_qh, maps, group, d, dv = FORMS[form]
    torch.manual_seed(5)
    scale, start, rows, bs = 0.7 * d ** -0.5, 4470, 97, 64
    cap, db, sig, hb, sink = terms(form, n_qh)
    kd, vd, table, kv = pages(form, [start + rows], bs)
    q = torch.randn(rows, n_qh * d).bfloat16()
    want = dense(q.double().view(rows, n_qh, d), *kv[0], torch.arange(start, start + rows), scale, mask, size, keep, cap, db,
                 sink, sig, hb)
    tiles = torch.tensor(mx.tile_list(0, rows), dtype=torch.int32).cuda()
    out_f32 = form.startswith("diff")
    got = mx.attention(q.cuda(), kd, vd, torch.arange(start, start + rows).cuda(), torch.zeros(rows, dtype=torch.int32).cuda(),
                       table, bs, n_qh, maps, group, d, dv, scale, mask, size, 1, out_f32, tiles, rows, softcap=cap,
                       dist_bias=None if db is None else tuple(map(cuda, db)), head_bias=cuda(hb), keep_first=keep,
                       sink=cuda(sink), fine_weights=form == "fine").cpu().double()
    err = float((got - want).abs().max())  # (bounds of test_prompt_rows)
    assert err < (3e-4 if out_f32 else 2.0 ** -8 * (float(want.abs().max()) + 5.0)), err


@pytest.mark.gpu
def test_later_rows_values_that_are_not_finite():
    """Two blocks of 32 rows in a workgroup and tiles of 64 keys: an infinite value of the second block's rows is none of
    the first block's."""
    n_qh, maps, group, d, dv = FORMS["plain pair"]
    torch.manual_seed(6)
    kd, vd, table, kv = pages("plain pair", [64], 64)
    vd[int(table[0, 0]) * 64 + 40] = float("inf")
    q = torch.randn(64, n_qh * d).bfloat16()
    want = dense(q.double().view(64, n_qh, d), *kv[0], torch.arange(64), d ** -0.5, "causal", 0, 0, 0.0, None, None, False,
                 None)[:32]
    tiles = torch.tensor(mx.tile_list(0, 64), dtype=torch.int32).cuda()
    got = mx.attention(q.cuda(), kd, vd, torch.arange(64).cuda(), torch.zeros(64, dtype=torch.int32).cuda(), table, 64, n_qh,
                       maps, group, d, dv, d ** -0.5, "causal", 0, 1, False, tiles, 64).cpu().double()[:32]
    assert float((got - want).abs().max()) < 2.0 ** -8 * (float(want.abs().max()) + 5.0)


@pytest.mark.gpu
@pytest.mark.parametrize("mask,size", [("window", 1216), ("window", 1217), ("chunk", 1216), ("window", 33), ("window", 1)])
@pytest.mark.parametrize("form,cap", [("both", 30.0), ("both", 3.0), ("penalty", 0.0), ("both pair", 12.0)])
def test_score_terms_of_limited_distance(form, cap, mask, size):
    """Penalties from the table of distances (up to 1216 keys back, with the first and the last entry in use) and beside
    it; caps far above the scores (polynomial in every tile), near them (in some) and among them (in none)."""
    n_qh, maps, group, d, dv = FORMS["plain pair" if form == "both pair" else form]
    torch.manual_seed(7)
    scale, start, rows, bs = 0.7 * d ** -0.5, 1190, 131, 64
    db = (torch.rand(n_qh) * 2, torch.rand(n_qh) * 3 + 0.1)
    kd, vd, table, kv = pages("plain pair" if form == "both pair" else form, [start + rows], bs)
    q = torch.randn(rows, n_qh * d).bfloat16()
    want = dense(q.double().view(rows, n_qh, d), *kv[0], torch.arange(start, start + rows), scale, mask, size, 0, cap, db, None,
                 False, None)
    tiles = torch.tensor(mx.tile_list(0, rows), dtype=torch.int32).cuda()
    got = mx.attention(q.cuda(), kd, vd, torch.arange(start, start + rows).cuda(), torch.zeros(rows, dtype=torch.int32).cuda(),
                       table, bs, n_qh, maps, group, d, dv, scale, mask, size, 1, False, tiles, rows, softcap=cap,
                       dist_bias=tuple(map(cuda, db))).cpu().double()
    err = float((got - want).abs().max())  # (bound of test_prompt_rows)
    assert err < 2.0 ** -8 * (float(want.abs().max()) + 5.0), err


@pytest.mark.gpu
@pytest.mark.parametrize("form,cap", [("both", 30.0), ("both", 50.0), ("penalty", 0.0)])
@pytest.mark.parametrize("old", [(), (100,), (100, 250, 640), (3, 4, 870)])
def test_penalty_rows_whose_old_keys_count(form, cap, old):
    """Maxima among the first tiles, behind them and in the last one; scores on both sides of what each polynomial of the cap takes."""
    n_qh, maps, group, d, dv = FORMS[form]
    torch.manual_seed(13)
    scale, start, rows, bs, size = 0.7 * d ** -0.5, 900, 40, 64, 1000
    db = (torch.rand(n_qh), torch.rand(n_qh) + 0.1)
    kd, vd, table, kv = pages(form, [start + rows], bs)
    for i, j in enumerate(old):  # (powers of two: the keys stay bf16)
        kd[int(table[0, j // bs]) * bs + j % bs] *= 4 << i % 2
        kv[0][0][j] *= 4 << i % 2
    q = torch.randn(rows, n_qh * d).bfloat16()
    want = dense(q.double().view(rows, n_qh, d), *kv[0], torch.arange(start, start + rows), scale, "window", size, 0, cap, db,
                 None, False, None)
    tiles = torch.tensor(mx.tile_list(0, rows), dtype=torch.int32).cuda()
    got = mx.attention(q.cuda(), kd, vd, torch.arange(start, start + rows).cuda(), torch.zeros(rows, dtype=torch.int32).cuda(),
                       table, bs, n_qh, maps, group, d, dv, scale, "window", size, 1, False, tiles, rows, softcap=cap,
                       dist_bias=tuple(map(cuda, db))).cpu().double()
    # (bound of test_prompt_rows)
    assert float((got - want).abs().max()) < 2.0 ** -8 * (float(want.abs().max()) + 5.0)


@pytest.mark.parametrize("name,limit", [("kTanh", "kTanhMax"), ("kTanhFew", "kTanhMin")])
def test_polynomials_of_the_cap(name, limit):
    """tanh(y) / y as the kernel's coefficients give it over the range that each polynomial is taken for.  (The bounds of the
    results above could not tell: 1e-4 of a score is far below the rounding of a weight.)"""
    text = (Path(mx.__file__).parents[1] / "csrc" / "mixers" / "prompt_attention.hip").read_text()
    coef = [float(np.float32(x)) for x in re.search(rf"\b{name}\[\d\] = {{(.*?)}}", text)[1].replace("f", "").split(",")]
    top = float(re.search(rf"\b{limit} = ([\d.]+)f", text)[1])
    y = np.linspace(1e-6, top, 200001)
    exact = np.tanh(y) / y
    far = lambda c: np.abs(sum(a * y ** (2 * i) for i, a in enumerate(c)) / exact - 1).max()
    assert far(coef) < 6.3e-8, far(coef)
    # evaluated as the kernel does, in 32 bits: 2^-24 each for the leading coefficient times the scale, the sum and the product
    # (the other terms are 4 % of it at most)
    f = np.float32
    for s in (0.05, 1.0, 37.0):  # score = s y
        x, y2 = (s * y).astype(f), f(f(1 / s) * f(1 / s))
        c = [f(f(s) * f(a)) for a in coef]  # (scale and cap: the polynomial of x, times the cap)
        u = [f(c[i] * f(f(1 / s) * f(y2 ** i))) for i in range(len(c))]
        t, r = x * x, np.full_like(x, u[-1])
        for a in u[-2::-1]:
            r = (t.astype(np.float64) * r + a).astype(f)
        got = (x * r).astype(np.float64) / s
        assert np.abs(got / np.tanh(x.astype(np.float64) / s) - 1).max() < 6.3e-8 + 3 * 2.0 ** -24


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [600, 1501])
@pytest.mark.parametrize("form,keys", [("shared", 32), ("shared wide", 32), ("plain", 64)])
def test_rounding_of_the_weights(form, keys, rows):
    """A weight that enters its product as one bf16 is rounded relative to the maximum so far, so a row's largest weight in a
    tile that raises it is exactly 1: with tiles of more keys there are fewer of those.  The distance from exact sums is
    that of weights rounded tile by tile."""
    n_qh, maps, group, d, dv = FORMS[form]
    torch.manual_seed(17)
    scale = d ** -0.5
    kd, vd, table, ((K, V),) = pages(form, [rows], 64)
    q = torch.randn(rows, n_qh * d).bfloat16().cuda()
    tiles = torch.tensor(mx.tile_list(0, rows), dtype=torch.int32).cuda()
    pos = torch.arange(rows).cuda()
    got = mx.attention(q, kd, vd, pos, torch.zeros(rows, dtype=torch.int32).cuda(), table, 64, n_qh, maps, group, d, dv, scale,
                       "causal", 0, 1, False, tiles, rows).double().view(rows, n_qh, dv).transpose(0, 1)
    Q, K, V = (t.transpose(0, 1).contiguous() for t in (q.double().view(rows, n_qh, d), K.cuda(), V.cuda()))
    S = ((Q @ K.transpose(1, 2).contiguous()) * scale).masked_fill(pos[None, None] > pos[None, :, None], float("-inf"))
    want = torch.softmax(S, -1) @ V
    m = torch.full((n_qh, rows, 1), float("-inf"), dtype=torch.float64, device="cuda")
    l, O = torch.zeros_like(m), torch.zeros_like(want)
    for at in range(0, rows, keys):
        s = S[:, :, at:at + keys]
        new = torch.maximum(m, s.amax(-1, keepdim=True))
        w, fade = torch.exp(s - new), torch.exp(m - new)
        l, O, m = l * fade + w.sum(-1, keepdim=True), O * fade + w.bfloat16().double() @ V[:, at:at + keys].contiguous(), new
    far = lambda x: float((x - want).norm() / want.norm())
    # (twice as many keys a tile: 0.5 % more; the kernel's own sums and exponentials are in 32 bits, 2^-14 of a rounding to bf16)
    assert far(got) <= 1.002 * far((O / l).bfloat16().double()), (far(got), far((O / l).bfloat16().double()))


@pytest.mark.gpu
@pytest.mark.parametrize("mask,size", [("causal", 0), ("chunk", 1500)])
@pytest.mark.parametrize("form", ["shared", "plain", "diff", "sigmoid"])
@pytest.mark.parametrize("ctx", [[4000, 33, 1, 2500, 700], [1, 3000], [300 + 61 * i for i in range(20)],
                                 [1 + 37 * (i % 9) for i in range(64)], [65] * 65], ids=len)
def test_decode_parts_of_unequal_rows(ctx, form, mask, size):
    """Rows of one tile beside rows of a hundred, more parts asked for than there are tiles."""
    n_qh, maps, group, d, dv = FORMS[form]
    torch.manual_seed(17)
    scale, B, bs = 0.7 * d ** -0.5, len(ctx), 64
    cap, db, sig, hb, sink = terms(form, n_qh)
    kd, vd, table, kv = pages(form, ctx, bs)
    q = torch.randn(B, n_qh * d).bfloat16()
    want = torch.cat([dense(q[i:i + 1].double().reshape(1, n_qh, d), *kv[i], torch.tensor([c - 1]), scale, mask, size, 0, cap, db,
                            sink, sig, hb) for i, c in enumerate(ctx)])
    for parts in (2, 16):
        got = mx.attention(q.cuda(), kd, vd, torch.tensor([c - 1 for c in ctx]).cuda(), None, table, bs, n_qh, maps, group, d, dv,
                           scale, mask, size, parts, True, weights="sigmoid" if sig else "softmax", head_bias=cuda(hb),
                           sink=cuda(sink)).cpu().double()
        err, top = float((got - want).abs().max()), float(want.abs().max())
        assert err < 3e-4 * (max(top, 1.0) if sig else 1.0), (parts, err)  # (bound of test_decode_rows, fp32 results)


@pytest.mark.gpu
@pytest.mark.parametrize("mask,size", [("window", 100), ("causal", 0)])
@pytest.mark.parametrize("form", ["both", "both pair", "penalty", "sigmoid capped"])
def test_scores_of_the_last_channels(form, mask, size):
    """Scores that the last product of a row makes alone (the other channels are 0), most of them at 1 to 4 times the cap: what
    the cap is decided by waits for that product."""
    n_qh, maps, group, d, dv = FORMS["plain pair" if form == "both pair" else form]
    torch.manual_seed(19)
    scale, start, rows, bs, sig = 0.7 * d ** -0.5, 75, 131, 64, form == "sigmoid capped"
    cap = 0.0 if form == "penalty" else 0.3
    db = None if sig else (torch.rand(n_qh) * 2, torch.rand(n_qh) * 3 + 0.1)
    hb = torch.randn(n_qh) - 2.0 if sig else None
    kd, vd, table, kv = pages("plain pair" if form == "both pair" else form, [start + rows], bs)
    last = (torch.arange(d) >= d - 16).double()
    kd = (kd.view(-1, d) * last.bfloat16().cuda()).view(kd.shape)
    q = (torch.randn(rows, n_qh, d) * 3 * last).bfloat16()
    want = dense(q.double(), kv[0][0] * last, kv[0][1], torch.arange(start, start + rows), scale, mask, size, 0, cap, db, None, sig,
                 hb)
    tiles = torch.tensor(mx.tile_list(0, rows), dtype=torch.int32).cuda()
    got = mx.attention(q.view(rows, -1).cuda(), kd, vd, torch.arange(start, start + rows).cuda(),
                       torch.zeros(rows, dtype=torch.int32).cuda(), table, bs, n_qh, maps, group, d, dv, scale, mask, size, 1,
                       False, tiles, rows, softcap=cap, dist_bias=None if db is None else tuple(map(cuda, db)),
                       weights="sigmoid" if sig else "softmax", head_bias=cuda(hb)).cpu().double()
    err, top = float((got - want).abs().max()), float(want.abs().max())  # (bound of test_prompt_rows)
    assert err < 2.0 ** -8 * (top + (top if sig else 5.0)), err


@pytest.mark.gpu
@pytest.mark.parametrize("cap", [1e6, 1e25, 1e38])
@pytest.mark.parametrize("form", ["both", "both pair", "capped", "sigmoid capped"])
def test_scores_and_caps_at_the_ends_of_the_number_range(form, cap):
    """Scores of 1e20 below caps that are larger still (and, at 1e6, far above it): a row that sees itself alone gets its own
    value."""
    n_qh, maps, group, d, dv = FORMS["plain pair" if form == "both pair" else form]
    torch.manual_seed(23)
    rows, sig = 70, form == "sigmoid capped"
    db = (torch.rand(n_qh), torch.rand(n_qh) + 0.1) if form.startswith("both") else None
    kd, vd, table, kv = pages("plain pair" if form == "both pair" else form, [rows], 64)
    tiles = torch.tensor(mx.tile_list(0, rows), dtype=torch.int32).cuda()
    got = mx.attention(torch.full((rows, n_qh * d), 1e10).bfloat16().cuda(), torch.full_like(kd, 1e8), vd,
                       torch.arange(rows).cuda(), torch.zeros(rows, dtype=torch.int32).cuda(), table, 64, n_qh, maps, group, d, dv,
                       d ** -0.5, "window", 1, 1, False, tiles, rows, softcap=cap,
                       dist_bias=None if db is None else tuple(map(cuda, db)), weights="sigmoid" if sig else "softmax",
                       head_bias=torch.zeros(n_qh).cuda() if sig else None)
    want = kv[0][1]
    if sig and cap == 1e38:  # (2^-24 of the cap: the score is lost in its rounding)
        want = want / 2
    assert torch.equal(got.cpu().double(), want)


CUT_AT_500 = ("capped", "penalty", "both", "diff pair", "shared wide", "shared pair")


@pytest.mark.parametrize("form", FORMS)
def test_rule_of_prompt_parts(form):
    """The keys that a row sees decide, not the context: a window's and those behind the start of a chunk, of which rows that reach
    back over it see a whole one; many rows are not cut."""
    n_qh, maps, group, d, dv = FORMS[form]

    def cut(rows, tiles, keys, mask="causal", size=0, keep=0, heads=n_qh):
        return mx._prompt_parts(rows, tiles, keys, mask, size, keep, heads, maps, heads // maps if form.startswith("shared") else group,
                                d, dv, 64, form.startswith("shared"), form in ("capped", "penalty", "both", "sigmoid capped"),
                                int(form.startswith("sigmoid")), form.startswith("diff"), form == "fine")[0] > 1

    assert cut(88, 3, 1088) and not cut(16, 1, 128) and not cut(1024, 8, 100000, heads=64 * n_qh)
    for size in (900, 2000):
        assert cut(88, 3, 100000, "window", size, 70)
    assert cut(88, 3, 100000, "window", 300, 70) == (form in CUT_AT_500) == cut(88, 3, 498)
    assert not cut(16, 1, 100000, "window", 100)
    for keys, seen in ((999, True), (1000, True), (1001, True), (1016, True), (1017, False), (1100, False), (1990, True), (2000, True),
                       (2016, True), (2017, False)):
        assert cut(16, 1, keys, "chunk", 1000) == seen, keys


@pytest.mark.gpu
@pytest.mark.parametrize("parts", [None, (2, 0), (3, 0), (8, 0), (4, 200)])
@pytest.mark.parametrize("mask,size,keep", [("causal", 0, 0), ("window", 300, 70), ("chunk", 500, 0), ("window", 900, 70),
                                            ("chunk", 1000, 0)])
@pytest.mark.parametrize("form", FORMS)
def test_prompt_rows_in_parts(monkeypatch, form, mask, size, keep, parts):
    """Few prompt rows behind long contexts, their keys cut into parts (None: as many as the rule takes): parts without a
    tile, rows that see nothing of a part, rows of one sequence that has a single tile, workgroups that stay whole."""
    n_qh, maps, group, d, dv = FORMS[form]
    torch.manual_seed(17)
    scale = 0.7 * d ** -0.5
    starts, rows, bs = [1030, 0, 491], [17, 1, 70], 64
    cap, db, sig, hb, sink = terms(form, n_qh)
    gate = torch.randn(sum(rows), n_qh // maps).bfloat16() if form == "gated" else None
    kd, vd, table, kv = pages(form, [s + r for s, r in zip(starts, rows)], bs)
    q = torch.randn(sum(rows), n_qh * d).bfloat16()
    want = []
    for i, (s, r) in enumerate(zip(starts, rows)):
        r0 = sum(rows[:i])
        want.append(dense(q[r0:r0 + r].double().reshape(r, n_qh, d), *kv[i], torch.arange(s, s + r), scale, mask, size, keep,
                          cap, db, sink, sig, hb))
    want = torch.cat(want)
    if gate is not None:
        want = want * torch.sigmoid(gate.double()).repeat_interleave(maps, 1)[:, :, None]
    if parts:
        monkeypatch.setattr(mx, "_prompt_parts", lambda *a: parts)
    else:
        rule, seen = mx._prompt_parts, []
        monkeypatch.setattr(mx, "_prompt_parts", lambda *a: seen.append(rule(*a)) or seen[-1])
    pos = torch.cat([torch.arange(s, s + r) for s, r in zip(starts, rows)]).cuda()
    seq = torch.tensor([i for i, r in enumerate(rows) for _ in range(r)], dtype=torch.int32).cuda()
    tiles = torch.tensor([t for i in range(3) for t in mx.tile_list(sum(rows[:i]), rows[i])], dtype=torch.int32).cuda()
    out_f32 = form.startswith("diff")
    got = mx.attention(q.cuda(), kd, vd, pos, seq, table, bs, n_qh, maps, group, d, dv, scale, mask, size, 1, out_f32, tiles,
                       sum(rows), softcap=cap, dist_bias=None if db is None else tuple(map(cuda, db)),
                       weights="sigmoid" if sig else "softmax", head_bias=cuda(hb), head_gate=cuda(gate), keep_first=keep,
                       sink=cuda(sink), fine_weights=form == "fine").cpu().double()
    if not parts:  # (the rule: 500 keys are cut only where a key takes longest)
        assert (seen[0][0] > 1) == (mask == "causal" or size > 500 or form in CUT_AT_500)
    err, top = float((got - want).abs().max()), float(want.abs().max())
    # (as in test_prompt_rows: the parts are joined in fp32)
    assert err < (3e-4 if out_f32 else 2.0 ** -8 * (top + (top if sig else 5.0))), err


@pytest.mark.gpu
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("parts", [1, 5])
@pytest.mark.parametrize("pre", [(4, 0), (3, 200), (8, 10000)])
@pytest.mark.parametrize("form", ["plain", "gated", "sigmoid", "both", "plain pair", "diff", "shared", "fine"])
def test_prompt_rows_in_parts_beside_decode_rows(monkeypatch, form, pre, parts, shift):
    """One join for a step's prompt rows and its decode rows (in one part: for the prompt rows alone); prompt rows that are cut,
    that are not, and both; a gate whose rows go on into the decode rows; queries (`shift`) whose address the kernels for whole
    tiles do not take, so that nothing is in parts."""
    n_qh, maps, group, d, dv = FORMS[form]
    torch.manual_seed(19)
    scale, bs = 0.7 * d ** -0.5, 64
    lengths, rows = [700, 40, 1300, 5, 650], [20, 40, 1, 1, 1]
    cap, db, sig, hb, sink = terms(form, n_qh)
    T, Tp = sum(rows), 60
    gate = torch.randn(T, n_qh // maps).bfloat16() if form == "gated" else None
    kd, vd, table, kv = pages(form, lengths, bs)
    q = torch.randn(T, n_qh * d).bfloat16()
    want, pos = [], []
    for i, (n, r) in enumerate(zip(lengths, rows)):
        r0, p = sum(rows[:i]), torch.arange(n - r, n)
        pos.append(p)
        want.append(dense(q[r0:r0 + r].double().reshape(r, n_qh, d), *kv[i], p, scale, "causal", 0, 0, cap, db, sink, sig, hb))
    want = torch.cat(want)
    if gate is not None:
        want = want * torch.sigmoid(gate.double()).repeat_interleave(maps, 1)[:, :, None]
    monkeypatch.setattr(mx, "_prompt_parts", lambda *a: pre)
    seq = torch.tensor([i for i, r in enumerate(rows) for _ in range(r)], dtype=torch.int32).cuda()
    tiles = torch.tensor(mx.tile_list(0, 20) + mx.tile_list(20, 40), dtype=torch.int32).cuda()
    out_f32 = form.startswith("diff")
    qd = torch.empty(T * n_qh * d + 8, dtype=torch.bfloat16, device="cuda")[4 * shift:4 * shift + T * n_qh * d].view(T, -1)
    qd.copy_(q)
    got = mx.attention(qd, kd, vd, torch.cat(pos).cuda(), seq, table, bs, n_qh, maps, group, d, dv, scale, "causal", 0, parts,
                       out_f32, tiles, Tp, softcap=cap, dist_bias=None if db is None else tuple(map(cuda, db)),
                       weights="sigmoid" if sig else "softmax", head_bias=cuda(hb), head_gate=cuda(gate), sink=cuda(sink),
                       fine_weights=form == "fine").cpu().double()
    err, top = float((got - want).abs().max()), float(want.abs().max())
    # (as in test_prompt_rows)
    assert err < (3e-4 if out_f32 else 2.0 ** -8 * (top + (top if sig else 5.0))), err


@pytest.mark.gpu
@pytest.mark.parametrize("pre,parts", [((1, 0), 1), ((2, 0), 2), ((8, 0), 16), ((4, 200), 5)])
@pytest.mark.parametrize("at", [3, 500, 1035])
@pytest.mark.parametrize("mask,size", [("causal", 0), ("window", 900)])
@pytest.mark.parametrize("form", ["plain", "fine", "both", "sigmoid", "diff", "shared"])
def test_rows_that_see_a_nan(monkeypatch, form, mask, size, at, pre, parts):
    """A key that holds a NaN, in the first, a middle and the last part of the contexts of prompt and decode rows, and query
    vectors that do: the rows and heads that see it are NaN however the keys are cut, with a sink and without, and no others."""
    n_qh, maps, group, d, dv = FORMS[form]
    torch.manual_seed(47)
    scale, bs = 0.7 * d ** -0.5, 64
    lengths, rows, Tp = [1047, 531, 1047, 650], [17, 40, 1, 1], 57
    cap, db, sig, hb, sink = terms(form, n_qh)
    kd, vd, table, kv = pages(form, lengths, bs)
    col = 200 if form == "shared" else 5  # (of a shared row: a column that is no value's)
    for i in (0, 2):
        kd[int(table[i, at // bs]) * bs + at % bs, col] = float("nan")
    q, q_nan = torch.randn(sum(rows), n_qh, d).bfloat16(), torch.zeros(sum(rows), n_qh, dtype=torch.bool)
    q_nan[20, 1] = q_nan[-1, 1] = True
    heads = torch.arange(n_qh) // maps
    hit = ((heads // group == 0) & (torch.arange(n_qh) % maps == 0)) | (form == "shared")  # heads of the key with the NaN
    want, pos = [], []
    for i, (n, r) in enumerate(zip(lengths, rows)):
        p = torch.arange(n - r, n)
        pos.append(p)
        w = dense(q[sum(rows[:i]):sum(rows[:i + 1])].double(), *kv[i], p, scale, mask, size, 0, cap, db, sink, sig, hb)
        if i in (0, 2):
            w[((p >= at) & (mx.first_visible(p, mask, size) <= at))[:, None] & hit] = float("nan")
        want.append(w)
    want = torch.cat(want)
    want[q_nan] = float("nan")
    q[q_nan] = float("nan")
    monkeypatch.setattr(mx, "_prompt_parts", lambda *a: pre)
    seq = torch.tensor([i for i, r in enumerate(rows) for _ in range(r)], dtype=torch.int32).cuda()
    tiles = torch.tensor(mx.tile_list(0, 17) + mx.tile_list(17, 40), dtype=torch.int32).cuda()
    got = mx.attention(q.view(sum(rows), -1).cuda(), kd, vd, torch.cat(pos).cuda(), seq, table, bs, n_qh, maps, group, d, dv, scale,
                       mask, size, parts, form == "diff", tiles, Tp, softcap=cap,
                       dist_bias=None if db is None else tuple(map(cuda, db)), weights="sigmoid" if sig else "softmax",
                       head_bias=cuda(hb), sink=cuda(sink), fine_weights=form == "fine").cpu().double()
    assert torch.equal(got.isnan(), want.isnan())
    err, top = float((got - want).nan_to_num().abs().max()), float(want.nan_to_num().abs().max())
    # (as in test_prompt_rows)
    assert err < (3e-4 if form == "diff" else 2.0 ** -8 * (top + (top if sig else 5.0))), err


@pytest.mark.gpu
@pytest.mark.parametrize("mask,size,keep", [("causal", 0, 0), ("window", 100, 40), ("window", 1, 0), ("chunk", 192, 0)])
@pytest.mark.parametrize("form", ["plain", "both", "sigmoid", "diff"])
def test_decode_rows_that_read_much(form, mask, size, keep):
    """Launches on both sides of the line beyond which cache lines are read nontemporally, with rows of both kinds in one: how
    a line is read changes no bit, so each row is what it is in a launch of eight."""
    n_qh, maps, group, d, dv = FORMS[form]
    torch.manual_seed(41)
    cap, db, sig, hb, sink = terms(form, n_qh)
    lengths, bs = [2000, 33, 96, 350, 1, 200], 32
    kd, vd, table, _ = pages(form, lengths, bs)
    for n, parts in ((600, 1), (64 if form == "diff" else 100, 2)):
        seq = torch.arange(n, dtype=torch.int32) % len(lengths)
        pos = torch.tensor(lengths)[seq.long()] - 1
        tiles = ((96 if mask == "window" else 160) << 20) // (2 * 32 * (kd.shape[1] + vd.shape[1]) * n)
        assert 1 <= tiles < 2000 // 32  # (rows of more tiles do not keep their lines)
        q, pos, seq = torch.randn(n, n_qh * d).bfloat16().cuda(), pos.cuda(), seq.cuda()

        def run(i, j):
            return mx.attention(q[i:j], kd, vd, pos[i:j], seq[i:j], table, bs, n_qh, maps, group, d, dv, 0.7 * d ** -0.5, mask,
                                size, parts, True, softcap=cap, dist_bias=None if db is None else tuple(map(cuda, db)),
                                weights="sigmoid" if sig else "softmax", head_bias=cuda(hb), keep_first=keep, sink=cuda(sink))
        got = run(0, n)
        for i in (0, 8, n // 2, n - 8):
            assert bool((got[i:i + 8] == run(i, i + 8)).all()), (n, i)


@pytest.mark.gpu
@pytest.mark.parametrize("mask,size,keep", [("causal", 0, 0), ("window", 1000, 40), ("chunk", 1500, 0)])
@pytest.mark.parametrize("form", ["plain", "capped", "sigmoid", "diff", "shared"])
def test_decode_rows_of_a_step_of_several_layers(form, mask, size, keep):
    """Rows on both sides of the line that holds where a step goes through several layers (48 MB), below one layer's."""
    n_qh, maps, group, d, dv = FORMS[form]
    torch.manual_seed(43)
    cap, db, sig, hb, sink = terms(form, n_qh)
    lengths, bs = [2000, 33, 96, 1350, 1, 700], 32
    kd, vd, table, _ = pages(form, lengths, bs)
    for n in (30 if form == "diff" else 60, 3):
        seq = torch.arange(n, dtype=torch.int32) % len(lengths)
        pos = torch.tensor(lengths)[seq.long()] - 1
        q, pos, seq = torch.randn(n, n_qh * d).bfloat16().cuda(), pos.cuda(), seq.cuda()

        def run(**kw):
            return mx.attention(q, kd, vd, pos, seq, table, bs, n_qh, maps, group, d, dv, 0.7 * d ** -0.5, mask, size, 2, True,
                                softcap=cap, weights="sigmoid" if sig else "softmax", head_bias=cuda(hb), keep_first=keep,
                                sink=cuda(sink), **kw)
        assert bool((run(layers=24) == run()).all()), n
