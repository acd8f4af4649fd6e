"""The chunked linear recurrences (csrc/mixers/chunk_scan.hip) against float64 recurrences, at the edges of their chunks and
with sequences taken by length."""
from __future__ import annotations

import pytest
import torch

from dynamo_exp_amd.ops import recurrent as rc


def recurrence(q, k, v, decay, step, S):
    """One sequence, float64: q, k [n, H, dk], v [n, H, dv], decay [n, H, 1 or dk], step [n, H], S [H, dk, dv]."""
    out = torch.empty(v.shape, dtype=torch.float64)
    for t in range(q.shape[0]):
        S = decay[t][..., None] * S + k[t][:, :, None] * (step[t][:, None] * v[t])[:, None]
        out[t] = torch.einsum("hi,hij->hj", q[t], S)
    return out, S


def rel(a, b):
    return float((a.double().cpu() - b).norm() / b.norm())


ROWS = [[64], [63, 65], [8, 7, 129, 1, 128], [200, 9, 0, 66, 31, 8], [9] * 70]


def scan(kind, rows, H, dk, dv):
    torch.manual_seed(len(rows) + H)
    T, n_seq, G = sum(rows), len(rows), 1 if kind == "ssd" else H
    p = torch.randn(T, 2 * G * dk + H * dv + 8).bfloat16()
    q, k, v = (x.cuda() for x in p.split([G * dk, G * dk, H * dv, 8], 1)[:3])
    g = (torch.randn(T, H * dk if kind == "gla" else H) - 1.0).bfloat16()
    bias, rate, skip = torch.randn(H * dk if kind == "gla" else H), torch.rand(H) * 3 + 0.1, torch.randn(H)
    fixed = 1.0 - 2.0 ** (-3.0 - torch.arange(H) % 6)
    first, starts = [0] + torch.tensor(rows).cumsum(0).tolist(), [0 if i % 2 else 5 for i in range(n_seq)]
    slots = torch.randperm(n_seq + 1)[:n_seq].to(torch.int32)
    if n_seq > 4:
        slots[4] = -1  # padding rows
    state0 = torch.randn(n_seq + 1, H, dv, dk)
    pos = torch.cat([torch.arange(s, s + r) for s, r in zip(starts, rows)])
    state, at = state0.cuda(), (pos.cuda(), torch.tensor(first, dtype=torch.int32).cuda(), slots.cuda())
    if kind == "retention":
        o = rc.retention(q, k, v, fixed.cuda(), dk ** -0.5, state, *at, H, dk, dv)
    elif kind == "ssd":
        o = rc.ssd(v, k, q, g.cuda(), bias.cuda(), rate.cuda(), skip.cuda(), state, *at, H, 1, dk, dv)
    else:
        o = rc.gated_linear_attention(q, k, v, g.cuda(), bias.cuda(), 16.0, dk ** -0.5, state, *at, H, dk, dv)
    Q, K = (x.cpu().double().view(T, G, dk).expand(T, H, dk) for x in (q, k))
    V, z, one = v.cpu().double().view(T, H, dv), g.double() + bias.double(), torch.ones(T, H, dtype=torch.float64)
    Q, K = (Q * dk ** -0.5, K) if kind == "gla" else (Q, K * dk ** -0.5) if kind == "retention" else (Q, K)
    step = torch.nn.functional.softplus(z) if kind == "ssd" else one
    decay = {"retention": lambda: fixed.double() * one, "ssd": lambda: torch.exp(-rate.double() * step),
             "gla": lambda: torch.sigmoid(z).pow(1 / 16)}[kind]().view(T, H, -1)
    want, want_state = torch.zeros(T, H, dv, dtype=torch.float64), state0.double().clone()
    for i in range(n_seq):
        a, b, s = first[i], first[i + 1], int(slots[i])
        if s < 0 or a == b:
            continue
        S = want_state[s].transpose(1, 2) * (starts[i] > 0)
        want[a:b], S = recurrence(Q[a:b], K[a:b], V[a:b], decay[a:b], step[a:b], S)
        want_state[s] = S.transpose(1, 2)
        if kind == "ssd":
            want[a:b] += skip.double()[:, None] * V[a:b]
    return rel(o.view(T, H, dv), want), rel(state, want_state), o.view(T, H, dv), want


@pytest.mark.gpu
@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("kind,H,dk,dv", [("retention", 32, 128, 128), ("ssd", 64, 128, 64), ("gla", 32, 128, 128),
                                          ("retention", 3, 64, 64), ("ssd", 4, 32, 128), ("gla", 5, 32, 64)])
def test_chunks(rows, kind, H, dk, dv):
    """Whatever carries a decay or the state has 16 bits of mantissa (a sum of two bf16), every sum is fp32: 2^-16 of the
    results' norm."""
    eo, es, o, want = scan(kind, rows, H, dk, dv)
    assert eo < 2.0 ** -16 and es < 2.0 ** -16, (eo, es)
    assert bool((o.cpu()[want.abs().sum((1, 2)) == 0] == 0).all())  # padding rows


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [[130, 9, 0, 300, 130, 7, 64, 200], [300, 8, 200, 200, 129, 31, 7, 1, 0, 64],
                                  [16 + i % 7 * 9 for i in range(36)] + [5, 0, 300], [10] * 70], ids=len)
@pytest.mark.parametrize("kind,H,dk,dv", [("retention", 32, 128, 128), ("ssd", 64, 128, 64), ("gla", 32, 128, 128),
                                          ("retention", 24, 32, 128)])
def test_sequences_by_length(rows, kind, H, dk, dv):
    """More workgroups of long sequences than the chip takes at once, so that they go out by length: equal lengths, padding
    slots, runs too short for a chunk and empty ones among them, and more sequences than are put in order."""
    if (kind, H) == ("retention", 24):
        rows = rows * 2 if len(rows) < 20 else rows + [9] * 20
    assert H * (dv // 64) * min(len(rows), sum(rows) // 128) > 256  # launch_chunk_scan's rule
    eo, es, o, want = scan(kind, rows, H, dk, dv)
    assert eo < 2.0 ** -16 and es < 2.0 ** -16, (eo, es)  # (test_chunks)
    assert bool((o.cpu()[want.abs().sum((1, 2)) == 0] == 0).all())


MANY = [n for i in range(26) for n in (33 + i % 7 * 9, (1, 0, 3, 7)[i % 4])]


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [MANY, MANY + [1, 2] * 6, MANY + [1, 2] * 6 + [200]], ids=len)
@pytest.mark.parametrize("kind,H,dk,dv", [("retention", 32, 128, 128), ("ssd", 64, 128, 64), ("gla", 32, 128, 128),
                                          ("retention", 24, 32, 128)])
def test_short_sequences_behind_many(rows, kind, H, dk, dv):
    """Short sequences in the launch of more long ones than are put in order, of 64 in all and of more than a wave compares:
    each goes through once (one left out, or taken twice, is a hundredth of the results)."""
    assert H * (dv // 64) * min(len(rows), sum(rows) // 128) > 256 and H * (dv // 64) * len(rows) <= 8192  # launch_chunk_scan's rules
    eo, es, o, want = scan(kind, rows, H, dk, dv)
    assert eo < 2.0 ** -16 and es < 2.0 ** -16, (eo, es)  # (test_chunks)
    assert bool((o.cpu()[want.abs().sum((1, 2)) == 0] == 0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("stride", [0, 8, 64])
@pytest.mark.parametrize("kind", ["retention", "ssd", "gla"])
def test_rows_that_overlap(kind, stride):
    """Rows of one buffer that overlap or are all the same one (also the step's logits), the second sequence's end in the
    middle of a chunk and an infinite key in its last row: the bits of the same rows laid out one behind the other."""
    torch.manual_seed(3)
    H, dk, dv, rows = 3, 128, 64, [64, 150]
    T = sum(rows)

    def row_view(width, step):
        return torch.randn(T * max(step, 1) + width).bfloat16().cuda().as_strided((T, width), (step, 1))

    q, k, v, g = row_view(H * dk, stride), row_view(H * dk, stride), row_view(H * dv, stride), row_view(H * dk, stride)
    dt = row_view(H, stride // 8)
    if stride:
        k[-1, -1] = float("inf")
    pos, first = torch.arange(T).cuda() + 1, torch.tensor([0, rows[0], T], dtype=torch.int32).cuda()
    slots, state0 = torch.tensor([1, 0], dtype=torch.int32).cuda(), torch.randn(2, H, dv, dk).cuda()
    bias, rate, fixed = torch.randn(H * dk).cuda(), torch.rand(H).cuda() + 0.1, 1.0 - torch.rand(H).cuda() / 8

    def run(q, k, v, g, dt):
        state = state0.clone()
        if kind == "retention":
            o = rc.retention(q, k, v, fixed, 0.1, state, pos, first, slots, H, dk, dv)
        elif kind == "ssd":
            o = rc.ssd(v, k, q, dt, bias[:H], rate, None, state, pos, first, slots, H, H, dk, dv)
        else:
            o = rc.gated_linear_attention(q, k, v, g, bias, 16.0, 0.1, state, pos, first, slots, H, dk, dv)
        return o, state

    for got, want in zip(run(q, k, v, g, dt), run(*(x.contiguous() for x in (q, k, v, g, dt)))):
        torch.testing.assert_close(got, want, rtol=0, atol=0, equal_nan=True)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [[200, 1, 7, 3, 1, 70, 1], [9, 1], [1] * 20 + [130, 140], [1, 2, 300, 0, 5, 129, 7] * 4])
@pytest.mark.parametrize("kind,H,dk,dv", [("retention", 32, 128, 128), ("ssd", 64, 128, 64), ("gla", 32, 128, 128),
                                          ("retention", 2, 64, 64), ("ssd", 4, 32, 128), ("gla", 5, 64, 64), ("gla", 3, 32, 64)])
def test_short_sequences_beside_long_ones(rows, kind, H, dk, dv):
    """Sequences too short for a chunk, in the launch of the long ones: the same bits as in a step of their own."""
    torch.manual_seed(len(rows) + H)
    T, n = sum(rows), len(rows)
    q, k, v = (torch.randn(T, H * w).bfloat16().cuda() for w in (dk, dk, dv))
    g = (torch.randn(T, H * dk if kind == "gla" else H) - 1.0).bfloat16().cuda()
    bias, rate, skip = torch.randn(g.shape[1]).cuda(), torch.rand(H).cuda() * 3 + 0.1, torch.randn(H).cuda()
    fixed = (1.0 - 2.0 ** (-3.0 - torch.arange(H) % 6)).cuda()
    state0, slots = torch.randn(n, H, dv, dk).cuda(), torch.randperm(n).to(torch.int32)
    pos = torch.cat([torch.arange(i % 3, i % 3 + r) for i, r in enumerate(rows)])

    def step(which):
        first = [0]
        for i in which:
            first.append(first[-1] + rows[i])
        at = torch.cat([torch.arange(sum(rows[:i]), sum(rows[:i + 1])) for i in which])
        S = state0.clone()
        here = (pos[at].cuda(), torch.tensor(first, dtype=torch.int32).cuda(), slots[list(which)].cuda(), H)
        at = at.cuda()
        if kind == "retention":
            o = rc.retention(q[at], k[at], v[at], fixed, dk ** -0.5, S, *here, dk, dv)
        elif kind == "ssd":
            o = rc.ssd(v[at], k[at], q[at], g[at], bias, rate, skip, S, *here, H, dk, dv)
        else:
            o = rc.gated_linear_attention(q[at], k[at], v[at], g[at], bias, 16.0, dk ** -0.5, S, *here, dk, dv)
        return [o[first[j]:first[j + 1]] for j in range(len(which))], S

    both, S = step(range(n))
    for i, r in enumerate(rows):
        if 0 < r < 8:
            alone, A = step([i])
            assert torch.equal(both[i], alone[0]) and torch.equal(S[slots[i].item()], A[slots[i].item()]), (i, r)


@pytest.mark.gpu
@pytest.mark.parametrize("stride", [1 << 24, (1 << 24) + 8])
@pytest.mark.parametrize("dk", [32, 128])
def test_rows_far_apart(dk, stride):
    """Rows on both sides of what 32-bit offsets inside a chunk reach: the same bits as rows that lie together."""
    torch.manual_seed(dk)
    H, dv, rows = 2, 64, [41, 9]
    T, n = sum(rows), 2 * dk
    x = torch.randn(T, 3 * n + H * dv, device="cuda").bfloat16()
    far = torch.empty((T - 1) * stride + x.shape[1], dtype=x.dtype, device="cuda").as_strided(x.shape, (stride, 1))
    far.copy_(x)
    first, pos = torch.tensor([0, *rows]).cumsum(0).to(torch.int32).cuda(), torch.cat([torch.arange(r) for r in rows]).cuda()
    slots, bias = torch.tensor([1, 0], dtype=torch.int32).cuda(), torch.randn(n, device="cuda")
    got = []
    for p in (x, far):
        state = torch.zeros(2, H, dv, dk, device="cuda")
        got.append((rc.gated_linear_attention(p[:, :n], p[:, n:2 * n], p[:, 3 * n:], p[:, 2 * n:3 * n], bias, 16.0, dk ** -0.5, state,
                                              pos, first, slots, H, dk, dv), state))
    assert float(got[0][0].abs().sum()) > 0
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
