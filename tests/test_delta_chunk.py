"""The delta rule's chunked form (csrc/mixers/delta_chunk.hip) against a float64 recurrence, and its error beside the
token-by-token kernel's on the same inputs (which float32 copies of them take)."""
from __future__ import annotations

import math

import pytest
import torch

from dynamo_exp_amd.ops import recurrent as rc

SCALE = rc.DELTA_DECAY_SCALE


def recurrence(r, k, v, a, w, ab, wb, S, H, dv, scale, eps=1e-6):
    """One sequence, float64: r, k, a, w [n, H 128], v [n, H dv], S [H, 128, dv] -> (o [n, H dv], S)."""
    n = r.shape[0]
    r, k, a, w = (x.double() for x in (r, k, a, w))
    wf = torch.exp(-scale * torch.sigmoid(w + wb.double())).view(n, H, 128)
    af = torch.sigmoid(a + ab.double()).view(n, H, 128)
    r, k, v = r.view(n, H, 128), k.view(n, H, 128), v.double().view(n, H, dv)
    u = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + eps)
    out = torch.empty(n, H, dv, dtype=torch.float64)
    for t in range(n):
        us = torch.einsum("hi,hij->hj", u[t], S)
        S = wf[t][:, :, None] * S - (af[t] * u[t])[:, :, None] * us[:, None] + k[t][:, :, None] * v[t][:, None]
        out[t] = torch.einsum("hi,hij->hj", r[t], S)
    return out.view(n, H * dv), S


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [[64], [15, 17, 1, 33], [64, 0, 50, 1, 1], [9, 8, 16, 31], [250], [9] * 18])
@pytest.mark.parametrize("kind", ["plain", "fast decay", "slow decay", "one key", "grown"])
@pytest.mark.parametrize("H,dv", [(2, 128), (3, 16), (1, 48)])
def test_delta_chunks(rows, kind, H, dv):
    """Sequences of ragged lengths (also empty ones, single tokens and a padding slot), from zero state and from a state
    of their own; decay logits at their ends, all keys equal, and a negative decay scale (a state that grows)."""
    torch.manual_seed(5)
    T, n_seq, n = sum(rows), len(rows), H * 128
    p = torch.randn(T, 3 * n + H * dv).bfloat16()
    wl = (torch.randn(T, n) * 0.5).bfloat16()
    scale = SCALE
    if kind == "fast decay":
        wl, scale = wl + 8, 4.0
    elif kind == "slow decay":
        wl = wl - 12
    elif kind == "one key":
        p[:, n:2 * n] = p[:1, n:2 * n]
    elif kind == "grown":
        scale = -0.25
    ab, wb = torch.randn(n) * 0.5, torch.randn(n)
    starts = [0 if i % 2 == 0 else 5 for i in range(n_seq)]
    slots = torch.randperm(n_seq + 2)[:n_seq].to(torch.int32)
    if n_seq > 2:
        slots[2] = -1
    state0 = torch.randn(n_seq + 2, H, dv, 128)
    firsts = [sum(rows[:i]) for i in range(n_seq + 1)]
    pos = torch.cat([torch.arange(s, s + r) for s, r in zip(starts, rows)])
    want, want_state = torch.zeros(T, H * dv, dtype=torch.float64), state0.double().clone()
    for i, (s, r) in enumerate(zip(starts, rows)):
        if slots[i] < 0 or r == 0:
            continue
        x = slice(firsts[i], firsts[i + 1])
        S = state0[slots[i]].double().transpose(1, 2) if s else torch.zeros(H, 128, dv, dtype=torch.float64)
        want[x], S = recurrence(p[x, :n], p[x, n:2 * n], p[x, 3 * n:], p[x, 2 * n:3 * n], wl[x], ab, wb, S, H, dv, scale)
        want_state[slots[i]] = S.transpose(1, 2)
    errs = []
    for dt in (torch.bfloat16, torch.float32):
        q, w, state = p.cuda().to(dt), wl.cuda().to(dt), state0.cuda()
        got = rc.delta_rule(q[:, :n], q[:, n:2 * n], q[:, 3 * n:], q[:, 2 * n:3 * n], w, ab.cuda(), wb.cuda(), state, pos.cuda(),
                            torch.tensor(firsts, dtype=torch.int32).cuda(), slots.cuda(), H, 128, dv, decay_scale=scale)
        rel = lambda x, y: float((x.cpu().double() - y).norm() / y.norm())
        errs.append((rel(got, want), rel(state, want_state)))
    # fp32 sums of 128 to 2000 products, each rounded to 2^-24 of it: sqrt(2000) 2^-24 = 3e-6 relative to the terms; and
    # no further off than the token-by-token form but for a few roundings (2^-24 each)
    for got, serial in zip(*errs):
        assert got < 3e-6 and got < 1.25 * serial + 1e-7, errs


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [[40, 64, 50, 33, 0, 1, 32, 70, 20], [64, 31, 33, 48, 5, 0, 40, 32, 1, 100, 17, 36, 63, 1, 34, 2],
                                  [35, 3] * 17])
@pytest.mark.parametrize("kind", ["plain", "slow decay", "one key", "grown"])
def test_delta_chunks_of_many_heads(rows, kind):
    """Workgroups of two column blocks, four of them to a head, sequences in order of their length (9 and 16) and as they
    come (34, whose short ones take four columns a thread)."""
    test_delta_chunks(rows, kind, 16, 128)


@pytest.mark.gpu
@pytest.mark.parametrize("dv,n_seq", [(32, 2), (16, 1), (32, 40)])  # (one column block per workgroup, and two)
@pytest.mark.parametrize("what", ["k", "v", "a", "w", "r", "state"])
@pytest.mark.parametrize("bad", [math.nan, math.inf])
def test_values_that_are_not_finite(dv, n_seq, what, bad):
    """They reach what they reach token by token: their own and later rows (of a value: its column), the state, no row in
    front of them, no other head or sequence."""
    torch.manual_seed(3)
    H, rows, at = 16, 70, 37
    n, T = H * 128, 70 * n_seq
    p, wl = torch.randn(T, 3 * n + H * dv).bfloat16(), (torch.randn(T, n) * 0.5).bfloat16()
    state0 = torch.randn(n_seq, H, dv, 128)
    first = {"r": 0, "k": n, "a": 2 * n, "v": 3 * n}
    if what == "w":
        wl[at, 130] = bad
    elif what == "state":
        state0[0, 1, 3, 5] = bad
    else:
        p[at, first[what] + (dv if what == "v" else 128) + 2] = bad  # head 1
    ab, wb = torch.randn(n) * 0.5, torch.randn(n)
    pos = torch.arange(5, 5 + rows).repeat(n_seq)
    starts = (torch.arange(n_seq + 1) * rows).to(torch.int32)
    res = []
    for dt in (torch.bfloat16, torch.float32):  # float32 copies run token by token
        q, w, state = p.cuda().to(dt), wl.cuda().to(dt), state0.cuda()
        out = rc.delta_rule(q[:, :n], q[:, n:2 * n], q[:, 3 * n:], q[:, 2 * n:3 * n], w, ab.cuda(), wb.cuda(), state, pos.cuda(),
                            starts.cuda(), torch.arange(n_seq, dtype=torch.int32).cuda(), H, 128, dv)
        res.append((out.cpu(), state.cpu()))
    for got, want in zip(*res):
        ok = torch.isfinite(want)
        assert torch.equal(torch.isfinite(got), ok)
        assert float((got[ok] - want[ok]).abs().max()) < 1e-5 * float(want[ok].abs().max())


@pytest.mark.gpu
def test_delta_chunk_rule():
    """Which rows take the chunks: bf16 prompt rows, keys of 128, whole blocks of values, a bounded decay, alignment."""
    ok = rc._m().delta_chunk_floats
    yes = (640, 3, 2, 128, 64, 0, SCALE, 16, 8)
    assert ok(*yes) == (40 + 3) * 2 * (4 * 2048 + 512 + 128)
    for i, x in ((0, 23), (3, 64), (4, 40), (5, 1), (6, 4.5), (6, math.nan), (7, 8), (8, 4)):
        assert ok(*yes[:i], x, *yes[i + 1:]) == 0


def run(p, wl, ab, wb, state, pos, starts, slots, H, dv, scale=SCALE):
    """The rows [r | k | a | v] on the GPU -> outputs, with `state` updated."""
    n = H * 128
    return rc.delta_rule(p[:, :n], p[:, n:2 * n], p[:, 3 * n:], p[:, 2 * n:3 * n], wl, ab, wb, state, pos,
                         None if starts is None else torch.tensor(starts, dtype=torch.int32).cuda(),
                         torch.tensor(slots, dtype=torch.int32).cuda(), H, 128, dv, decay_scale=scale)


@pytest.mark.gpu
@pytest.mark.parametrize("H,dv,rows", [
    (2, 128, [1, 31, 32, 200, 5, 1]), (3, 16, [70, 1, 33, 30]), (1, 48, [1, 1, 100, 33, 32, 31, 1, 80]),
    (16, 128, [1, 32, 90, 2, 65, 0, 1, 31, 129]),  # two column blocks a workgroup
    (8, 128, [200] + [1] * 150), (2, 32, [1] * 90 + [64]),  # more sequences than eight rows each would allow
    (32, 128, [1] * 70 + [80])])  # (as a decode step of their own: tiles of 2 columns a thread)
def test_a_sequence_does_not_depend_on_its_step(H, dv, rows):
    """Every sequence's rows and state are bit for bit what they are in a step of its own."""
    torch.manual_seed(23)
    T, n, B = sum(rows), H * 128, len(rows)
    p, wl = torch.randn(T, 3 * n + H * dv, device="cuda").bfloat16(), (torch.randn(T, n, device="cuda") * 0.5).bfloat16()
    ab, wb = torch.randn(n, device="cuda") * 0.5, torch.randn(n, device="cuda")
    firsts = [sum(rows[:i]) for i in range(B + 1)]
    pos = torch.cat([torch.arange(7 * (i % 2), 7 * (i % 2) + r) for i, r in enumerate(rows)]).cuda()
    state0 = torch.randn(B, H, dv, 128, device="cuda")
    together = state0.clone()
    out = run(p, wl, ab, wb, together, pos, firsts, list(range(B)), H, dv)
    for i, r in enumerate(rows):
        if r == 0:
            assert torch.equal(together[i], state0[i])
            continue
        if i and r == 1 and rows[i - 1] == 1 and i % 16:  # (a few of many equal ones)
            continue
        x, alone = slice(firsts[i], firsts[i + 1]), state0.clone()
        for starts in ([0, r],) if r > 1 else ([0, 1], None):  # (a decode step names no rows)
            alone.copy_(state0)
            got = run(p[x], wl[x], ab, wb, alone, pos[x], starts, [i], H, dv)
            assert torch.equal(got, out[x]) and torch.equal(alone[i], together[i]), (i, r)


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [SCALE, 1.0, 4.0, -1.0])
@pytest.mark.parametrize("what,size", [("k", 1e12), ("k", 1e18), ("k", 1e35), ("r", 1e-12), ("r", 1e-25), ("r", 1e18), ("v", 1e30),
                                       ("v", 1e-30)])
def test_rows_of_any_size(scale, what, size):
    """One row far larger or smaller than the others, at every place of a chunk, with decays at their fastest: rows are
    finite where they are token by token, and as near to float64, each relative to its own size."""
    torch.manual_seed(29)
    H, dv, n, B = 1, 32, 128, 16
    rows = 50
    T = rows * B
    p, wl = torch.randn(T, 3 * n + dv).bfloat16(), (torch.randn(T, n) * 0.5 + 8).bfloat16()
    first, wide = {"r": (0, n), "k": (n, n), "v": (3 * n, dv)}[what]
    for i in range(B):
        p[i * rows + 16 + i, first:first + wide] *= size
    ab, wb = torch.randn(n) * 0.5, torch.randn(n)
    state0, pos = torch.randn(B, H, dv, 128), torch.arange(5, 5 + rows).repeat(B)
    want = torch.cat([recurrence(p[x, :n], p[x, n:2 * n], p[x, 3 * n:], p[x, 2 * n:3 * n], wl[x], ab, wb,
                                 state0[i].double().transpose(1, 2), H, dv, scale)[0]
                      for i, x in enumerate(slice(j, j + rows) for j in range(0, T, rows))])
    res = []
    for dt in (torch.bfloat16, torch.float32):  # float32 copies run token by token
        state = state0.cuda()
        out = run(p.cuda().to(dt), wl.cuda().to(dt), ab.cuda(), wb.cuda(), state, pos.cuda(), list(range(0, T + 1, rows)),
                  list(range(B)), H, dv, scale)
        res.append((out.cpu().double(), torch.isfinite(state).cpu()))
    (got, got_ok), (serial, serial_ok) = res
    ok = torch.isfinite(serial).all(1)
    assert torch.equal(torch.isfinite(got), torch.isfinite(serial)) and torch.equal(got_ok, serial_ok) and bool(ok.any())
    # (where a large row is removed again what is left has lost the same bits in both: measured 0.2 to 1.6 of each other)
    err, err_serial = (float(((x - want)[ok].norm(dim=1) / want[ok].norm(dim=1)).max()) for x in (got, serial))
    assert err < 4 * err_serial + 1e-5, (err, err_serial)


@pytest.mark.gpu
@pytest.mark.parametrize("H,dv,rows", [(2, 128, [33, 1, 70, 20]), (3, 16, [250]), (1, 48, [47, 32]),
                                       (16, 32, [1] * 40 + [33, 70, 17] + [2] * 21)])  # the last: two column blocks a workgroup
def test_value_rows_anywhere(H, dv, rows):
    """Values in rows of an odd stride behind an odd offset, with NaN around every row and behind the last one (a chunk
    that the sequence does not fill reads zeros there): bit for bit what packed rows give."""
    torch.manual_seed(31)
    T, n = sum(rows), H * 128
    p, wl = torch.randn(T, 3 * n + H * dv, device="cuda").bfloat16(), (torch.randn(T, n, device="cuda") * 0.5).bfloat16()
    wide = torch.full((T + 16, H * dv + 5), math.nan, dtype=torch.bfloat16, device="cuda")
    wide[:T, 1:1 + H * dv] = p[:, 3 * n:]
    ab, wb = torch.randn(n, device="cuda") * 0.5, torch.randn(n, device="cuda")
    starts = torch.tensor([sum(rows[:i]) for i in range(len(rows) + 1)], dtype=torch.int32).cuda()
    pos, slots = torch.cat([torch.arange(r) for r in rows]).cuda(), torch.arange(len(rows), dtype=torch.int32).cuda()
    res = []
    for v in (p[:, 3 * n:].contiguous(), wide[:T, 1:1 + H * dv]):
        state = torch.zeros(len(rows), H, dv, 128, device="cuda")
        res.append((rc.delta_rule(p[:, :n], p[:, n:2 * n], v, p[:, 2 * n:3 * n], wl, ab, wb, state, pos, starts, slots, H, 128,
                                  dv), state))
    assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1]) and bool(torch.isfinite(res[0][0]).all())


@pytest.mark.gpu
@pytest.mark.parametrize("z", [0.0, 20.0, 87.0, 88.5, 100.0, 3e38, math.inf])
def test_gates_at_their_ends(z):
    """Removal and decay gates of logits +-z, also far enough that exp() of them is 0 or infinite; and no biases at all, bit
    for bit what biases of zero give."""
    torch.manual_seed(37)
    H, dv, T, n = 2, 32, 50, 256
    p, wl = torch.randn(T, 3 * n + H * dv).bfloat16(), torch.full((T, n), z).bfloat16()
    wl[::2] *= -1
    p[:, 2 * n:3 * n] = wl.flip(1)
    p[::3, 2 * n:3 * n] *= -1
    zero, state0 = torch.zeros(n), torch.randn(1, H, dv, 128)
    want, want_state = recurrence(p[:, :n], p[:, n:2 * n], p[:, 3 * n:], p[:, 2 * n:3 * n], wl, zero, zero,
                                  state0[0].double().transpose(1, 2), H, dv, SCALE)
    res = []
    for bias in (zero.cuda(), None):
        state = state0.cuda()
        out = run(p.cuda(), wl.cuda(), bias, bias, state, torch.arange(5, 5 + T).cuda(), [0, T], [0], H, dv)
        res.append((out.cpu(), state.cpu()))
    assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])
    rel = lambda x, y: float((x.double() - y).norm() / y.norm())
    # (fp32 sums of 128 to 2000 products, each rounded to 2^-24 of it: sqrt(2000) 2^-24 relative to the terms)
    assert rel(res[0][0], want) < 3e-6 and rel(res[0][1][0], want_state.transpose(1, 2)) < 3e-6


@pytest.mark.gpu
@pytest.mark.parametrize("n,H,dv", [(1, 1, 1), (3, 2, 20), (5, 3, 128), (2, 1, 200), (33, 8, 128), (70, 16, 48), (130, 32, 128)])
@pytest.mark.parametrize("dtype,bias", [(torch.bfloat16, True), (torch.bfloat16, False), (torch.float32, True)])
def test_delta_step(n, H, dv, dtype, bias):
    """A decode step of keys of 128 channels, one, two and four columns a thread: sequences in front of position 0 and behind,
    a padding slot, rows at odd strides.  fp32 throughout: a sum of 128 products of size one is rounded at its partial sums,
    of up to sqrt(128) and at most 2^-24 each, 16 in a row in a lane: 2^-21 of sqrt(128) an element (an element itself may be
    smaller, where products cancel)."""
    torch.manual_seed(n)
    D = H * 128
    p = torch.randn(n, 4 * D + H * dv + 3).to(dtype).cuda()
    r, k, a, w = (p[:, i * D:(i + 1) * D] for i in range(4))
    v = p[:, 4 * D + 1:4 * D + 1 + H * dv]
    ab, wb = (torch.randn(D) * 0.5, torch.randn(D)) if bias else (None, None)
    slots = torch.randperm(n + 2)[:n].to(torch.int32)
    if n > 2:
        slots[2] = -1
    pos = torch.arange(n) % 3
    state0 = torch.randn(n + 2, H, dv, 128)
    state = state0.cuda()
    dev = lambda t: None if t is None else t.cuda()  # noqa: E731
    o = rc.delta_rule(r, k, v, a, w, dev(ab), dev(wb), state, pos.cuda(), None, slots.cuda(), H, 128, dv)
    want, want_state = torch.zeros(n, H * dv, dtype=torch.float64), state0.double().clone()
    zero = torch.zeros(D)
    for i in range(n):
        s = int(slots[i])
        if s < 0:
            continue
        S = want_state[s].transpose(1, 2) * (int(pos[i]) > 0)
        x = [t[i:i + 1].cpu() for t in (r, k, v, a, w)]
        out, S = recurrence(*x, zero if ab is None else ab, zero if wb is None else wb, S, H, dv, SCALE)
        want[i], want_state[s] = out[0], S.transpose(1, 2)
    for got, ref in ((o, want), (state, want_state)):
        assert float((got.double().cpu() - ref).norm()) < 2.0 ** -21 * max(float(ref.norm()), (128 * ref.numel()) ** 0.5)
    if n > 2:
        assert bool((o[2] == 0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("n,H", [(3, 2), (40, 16), (70, 32)])
def test_delta_step_beside_prompt(n, H):
    """A decode row's result and state are the same bits in a step of its own and beside a prompt."""
    torch.manual_seed(n)
    D, T = H * 128, n + 64
    p = torch.randn(T, 5 * D).bfloat16().cuda()
    ab, wb, state = torch.randn(D).cuda(), torch.randn(D).cuda(), torch.randn(n + 1, H, 128, 128).cuda()
    both, pos = state.clone(), torch.cat([torch.arange(n) + 1, torch.arange(64)]).cuda()
    rows = torch.tensor(list(range(n + 1)) + [T], dtype=torch.int32).cuda()
    slots = torch.arange(n + 1, dtype=torch.int32).cuda()
    secs = [p[:, i * D:(i + 1) * D] for i in range(5)]
    a = rc.delta_rule(*(x[:n] for x in secs), ab, wb, state, pos[:n], None, slots[:n], H, 128, 128)
    b = rc.delta_rule(*secs, ab, wb, both, pos, rows, slots, H, 128, 128)
    assert torch.equal(a, b[:n]) and torch.equal(state[:n], both[:n])


def test_rows_that_32_bit_offsets_do_not_reach():
    """The chunked form asks for no workspace, and its launch refuses, where 16 rows of v or of the result span 4 GiB."""
    m = rc._m()
    for H, dv, vs, ok in ((2, 128, 256, True), (2, 128, 1 << 27, True), (2, 128, (1 << 27) + 8, False), (2, 128, 1 << 31, False),
                          (1 << 13, 1 << 13, 1 << 26, True), (1 << 14, 1 << 13, 1 << 27, False)):
        assert (m.delta_chunk_floats(64, 1, H, 128, dv, 0, SCALE, 0, 256, vs) > 0) == ok, (H, dv, vs)
        if not ok:
            with pytest.raises(RuntimeError, match="code 2"):
                m.delta_chunk(16, 16, 1, 16, 16, 256, 16, 256, 16, vs, 16, 256, 16, 256, 0, 0, SCALE, 1e-6, 16, 16, 16, 1, 64, H,
                              dv, 0)
