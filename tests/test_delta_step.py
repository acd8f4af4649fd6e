"""The delta rule's decode step (recurrent.hip, delta_step_kernel) and gated linear attention token by token at column counts
that do not fill a workgroup, with and without biases, beside fresh sequences whose slot holds anything and padding rows."""
import pytest
import torch

from dynamo_exp_amd.ops import recurrent as rc

D = 128


def rows(n, H, dv, dtype):
    g = torch.Generator(device="cuda").manual_seed(100 * n + dv)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x = [rn(n, H * D).to(dtype) for _ in range(4)] + [rn(n, H * dv).to(dtype)]
    state = rn(n + 1, H, dv, D)
    pos, slots = torch.arange(n, device="cuda") * 5, torch.randperm(n + 1, generator=g, device="cuda")[:n].to(torch.int32)
    state[slots[0].long()] = float("nan")  # at position 0: not looked at
    if n > 2:
        slots[2] = -1
    return x, state, pos, slots, (rn(H * D), rn(H * D))


def before(state, pos, slots):
    S = state[slots.clamp_min(0).long()].double()
    S[pos == 0] = 0
    return S  # [n, H, dv, D]


def check(got, state, was, slots, o, S):
    live = slots >= 0
    # fp32 sums of 128 products of unit size, a few in a row: 128 x 2^-24 of the largest partial sums, some 30
    assert bool((got[~live] == 0).all())
    assert bool(((got[live].double() - o[live]).abs() <= 3e-4).all())
    at = slots[live].long()
    assert bool(((state[at].double() - S[live]).abs() <= 3e-5).all())
    rest = torch.ones(len(state), dtype=torch.bool)
    rest[at.cpu()] = False
    assert torch.equal(state[rest].nan_to_num(), was[rest].nan_to_num())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("biases", [True, False])
@pytest.mark.parametrize("n,H,dv", [(1, 1, 1), (3, 2, 3), (5, 3, 40), (4, 2, 200), (40, 16, 33), (70, 16, 33), (130, 16, 72)])
def test_delta_step(n, H, dv, biases, dtype):
    (r, k, a, w, v), state, pos, slots, (ab, wb) = rows(n, H, dv, dtype)
    ab, wb = (ab, wb) if biases else (None, None)
    was, S = state.clone(), before(state, pos, slots)
    got = rc.delta_rule(r, k, v, a, w, ab, wb, state, pos, None, slots, H, D, dv)
    f = lambda t, b=None: (t.double() + (0 if b is None else b.double())).view(n, H, 1, -1)
    decay = torch.exp(-rc.DELTA_DECAY_SCALE * torch.sigmoid(f(w, wb)))
    u = f(k) / torch.sqrt((f(k) ** 2).sum(-1, keepdim=True) + 1e-6)
    S = S * decay - torch.sigmoid(f(a, ab)) * u * (S * u).sum(-1, keepdim=True) + f(k) * v.double().view(n, H, dv, 1)
    check(got, state, was, slots, (S * f(r)).sum(-1).reshape(n, -1), S)


@pytest.mark.gpu
@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("n,H,dv", [(1, 1, 32), (5, 3, 64), (40, 4, 128)])
def test_gated_linear_step(n, H, dv, bias):
    (q, k, z, _, v), state, pos, slots, (zb, _) = rows(n, H, dv, torch.bfloat16)
    zb = zb if bias else None
    was, S = state.clone(), before(state, pos, slots)
    got = rc.gated_linear_attention(q, k, v, z, zb, 16.0, D ** -0.5, state, pos, None, slots, H, D, dv)
    f = lambda t, b=None: (t.double() + (0 if b is None else b.double())).view(n, H, 1, -1)
    S = S * torch.sigmoid(f(z, zb)) ** (1 / 16) + f(k) * v.double().view(n, H, dv, 1)
    check(got, state, was, slots, (S * f(q)).sum(-1).reshape(n, -1) * D ** -0.5, S)
