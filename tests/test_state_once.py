"""Decode steps whose states are read and written nontemporally (128 MB of them and more) against the same rows in steps of
half the sequences, which keep the lines: no bit of a result or a state depends on it, fresh sequences and padding rows
included."""
import pytest
import torch

from dynamo_exp_amd.ops import recurrent as rc


def step(rule, p, state, pos, slots, H, dk, dv):
    n = H * dk
    q, k, z, w, v = p[:, :n], p[:, n:2 * n], p[:, 2 * n:3 * n], p[:, 3 * n:4 * n], p[:, 4 * n:4 * n + H * dv]
    bias = torch.linspace(-1, 1, n, device="cuda")
    if rule == "retention":
        return rc.retention(q, k, v, torch.linspace(0.6, 0.99, H, device="cuda"), dk ** -0.5, state, pos, None, slots, H, dk, dv)
    if rule == "gla":
        return rc.gated_linear_attention(q, k, v, z, bias, 16.0, dk ** -0.5, state, pos, None, slots, H, dk, dv)
    if rule == "ssd":
        return rc.ssd(v, k[:, :dk], q[:, :dk], z[:, :H], bias[:H], torch.linspace(0.5, 8, H, device="cuda"), bias[:H], state, pos, None,
                      slots, H, 1, dk, dv)
    return rc.delta_rule(q, k, v, z, w, bias, bias, state, pos, None, slots, H, dk, dv)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rule,n,H,dk,dv", [("retention", 128, 8, 128, 256), ("gla", 64, 32, 128, 128), ("ssd", 32, 128, 128, 64),
                                            ("delta", 64, 32, 128, 128), ("delta", 129, 16, 128, 128)])
def test_states_that_are_not_kept(rule, n, H, dk, dv, dtype):
    torch.manual_seed(n)
    assert n * H * dk * dv * 4 >= 128 << 20
    p = torch.randn(n, 4 * H * dk + H * dv, device="cuda").to(dtype)
    state = torch.randn(n + 1, H, dv, dk, device="cuda")
    pos, slots = torch.arange(n, device="cuda") * 3, torch.randperm(n, device="cuda").to(torch.int32)
    slots[1] = -1
    both = state.clone()
    got = step(rule, p, state, pos, slots, H, dk, dv)
    h = n // 2
    want = torch.cat([step(rule, p[:h], both, pos[:h], slots[:h], H, dk, dv), step(rule, p[h:], both, pos[h:], slots[h:], H, dk, dv)])
    assert bool((got == want).all()) and bool((state == both).all()) and bool((got[1] == 0).all())
