"""Decode steps whose states are read and written nontemporally (128 MB of them and more, or 44 MB where the step goes through
several layers) against steps that keep the lines: no bit of a result or a state depends on it, fresh sequences and padding
rows included."""
import pytest
import torch

from dynamo_exp_amd.engine.engine import EngineConfig, LLMEngine
from dynamo_exp_amd.models.config import get_config
from dynamo_exp_amd.models.registry import build_model
from dynamo_exp_amd.ops import mixers as mx
from dynamo_exp_amd.ops import recurrent as rc


def step(rule, p, state, pos, slots, H, dk, dv, **kw):
    n = H * dk
    q, k, z, w, v = p[:, :n], p[:, n:2 * n], p[:, 2 * n:3 * n], p[:, 3 * n:4 * n], p[:, 4 * n:4 * n + H * dv]
    bias = torch.linspace(-1, 1, n, device="cuda")
    if rule == "retention":
        return rc.retention(q, k, v, torch.linspace(0.6, 0.99, H, device="cuda"), dk ** -0.5, state, pos, None, slots, H, dk, dv,
                            **kw)
    if rule == "gla":
        return rc.gated_linear_attention(q, k, v, z, bias, 16.0, dk ** -0.5, state, pos, None, slots, H, dk, dv, **kw)
    if rule == "ssd":
        return rc.ssd(v, k[:, :dk], q[:, :dk], z[:, :H], bias[:H], torch.linspace(0.5, 8, H, device="cuda"), bias[:H], state, pos, None,
                      slots, H, 1, dk, dv, **kw)
    return rc.delta_rule(q, k, v, z, w, bias, bias, state, pos, None, slots, H, dk, dv, **kw)


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


@pytest.mark.gpu
@pytest.mark.parametrize("rule,n,H,dk,dv", [("retention", 44, 8, 128, 256), ("gla", 22, 32, 128, 128), ("ssd", 11, 128, 128, 64),
                                            ("delta", 22, 32, 128, 128), ("delta", 3, 32, 128, 128), ("retention", 5, 3, 64, 48)])
def test_layers_of_a_step(rule, n, H, dk, dv):
    """At the line of 44 MB, one sequence below it and far below."""
    torch.manual_seed(n)
    for n in (n, n - 1):
        p = torch.randn(n, 4 * H * dk + H * dv, device="cuda").bfloat16()
        state = torch.randn(n + 1, H, dv, dk, device="cuda")
        pos, slots = torch.arange(n, device="cuda") * 3, torch.randperm(n, device="cuda").to(torch.int32)
        one, many = state.clone(), state.clone()
        want = step(rule, p, one, pos, slots, H, dk, dv)
        assert bool((step(rule, p, many, pos, slots, H, dk, dv, layers=24) == want).all()) and bool((many == one).all())


@pytest.mark.parametrize("preset", ["bekulix-tiny", "bolinex-tiny", "nefivik-tiny", "sobivik-tiny", "povurax-tiny", "kilatar-tiny"])
def test_models_say_how_many_layers_a_step_has(monkeypatch, preset):
    cfg, seen = get_config(preset), []
    model = build_model(cfg, torch.device("cpu"), dtype="float32")
    model.load_state(model.random_state(0))

    def watch(mod, name, shared):
        real = getattr(mod, name)

        def call(*a, **kw):
            if not shared or a[1] is not a[2]:  # (a row that is key and value: one way to read it)
                seen.append(kw.get("layers", 1))
            return real(*a, **kw)
        monkeypatch.setattr(mod, name, call)
    for name in ("delta_rule", "retention", "ssd", "gated_linear_attention"):
        watch(rc, name, False)
    watch(mx, "attention", True)
    eng = LLMEngine(EngineConfig(model="t", device="cpu", dtype="float32", block_size=8, num_gpu_blocks=48, max_model_len=384,
                                 max_num_seqs=4, enable_prefix_caching=False, use_cuda_graph=False, async_schedule=False),
                    model_cfg=cfg, model=model)
    eng.forced_step([("a", [5, 6, 7], [0, 1, 2])], ["a"])
    assert seen and set(seen) == {len(model.layers)}
