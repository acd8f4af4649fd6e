"""The work that serving does on one GPU, as cases that can be timed: the attention, recurrent and expert parts of an
engine step for every kind of layer that the models list, and whole prompt steps of the Llama path.

A case is one pass of one kind of layer over the rows of an engine step (prompt chunks of ragged lengths, decode rows
of ragged contexts, or both), through dynamo_exp_amd's ops as the model classes call them, at the layer sizes of
`llama3-8b` / the `*-8b-shapes` presets (32 query heads, 8 key/value heads, width 4096) and of the bench's
`1b-shapes` (16, 4, 2048).  Decode passes run `layers` layers, each with a cache or state of its own, captured in
one graph, as the model runner captures a decode step; steps with prompt rows run eagerly.

  gqa      Llama's attention over paged caches (bf16 or e4m3 elements)
  llama    a prompt step of the Llama model: forward and logits
  plain    layer-listed models: grouped-query attention, causal / window / chunk masks (Povurax with fine weights)
  diff     two-map (differential) attention with its combine: window with kept first keys, or chunks
  latent   latent attention: one shared row per key is key and value
  capped   window attention with a tanh cap, a log-distance penalty
  sigmoid  window attention with sigmoid weights, bias and gate per head
  delta    the generalized delta rule with its head norm and gate
  ssd      Mamba-2: short convolution, state-space scan, gated group norm
  scan     retention and gated linear attention with their head norm and gate
  moe      routed experts: router, plan, grouped GEMMs, combine
"""
import math

import torch

from dynamo_exp_amd import ops
from dynamo_exp_amd.models.config import get_config
from dynamo_exp_amd.models.llama import AttnMeta
from dynamo_exp_amd.models.registry import build_model
from dynamo_exp_amd.ops import mixers as mx
from dynamo_exp_amd.ops import moe
from dynamo_exp_amd.ops import recurrent as rc

DEV = "cuda"
BF = torch.bfloat16
BS = 64  # tokens per cache page, the engine's default
EPS = 1e-5
KV_SCALES = (0.05, 0.04)
HEADS = {"8b": (32, 8, 4096), "1b": (16, 4, 2048)}  # query heads, key/value heads, width; heads of 128
D = 128
# (latent + key part, latent) widths: the layer-listed presets and bench
LATENT = {"r192": (256, 192), "r256": (256, 256)}
EXPERTS = {"8b": (16, 2, 3584), "1b": (8, 2, 2048)}  # experts, chosen, expert width


def _c(name, kind, size="8b", prompts=0, tokens=0, past=0, streams=0, ctx=0, layers=1, **more):
    return dict(name=name, kind=kind, size=size, prompts=prompts, tokens=tokens, past=past, streams=streams, ctx=ctx,
                layers=layers, **more)


def listed():
    return [
        # one short chat: the latency of a decode step, launches and all
        _c("gqa decode, one stream", "gqa", streams=1, ctx=700, layers=8, cache="bf16"),
        # a full server at the benchmark's lengths (3000 in, 150 out) with an e4m3 cache
        _c("gqa decode, 96 streams, fp8", "gqa", streams=96, ctx=3150, layers=2, cache="fp8"),
        # prompts of about that length through two layers of the model and its head
        _c("llama prompt step", "llama", prompts=3, tokens=6151),
        # prompt chunks beside decoding streams: the mixed step that a loaded engine runs most
        _c("diff mixed step", "diff", prompts=2, tokens=5003, past=1024, streams=16, ctx=2100, mask="window",
           win=1024, keep=64),
        _c("diff decode, 48 streams", "diff", streams=48, ctx=4100, layers=2, mask="window", win=1024, keep=64),
        _c("latent prompt step", "latent", prompts=3, tokens=4203, mask="causal", win=0, sink=False, width="r192"),
        _c("latent decode, 33 streams", "latent", streams=33, ctx=4000, layers=2, mask="causal", win=0, sink=False,
           width="r192"),
        _c("capped window prompt step", "capped", prompts=2, tokens=4500, win=1024),
        _c("delta prompt step", "delta", prompts=3, tokens=4001),
        _c("ssd decode, 64 streams", "ssd", streams=64, ctx=900, layers=2),
        _c("moe prompt step", "moe", tokens=2500, layers=1),
        _c("moe decode, 24 rows", "moe", tokens=24, layers=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more step of the same ranges: any kind of layer; prompt steps of 16 to 6000 tokens in one to six prompts,
    with and without tokens already cached; 1 to 128 streams of contexts from 64 to 6000 (together up to 300000)."""
    kind = rng.choice(["gqa", "gqa", "llama", "plain", "diff", "diff", "latent", "latent", "capped", "sigmoid", "delta",
                       "ssd", "scan", "moe"])
    size = rng.choice(["8b", "8b", "1b"])
    if kind == "llama":
        return {k: v for k, v in _c("", kind, prompts=rng.randint(1, 4), tokens=_log(rng, 600, 6000)).items() if k != "name"}
    if kind == "moe":
        t = _log(rng, 1, 4000)
        return {k: v for k, v in _c("", kind, size, tokens=t, layers=2 if t <= 128 else 1).items() if k != "name"}
    prompts = rng.choice([0, 0, rng.randint(1, 6)])
    tokens = max(prompts, _log(rng, 16, 5000)) if prompts else 0
    past = rng.choice([0, rng.randint(1, 3000)]) if prompts else 0
    streams = rng.choice([0, rng.randint(1, 32)]) if prompts else _log(rng, 1, 128)
    ctx = min(_log(rng, 64, 6000), 300000 // streams) if streams else 0
    more = {}
    if kind == "gqa":
        more = dict(cache=rng.choice(["bf16", "fp8"]))
    elif kind == "plain":
        more = dict(rng.choice([dict(mask="causal", win=0, fine=True), dict(mask="window", win=1024, fine=False),
                                dict(mask="chunk", win=2048, fine=False)]))
    elif kind == "diff":
        more = dict(rng.choice([dict(mask="window", win=1024, keep=64), dict(mask="chunk", win=2048, keep=0)]))
    elif kind == "latent":
        more = dict(rng.choice([dict(mask="causal", win=0, sink=False, width="r192"),
                                dict(mask="window", win=1024, sink=True, width="r192"),
                                dict(mask="window", win=1024, sink=False, width="r256")]))
    elif kind in ("capped", "sigmoid"):
        more = dict(win=rng.choice([512, 1024]))
    elif kind == "scan":
        more = dict(rule=rng.choice(["retention", "gla"]))
    c = _c("", kind, size, prompts, tokens, past, streams, ctx, layers=1 if prompts else rng.randint(1, 4), **more)
    return {k: v for k, v in c.items() if k != "name"}


# ------------------------------------------------------------------ rows of a step
def _sequences(case):
    """[(rows of the step, context including them)] per sequence: ragged prompt chunks, then decode rows."""
    n, T = case["prompts"], case["tokens"]
    out, left = [], T
    for i in range(n):
        r = left if i + 1 == n else max(1, min(left - (n - 1 - i), T * 2 * (i + 1) // (n * (n + 1)) + i % 2))
        left -= r
        out.append((r, r + (case["past"] if i % 2 == 0 else 0)))
    S, ctx = case["streams"], case["ctx"]
    return out + [(1, max(1, ctx - i * (ctx * 3 // 4) // S)) for i in range(S)]


class _Rows:
    """The step's rows as the model runner lays them out."""

    def __init__(self, case, g):
        seqs = _sequences(case)
        self.seqs, self.n = seqs, len(seqs)
        self.T = sum(r for r, _ in seqs)
        self.Tp = sum(r for r, _ in seqs[:case["prompts"]])
        self.max_ctx = max(c for _, c in seqs)
        i64 = dict(dtype=torch.int64, device=DEV)
        self.pos = torch.cat([torch.arange(c - r, c, **i64) for r, c in seqs])
        firsts = [0]
        for r, _ in seqs:
            firsts.append(firsts[-1] + r)
        self.firsts = firsts
        self.seq_rows = torch.tensor(firsts, dtype=torch.int32, device=DEV)
        self.row_seq = torch.cat([torch.full((r,), i, dtype=torch.int32, device=DEV) for i, (r, _) in enumerate(seqs)])
        tiles = [t for i in range(case["prompts"]) for t in mx.tile_list(firsts[i], seqs[i][0])]
        self.tiles = torch.tensor(tiles, dtype=torch.int32, device=DEV).view(-1, 2) if tiles else None
        # pages scattered over the cache, as an engine that has run for a while hands them out
        need = [-(-c // BS) for _, c in seqs]
        self.blocks = sum(need)
        perm = torch.randperm(self.blocks, generator=g, device=DEV).to(torch.int32)
        self.tables = torch.zeros(self.n, max(need), dtype=torch.int32, device=DEV)
        at = 0
        for i, k in enumerate(need):
            self.tables[i, :k] = perm[at:at + k]
            at += k

    def slots(self, i, lo, hi):
        j = torch.arange(lo, hi, device=DEV)
        return self.tables[i].long()[j // BS] * BS + j % BS


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _rn(g, *shape, std=1.0, dtype=BF):
    return torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, std, generator=g)


def _uni(g, n, lo, hi):
    return torch.rand(n, generator=g, device=DEV) * (hi - lo) + lo


# ------------------------------------------------------------------ inputs
def _attention_inputs(case, g):
    """One layer's queries and caches, and the arguments of its attention."""
    R = _Rows(case, g)
    H, G, _ = HEADS[case["size"]]
    kind = case["kind"]
    layers = []
    for _ in range(case["layers"]):
        L = {}
        if kind == "gqa":
            L["q"] = _rn(g, R.T, H + 2 * G, D)  # the fused projection's rows; the queries are its leading heads
            kv = [_rn(g, R.blocks, G, BS, D) for _ in range(2)]
            if case["cache"] == "fp8":
                kv = [(t.float() / s).to(torch.float8_e4m3fn) for t, s in zip(kv, KV_SCALES)]
            L["k"], L["v"] = kv
        elif kind == "latent":
            d, dv = LATENT[case["width"]]
            L["q"] = _rn(g, R.T, H * d)
            L["k"] = L["v"] = _rn(g, R.blocks * BS, d)
            if case["sink"]:
                L["sink"] = _rn(g, H, dtype=torch.float32)
        elif kind == "diff":
            L["q"] = _rn(g, R.T, (H + G) * D + G // 2 * 2 * D + H // 2)  # [q | k | v | gate]
            L["k"], L["v"] = _rn(g, R.blocks * BS, G * D), _rn(g, R.blocks * BS, G // 2 * 2 * D)
        else:
            L["q"] = _rn(g, R.T, (H + 2 * G) * D + H)  # [q | k | v | gate per head]
            L["k"], L["v"] = (_rn(g, R.blocks * BS, G * D) for _ in range(2))
            if kind == "capped":
                L["r1"], L["r2"] = _uni(g, H, 0.0, 1.0), _uni(g, H, 0.1, 1.1)
            if kind == "sigmoid":
                L["hb"] = _rn(g, H, dtype=torch.float32) - 2.0
        layers.append(L)
    return R, layers


def _parts(R, case, units, visible, target):
    rows = R.T - R.Tp
    return mx.row_attention_parts(max(rows, 1), units, min(R.max_ctx, visible) if visible else R.max_ctx, target)


def _attend(case, R, L, work):
    """One layer's attention over the step's rows, as its model calls it."""
    kind, (H, G, _) = case["kind"], HEADS[case["size"]]
    if kind == "gqa":
        q = L["q"][:, :H]
        out = torch.empty((R.T, H, D), dtype=BF, device=DEV)
        kw = dict(kv_scales=KV_SCALES if case["cache"] == "fp8" else (1.0, 1.0))
        np_ = case["prompts"]
        if R.Tp:
            ops.prefill_attention(q[:R.Tp], L["k"], L["v"], R.tables[:np_], R.seq_rows[:np_ + 1], work["ctx"][:np_], D ** -0.5,
                                  out[:R.Tp], work=work["list"], scratch=work["scratch"], **kw)
        if R.T > R.Tp:
            ops.decode_attention(q[R.Tp:], L["k"], L["v"], R.tables[np_:], work["ctx"][np_:], D ** -0.5, out[R.Tp:],
                                 work["parts"], workspace=work["ws"], **kw)
        return out
    seq, tables = (R.row_seq, R.tables) if R.Tp else (None, R.tables)
    tl = (R.tiles, R.Tp) if R.Tp else (None, 0)
    if kind == "latent":
        d, dv = LATENT[case["width"]]
        units = -(-H // 32)
        a = mx.attention(L["q"], L["k"], L["k"], R.pos, seq, tables, BS, H, 1, H, d, dv, d ** -0.5, case["mask"], case["win"],
                         _parts(R, case, units, case["win"], mx.LATENT_TARGET_GROUPS), False, *tl, sink=L.get("sink"))
        return a
    if kind == "diff":
        a = mx.attention(L["q"], L["k"], L["v"], R.pos, seq, tables, BS, H, 2, H // G, D, 2 * D, D ** -0.5, case["mask"],
                         case["win"], _parts(R, case, G, case["win"] + case["keep"], mx.GROUP_TARGET_WAVES), True, *tl,
                         keep_first=case["keep"])
        g0 = L["q"].shape[1] - H // 2
        return mx.diff_combine(a.view(R.T, H // 2, 2, 2 * D), 0.35, 0.7, EPS, BF, head_gate=L["q"][:, g0:])
    more = {}
    mask, win = case.get("mask", "window"), case["win"]
    if kind == "plain":
        more = dict(fine_weights=case["fine"])
    elif kind == "capped":
        more = dict(softcap=30.0, dist_bias=(L["r1"], L["r2"]))
    elif kind == "sigmoid":
        more = dict(weights="sigmoid", head_bias=L["hb"], head_gate=L["q"][:, (H + 2 * G) * D:])
    return mx.attention(L["q"], L["k"], L["v"], R.pos, seq, tables, BS, H, 1, H // G, D, D, D ** -0.5, mask, win,
                        _parts(R, case, G, win, mx.GROUP_TARGET_WAVES), False, *tl, **more)


def _gqa_work(case, R):
    """What the model runner builds for a step of Llama's attention."""
    if case["kind"] != "gqa":
        return None
    H, G, _ = HEADS[case["size"]]
    n, S = case["prompts"], case["streams"]
    ctx = [c for _, c in R.seqs]
    w = {"ctx": torch.tensor(ctx, dtype=torch.int32, device=DEV), "list": None, "scratch": None, "parts": 1, "ws": None}
    if n:
        w["list"] = torch.tensor(ops.prefill_work_list([r for r, _ in R.seqs[:n]], ctx[:n], H, G), dtype=torch.int32, device=DEV)
        if case["cache"] == "fp8":
            (_, _, nb, tab), = ops.fp8_scratch_plan(ctx[:n], BS, R.tables.shape[1], 1 << 20)
            w["scratch"] = (torch.from_numpy(tab).to(DEV), nb)
    if S:
        w["parts"] = ops.decode_num_parts(S, G, 8192)
        w["ws"] = ops.decode_workspace(S, H, D, w["parts"], torch.device(DEV))
    return w


def _recurrent_inputs(case, g):
    R = _Rows(case, g)
    H, _, W = HEADS[case["size"]]
    n = H * D
    R.slots_t = torch.randperm(R.n, generator=g, device=DEV).to(torch.int32)
    layers = []
    for _ in range(case["layers"]):
        L = {}
        if case["kind"] == "delta":
            L["p"], L["w"] = _rn(g, R.T, 5 * n + W), _rn(g, R.T, n, std=0.5)  # [r | k | v | gate | a | ...], decay logits
            L["ab"], L["wb"] = _rn(g, n, std=0.5, dtype=torch.float32), _rn(g, n, dtype=torch.float32)
            L["norm"] = 1.0 + _rn(g, n, std=0.1, dtype=torch.float32)
            L["S"] = _rn(g, R.n, H, D, D, dtype=torch.float32)
        elif case["kind"] == "ssd":
            Hs, P, N, Gs = 2 * W // 64, 64, 128, 8
            inner, C = Hs * P, Hs * P + 2 * Gs * N
            L["p"] = _rn(g, R.T, inner + C + Hs)  # [z | x | B | C | dt]
            L["cw"], L["cb"] = _rn(g, 4, C, std=0.5, dtype=torch.float32), _rn(g, C, std=0.1, dtype=torch.float32)
            L["dtb"], L["rate"] = _uni(g, Hs, -4.0, -1.0), torch.exp(_uni(g, Hs, 0.0, 2.5))
            L["skip"], L["norm"] = 1.0 + _rn(g, Hs, std=0.2, dtype=torch.float32), 1.0 + _rn(g, inner, std=0.1, dtype=torch.float32)
            L["S"], L["tail"] = _rn(g, R.n, Hs, P, N, dtype=torch.float32), _rn(g, R.n, 3, C)
        else:
            L["p"] = _rn(g, R.T, 4 * n)  # [q | k | v | gate]
            L["norm"] = 1.0 + _rn(g, n, std=0.1, dtype=torch.float32)
            L["S"] = _rn(g, R.n, H, D, D, dtype=torch.float32)
            if case["rule"] == "gla":
                L["z"], L["zb"] = _rn(g, R.T, n), _uni(g, n, 1.0, 5.0)
            else:
                L["decay"] = torch.tensor([1.0 - 2.0 ** (-5 - 3 * h / max(1, H - 1)) for h in range(H)], device=DEV)
        layers.append(L)
    return R, layers


def _recur(case, R, L):
    """One recurrent layer between its projections, as its model calls it; the state is updated in place."""
    H, _, W = HEADS[case["size"]]
    n, p = H * D, L["p"]
    seq_rows = R.seq_rows if R.Tp else None
    if case["kind"] == "delta":
        o = rc.delta_rule(p[:, :n], p[:, n:2 * n], p[:, 2 * n:3 * n], p[:, 4 * n:5 * n], L["w"], L["ab"], L["wb"], L["S"], R.pos,
                          seq_rows, R.slots_t, H, D, D)
        return rc.head_norm_gate(o, H, L["norm"], p[:, 3 * n:4 * n], EPS, BF)
    if case["kind"] == "ssd":
        Hs, P, N, Gs = 2 * W // 64, 64, 128, 8
        inner, C = Hs * P, Hs * P + 2 * Gs * N
        x = rc.causal_conv(p[:, inner:inner + C], L["cw"], L["tail"], R.pos, R.row_seq if R.Tp else None, seq_rows, R.slots_t,
                           bias=L["cb"], act="silu")
        y = rc.ssd(x[:, :inner], x[:, inner:inner + Gs * N], x[:, inner + Gs * N:], p[:, inner + C:], L["dtb"], L["rate"],
                   L["skip"], L["S"], R.pos, seq_rows, R.slots_t, Hs, Gs, N, P)
        return rc.gate_group_norm(y, p[:, :inner], L["norm"], Gs, EPS, BF)
    if case["rule"] == "gla":
        o = rc.gated_linear_attention(p[:, :n], p[:, n:2 * n], p[:, 2 * n:3 * n], L["z"], L["zb"], 16.0, D ** -0.5, L["S"], R.pos,
                                      seq_rows, R.slots_t, H, D, D)
    else:
        o = rc.retention(p[:, :n], p[:, n:2 * n], p[:, 2 * n:3 * n], L["decay"], D ** -0.5, L["S"], R.pos, seq_rows, R.slots_t,
                         H, D, D)
    return rc.head_norm_gate(o, H, L["norm"], p[:, 3 * n:], EPS, BF, gate_act="silu")


def _moe_inputs(case, g):
    _, _, W = HEADS[case["size"]]
    E, _, F = EXPERTS[case["size"]]
    layers = []
    for _ in range(case["layers"]):
        L = dict(h=_rn(g, case["tokens"], W), router=_rn(g, E, W, std=W ** -0.5, dtype=torch.float32),
                 corr=_rn(g, E, std=0.05, dtype=torch.float32), gu=_rn(g, E, 2 * F, W, std=W ** -0.5),
                 down=_rn(g, E, W, F, std=F ** -0.5))
        layers.append(L)
    return layers


def _experts(case, L):
    E, top, _ = EXPERTS[case["size"]]
    idx, w, _ = moe.router(L["h"], L["router"], E, L["corr"], top, score="softmax", renorm=True, scale=1.5)
    order, offsets = moe.plan(idx, E)
    a = moe.grouped_gemm(L["h"], L["wgu"], order, offsets, top, gather=True, scatter=False, glu=L["fused"])
    a = a if L["fused"] else mx.glu_act(a, "silu")
    y = moe.grouped_gemm(a, L["down"], order, offsets, top, gather=False, scatter=True)
    return moe.combine(y, w), idx


def _llama_config():
    return get_config("llama3-8b@2")


def _llama_state(case, seed):
    """The first two layers and the head, prepared as the engine prepares the model, and the step as its runner does."""
    cfg = _llama_config()
    m = build_model(cfg, device=torch.device(DEV)).random_init(seed)
    m.enable_fused_mlp()
    m.fold_norms()
    g = _gen(seed + 1)
    R = _Rows(case, g)
    ids = torch.randint(3, cfg.vocab_size, (R.T,), generator=g, device=DEV)
    ql = [r for r, _ in R.seqs]
    caches = [tuple(torch.zeros(R.blocks, m.n_kv, BS, D, dtype=BF, device=DEV) for _ in range(2)) for _ in range(2)]
    meta = AttnMeta(is_prefill=True, positions=R.pos,
                    slot_mapping=torch.cat([R.slots(i, c - r, c) for i, (r, c) in enumerate(R.seqs)]), block_tables=R.tables,
                    ctx_lens=torch.tensor([c for _, c in R.seqs], dtype=torch.int32, device=DEV),
                    logits_idx=torch.tensor([x - 1 for x in R.firsts[1:]], device=DEV), cu_seqlens_q=R.seq_rows,
                    work=torch.tensor(ops.prefill_work_list(ql, ql, m.n_q, m.n_kv), dtype=torch.int32, device=DEV),
                    num_prefill_tokens=R.T)
    return dict(model=m, ids=ids, meta=meta, caches=caches)


# ------------------------------------------------------------------ a pass
def _pass(st):
    case, kind = st["case"], st["case"]["kind"]
    if kind == "llama":
        h = st["model"].forward(st["ids"], st["meta"], st["caches"])
        return {"logits": st["model"].compute_logits(h), "caches": st["caches"]}
    if kind == "moe":
        return [_experts(case, L) for L in st["layers"]]
    if kind in ("delta", "ssd", "scan"):
        return [dict(out=_recur(case, st["rows"], L), state=L["S"], **({"tail": L["tail"]} if "tail" in L else {}))
                for L in st["layers"]]
    return [_attend(case, st["rows"], L, st["work"]) for L in st["layers"]]


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    st = {"case": case}
    with torch.inference_mode():
        if kind == "llama":
            st.update(_llama_state(case, seed))
        elif kind == "moe":
            st["layers"] = _moe_inputs(case, g)
            for L in st["layers"]:  # as the models load experts: interleaved where the fused SwiGLU epilogue serves the shape
                L["fused"] = moe.tile_gemm_ok(L["h"], L["gu"])
                L["wgu"] = moe.interleave_glu(L["gu"]) if L["fused"] else L["gu"]
                del L["gu"]
        elif kind in ("delta", "ssd", "scan"):
            st["rows"], st["layers"] = _recurrent_inputs(case, g)
        else:
            st["rows"], st["layers"] = _attention_inputs(case, g)
            st["work"] = _gqa_work(case, st["rows"])
        if case["prompts"] == 0 and not (kind == "moe" and case["tokens"] > 256):
            _capture(st)
    return st


def _capture(st):
    """The decode step as a graph, as the model runner captures it; recurrent state is put back after the warm-up."""
    keep = [(L[k], L[k].clone()) for L in st["layers"] for k in ("S", "tail") if k in L]
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        _pass(st)
    torch.cuda.current_stream().wait_stream(s)
    for t, was in keep:
        t.copy_(was)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        st["out"] = _pass(st)
    st["graph"] = g


def run(state):
    with torch.inference_mode():
        if "graph" in state:
            state["graph"].replay()
            return state["out"]
        return _pass(state)


# ------------------------------------------------------------------ what a pass cannot do without
def _visible(case, r, c):
    """(sum over a sequence's rows of the keys each sees, keys that any of them sees)."""
    mask, win, keep = case.get("mask", "causal"), case.get("win", 0), case.get("keep", 0)
    if case["kind"] in ("capped", "sigmoid"):
        mask = "window"
    total, first = 0, None
    for p in range(c - r, c):
        lo = max(0, p - win + 1) if mask == "window" else p // win * win if mask == "chunk" else 0
        first = lo if first is None else first
        total += p - lo + 1 + min(keep, lo)
    return total, c - first + min(keep, first)


def work(case):
    kind = case["kind"]
    H, G, W = HEADS[case["size"]]
    n = case["layers"]
    if kind == "llama":
        T, cfg = case["tokens"], _llama_config()
        F, V, B = cfg.intermediate_size, cfg.vocab_size, case["prompts"]
        per = (H + 2 * G) * D * W + W * H * D + 3 * W * F
        att = sum(_visible(case, r, c)[0] for r, c in _sequences(case)) * 4 * D * H
        return {"bytes": 2.0 * (2 * per + V * W + T * W + 2 * T * 2 * G * D + B * V), "flops": 2 * (2.0 * T * per + att) + 2.0 * B * V * W}
    if kind == "moe":
        E, top, F = EXPERTS[case["size"]]
        T = case["tokens"]
        used = E * (1 - (1 - top / E) ** T)  # experts that some token chooses
        return {"bytes": n * (used * 3 * F * W * 2.0 + E * W * 4 + T * W * 4), "flops": n * (6.0 * T * top * F * W + 2.0 * T * E * W)}
    seqs = _sequences(case)
    T = sum(r for r, _ in seqs)
    if kind == "delta":
        return {"bytes": n * (T * H * D * (6 * 2 + 2.0) + len(seqs) * H * D * D * 8), "flops": n * 10.0 * T * H * D * D}
    if kind == "ssd":
        inner, C = 2 * W, 2 * W + 2048
        return {"bytes": n * (T * (inner + C + inner // 64 + inner) * 2.0 + len(seqs) * (inner * 128 * 8 + 12 * C)),
                "flops": n * T * (8.0 * C + 6.0 * inner * 128)}
    if kind == "scan":
        wide = 6 if case["rule"] == "gla" else 5
        return {"bytes": n * (T * H * D * wide * 2.0 + len(seqs) * H * D * D * 8), "flops": n * 6.0 * T * H * D * D}
    d, dv, kb, el = D, D, 2 * G * D, 2
    if kind == "latent":
        d, dv = LATENT[case["width"]]
        kb = d
    elif kind == "diff":
        dv = 2 * D
    elif kind == "gqa":
        el = 1 if case["cache"] == "fp8" else 2
    vis = [_visible(case, r, c) for r, c in seqs]
    out = H * dv if kind != "diff" else H // 2 * dv
    return {"bytes": n * (2.0 * T * (H * d + out) + el * kb * sum(k for _, k in vis)),
            "flops": n * 2.0 * (d + dv) * H * sum(t for t, _ in vis)}


def tolerance(case):
    """bf16 results: one rounding of the result and of the softmax weights or activations on the way; the two-map
    combine divides by the size of a difference; two layers of the model add up the roundings of every activation."""
    kind = case["kind"]
    if kind == "llama":
        return {"rel": 0.018, "max": 0.3}  # 0.0044 from the 64-bit values
    if kind == "moe":
        return {"rel": 0.012, "max": 0.2, "differ": 0.003}  # 0.0029
    return {"rel": 0.008, "max": 0.2}  # 0.0017 to 0.0023


# ------------------------------------------------------------------ the same in 64 bits
def _exact_attention(case, R, L):
    kind, (H, G, _) = case["kind"], HEADS[case["size"]]
    maps = 2 if kind == "diff" else 1
    d, dv, group = D, D, H // G
    if kind == "latent":
        (d, dv), group = LATENT[case["width"]], H
    elif kind == "diff":
        dv = 2 * D
    mask, win, keep = case.get("mask", "causal"), case.get("win", 0), case.get("keep", 0)
    if kind in ("capped", "sigmoid"):
        mask = "window"
    out = torch.empty(R.T, H, dv, dtype=torch.float64, device=DEV)
    for i, (r, c) in enumerate(R.seqs):
        rows = slice(R.firsts[i], R.firsts[i + 1])
        if kind == "gqa":
            j = torch.arange(c, device=DEV)
            blk, off = R.tables[i].long()[j // BS], j % BS
            K, V = (L[x][blk, :, off].double() for x in ("k", "v"))
            if case["cache"] == "fp8":
                K, V = K * KV_SCALES[0], V * KV_SCALES[1]
        else:
            sl = R.slots(i, 0, c)
            K = L["k"][sl].double().view(c, -1, d)
            V = (L["k"][sl, :dv].double() if kind == "latent" else L["v"][sl].double()).view(c, -1, dv)
        Q = (L["q"][rows, :H] if kind == "gqa" else L["q"][rows, :H * d].reshape(r, H, d)).double()
        p = torch.arange(c - r, c, device=DEV)[:, None]
        j = torch.arange(c, device=DEV)[None, :]
        lo = (p - win + 1).clamp_min(0) if mask == "window" else p // win * win if mask == "chunk" else p * 0
        vis = (j <= p) & ((j >= lo) | (j < keep))
        for h in range(H):
            hd = h // maps
            s = (Q[:, h] @ K[:, hd // group * maps + h % maps].t()) * d ** -0.5
            if kind == "capped":
                s = 30.0 * torch.tanh(s / 30.0)
                s = s - L["r1"][h].double() * torch.log1p(L["r2"][h].double() * (p - j).clamp_min(0))
            if kind == "sigmoid":
                w = torch.sigmoid(s + L["hb"][h].double()) * vis
            else:
                s = s.masked_fill(~vis, float("-inf"))
                if "sink" in L:
                    s = torch.cat([s, L["sink"][h].double().expand(r, 1)], 1)
                w = torch.softmax(s, -1)[:, :c]
            out[rows, h] = w @ V[:, hd // group]
    if kind == "sigmoid":
        out = out * torch.sigmoid(L["q"][:, (H + 2 * G) * D:].double())[:, :, None]
    if kind == "diff":
        a = out.view(R.T, H // 2, 2, dv)
        o = a[:, :, 0] - 0.35 * a[:, :, 1]
        o = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + EPS) * 0.7
        return (o * torch.sigmoid(L["q"][:, L["q"].shape[1] - H // 2:].double())[:, :, None]).reshape(R.T, -1)
    return out


def _exact_recur(case, R, L):
    kind, (H, _, W) = case["kind"], HEADS[case["size"]]
    n, T, S = H * D, R.T, L["S"].double().transpose(2, 3).clone()  # [slots, H, dk, dv]
    slots = R.slots_t.long()
    p = L["p"].double()
    fresh = torch.tensor([c == r for r, c in R.seqs], device=DEV)
    S[slots[fresh]] = 0.0
    new_tail = None
    if kind == "ssd":
        Hs, P, N, Gs = 2 * W // 64, 64, 128, 8
        inner, C = Hs * P, Hs * P + 2 * Gs * N
        u, tail = p[:, inner:inner + C], L["tail"].double()
        x, new_tail = torch.empty_like(u), tail.clone()
        for i, (r, c) in enumerate(R.seqs):
            t = tail[slots[i]].clone()
            t[:max(0, 3 - (c - r))] = 0.0
            full = torch.cat([t, u[R.firsts[i]:R.firsts[i + 1]]])
            x[R.firsts[i]:R.firsts[i + 1]] = sum(full[j:j + r] * L["cw"][j].double() for j in range(4)) + L["cb"].double()
            new_tail[slots[i]] = full[-3:]
        x = x * torch.sigmoid(x)
        dt = torch.nn.functional.softplus(p[:, inner + C:] + L["dtb"].double(), threshold=1e6)
        decay = torch.exp(-L["rate"].double() * dt)[:, :, None, None]
        v = x[:, :inner].view(T, Hs, P)
        k, q = (x[:, inner + o:inner + o + Gs * N].view(T, Gs, N).repeat_interleave(Hs // Gs, 1) for o in (0, Gs * N))
        kv_scale = dt
    else:
        q, k, v = (p[:, i * n:(i + 1) * n].view(T, H, D) for i in range(3))
        kv_scale = None
        if kind == "delta":
            w = torch.exp(-math.exp(-0.5) * torch.sigmoid(L["w"].double() + L["wb"].double())).view(T, H, D)
            a = torch.sigmoid(p[:, 4 * n:5 * n] + L["ab"].double()).view(T, H, D)
            unit = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
        elif case["rule"] == "gla":
            decay = torch.exp(torch.nn.functional.logsigmoid(L["z"].double() + L["zb"].double()) / 16.0).view(T, H, D, 1)
            q = q * D ** -0.5
        else:
            decay = L["decay"].double().view(1, H, 1, 1).expand(T, H, 1, 1)
            k = k * D ** -0.5
    o = torch.empty(T, S.shape[1], S.shape[3], dtype=torch.float64, device=DEV)
    firsts = torch.tensor(R.firsts[:-1], device=DEV)
    lens = torch.tensor([r for r, _ in R.seqs], device=DEV)
    for t in range(max(r for r, _ in R.seqs)):
        on = lens > t
        sl, row = slots[on], firsts[on] + t
        s = S[sl]
        if kind == "delta":
            us = torch.einsum("bhi,bhij->bhj", unit[row], s)
            s = w[row][..., None] * s - (a[row] * unit[row])[..., None] * us[:, :, None]
            s += k[row][..., None] * v[row][:, :, None]
        else:
            kk = k[row] if kv_scale is None else k[row] * kv_scale[row][:, :, None]
            s = decay[row] * s + kk[..., None] * v[row][:, :, None]
        S[sl] = s
        o[row] = torch.einsum("bhi,bhij->bhj", q[row], s)
    if kind == "ssd":
        o = (o + L["skip"].double()[:, None] * v).reshape(T, -1)
        z = p[:, :inner]
        o = (o * z * torch.sigmoid(z)).view(T, Gs, -1)
        out = (o * torch.rsqrt((o * o).mean(-1, keepdim=True) + EPS)).reshape(T, -1) * L["norm"].double()
    else:
        out = (o * torch.rsqrt((o * o).mean(-1, keepdim=True) + EPS)).reshape(T, n) * L["norm"].double()
        z = p[:, 3 * n:4 * n]
        out = out * (torch.sigmoid(z) if kind == "delta" else z * torch.sigmoid(z))
    got = dict(out=out, state=S.transpose(2, 3).contiguous())
    if new_tail is not None:
        got["tail"] = new_tail
    return got


def _exact_moe(case, L):
    E, top, F = EXPERTS[case["size"]]
    h = L["h"].double()
    s = torch.softmax(h @ L["router"].double().t(), -1)
    idx = (s + L["corr"].double()).topk(top, -1).indices
    w = s.gather(1, idx)
    w = w / (w.sum(-1, keepdim=True) + 1e-20) * 1.5
    out = torch.zeros_like(h)
    for e in range(E):
        t, k = (idx == e).nonzero(as_tuple=True)
        if t.numel():
            gu = h[t] @ L["gu"][e].double().t()
            out[t] += (torch.nn.functional.silu(gu[:, :F]) * gu[:, F:]) @ L["down"][e].double().t() * w[t, k][:, None]
    return out, idx.to(torch.int32)


def _exact_llama(case, seed):
    cfg = _llama_config()
    W, F, V, n = cfg.hidden_size, cfg.intermediate_size, cfg.vocab_size, cfg.num_hidden_layers
    H, G = cfg.num_attention_heads, cfg.num_key_value_heads
    g = _gen(seed)  # the weights, in the order and with the spreads of random_init
    layers = [dict(qkv=_rn(g, (H + 2 * G) * D, W, std=1 / math.sqrt(W)),
                   o=_rn(g, W, H * D, std=1 / math.sqrt(H * D) / math.sqrt(n)), gu=_rn(g, 2 * F, W, std=1 / math.sqrt(W)),
                   down=_rn(g, W, F, std=1 / math.sqrt(F) / math.sqrt(n))) for _ in range(n)]
    embed, head = _rn(g, V, W), _rn(g, V, W, std=1 / math.sqrt(W))
    g = _gen(seed + 1)
    R = _Rows(case, g)
    ids = torch.randint(3, V, (R.T,), generator=g, device=DEV)
    x = embed[ids].double()
    ang = R.pos.double()[:, None] * (1.0 / cfg.rope_theta ** (torch.arange(0, D, 2, device=DEV).double() / D))
    cos, sin = torch.cos(ang)[:, None], torch.sin(ang)[:, None]

    def norm(t):
        return t * torch.rsqrt((t * t).mean(-1, keepdim=True) + cfg.rms_norm_eps)

    def rot(t):
        a, b = t[..., :D // 2], t[..., D // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    caches = []
    for L in layers:
        p = norm(x) @ L["qkv"].double().t()
        q, k = rot(p[:, :H * D].view(-1, H, D)), rot(p[:, H * D:(H + G) * D].view(-1, G, D))
        v = p[:, (H + G) * D:].view(-1, G, D)
        a = torch.empty_like(q)
        kv = [torch.zeros(R.blocks, G, BS, D, dtype=torch.float64, device=DEV) for _ in range(2)]
        for i, (r, c) in enumerate(R.seqs):
            s0, s1 = R.firsts[i], R.firsts[i + 1]
            j = torch.arange(r, device=DEV)
            for t, src in zip(kv, (k, v)):
                t[R.tables[i].long()[j // BS], :, j % BS] = src[s0:s1]
            future = j[None, :] > j[:, None]
            for h in range(H):
                s = (q[s0:s1, h] @ k[s0:s1, h // (H // G)].t()) * D ** -0.5
                a[s0:s1, h] = torch.softmax(s.masked_fill(future, float("-inf")), -1) @ v[s0:s1, h // (H // G)]
        caches.append(tuple(kv))
        x = x + a.view(-1, H * D) @ L["o"].double().t()
        gu = norm(x) @ L["gu"].double().t()
        x = x + (torch.nn.functional.silu(gu[:, :F]) * gu[:, F:]) @ L["down"].double().t()
    last = torch.tensor([t - 1 for t in R.firsts[1:]], device=DEV)
    return {"logits": norm(x[last]) @ head.double().t(), "caches": caches}


def exact(case, seed):
    g, kind = _gen(seed), case["kind"]
    with torch.inference_mode():
        if kind == "llama":
            return _exact_llama(case, seed)
        if kind == "moe":
            return [_exact_moe(case, L) for L in _moe_inputs(case, g)]
        if kind in ("delta", "ssd", "scan"):
            R, layers = _recurrent_inputs(case, g)
            return [_exact_recur(case, R, L) for L in layers]
        R, layers = _attention_inputs(case, g)
        return [_exact_attention(case, R, L) for L in layers]
