"""The weight-streaming grouped GEMM at the edges of its passes (16, 32 and 64 rows), of its widths (two waves up to 2048,
four beyond, waves without a piece) and for one token, against float64; and the rule that chooses it."""
import pytest
import torch

from dynamo_exp_amd.ops import moe


@pytest.mark.gpu
@pytest.mark.parametrize("counts,K,N", [((2, 0), 2048, 256), ((2, 0), 64, 64), ((2, 0), 2112, 64), ((1, 1, 0, 0), 2048, 96),
                                        ((15, 16, 17, 0, 32, 33), 2048, 64), ((63, 64, 65, 1), 2112, 64),
                                        ((128, 80, 81, 96, 97, 129), 192, 96), ((48, 49, 16), 4096, 256)])
def test_passes_and_waves(monkeypatch, counts, K, N):
    torch.manual_seed(K + N)
    monkeypatch.setattr(moe, "STREAM_ROWS", 1 << 20)
    monkeypatch.setattr(moe, "STREAM_TILES", 1 << 20)
    E, R = len(counts), sum(counts)
    e_of = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    order = torch.randperm(R).to(torch.int32)
    offsets = torch.tensor((0,) + counts).cumsum(0).to(torch.int32)
    a, w = torch.randn(R, K).bfloat16(), (torch.randn(E, N, K) * K ** -0.5).bfloat16()
    ac, wc, oc, fc = a.cuda(), w.cuda(), order.cuda(), offsets.cuda()
    assert moe.stream_gemm_ok(ac, wc, R)
    # result in bf16 (half a step of 2^-8) and sums of K products in float32 (random signs: K steps of 2^-24 of the terms at most)
    close = lambda got, want, bound: bool(((got.cpu().double() - want).abs() <= want.abs() * 2 ** -8 + bound).all())
    terms = float(K) * 2 ** -24 * 16 * K ** -0.5
    want = torch.stack([w[e].double() @ a[r].double() for e, r in zip(e_of.tolist(), order.tolist())])
    assert close(moe.grouped_gemm(ac, wc, oc, fc, 1, gather=True, scatter=False), want, terms)
    rows = torch.stack([w[e].double() @ a[r].double() for r, e in enumerate(e_of.tolist())])
    got = moe.grouped_gemm(ac, wc, oc, fc, 1, gather=False, scatter=True)
    assert close(got[oc.long()], rows, terms)
    if N % 256 == 0:  # (SwiGLU: silu has a slope of 1.1 at most, the up factor at most its largest value)
        got = moe.grouped_gemm(ac, moe.interleave_glu(wc), oc, fc, 1, gather=True, scatter=False, glu=True)
        gate, up = want[:, :N // 2], want[:, N // 2:]
        assert close(got, torch.nn.functional.silu(gate) * up, terms * 2.2 * float(want.abs().max()) + 1e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("E,N,K,most", [(8, 4096, 2048, 32), (16, 7168, 4096, 8), (8, 14336, 4160, 24), (8, 640, 1024, 32)])
def test_rows_it_is_taken_for(E, N, K, most):
    w = torch.empty(1, device="cuda", dtype=torch.bfloat16).expand(E, N, K)
    for R, ok in ((most * E, True), (most * E + 1, False)):
        assert moe.stream_gemm_ok(torch.empty(R, K, device="cuda", dtype=torch.bfloat16), w, R) is ok


@pytest.mark.gpu
@pytest.mark.parametrize("E,N,K,rows", [(16, 2048, 1024, 384), (16, 1024, 1024, 512), (32, 1024, 512, 768), (10, 3072, 1536, 256),
                                        (16, 1408, 2048, 512), (16, 2048, 1088, 512)])
def test_rows_it_is_taken_for_however_they_are_routed(E, N, K, rows):
    """Against the 256-tile kernel more than 24 rows per expert only up to 256 in all or where that kernel's grid is small: beyond,
    an expert that half of the tokens choose holds several passes.  (The last two that kernel does not take.)"""
    w = torch.empty(1, device="cuda", dtype=torch.bfloat16).expand(E, N, K)
    for R, ok in ((rows, True), (rows + 1, False)):
        assert moe.stream_gemm_ok(torch.empty(R, K, device="cuda", dtype=torch.bfloat16), w, R) is ok
