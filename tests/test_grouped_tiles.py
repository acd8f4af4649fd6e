"""Row tiles of the grouped 256-tile GEMM (csrc/kernels/gemm256.hip): experts whose runs of rows end at every kind of
edge -- of a 16-row block, of a tile of 32 to 256 rows, of the two phases -- and experts without rows."""
from __future__ import annotations

import pytest
import torch

from dynamo_exp_amd.ops import moe

RUNS = [
    [1, 0, 31, 33, 65, 0, 127],  # tiles of 1 to 4 blocks per wave
    [160, 128, 129, 161, 193, 225],  # 4 to 7, the second phase shorter or equal
    [256, 255, 257, 0, 289, 320],  # one full tile, two of unlike rows
    [512, 513, 769, 1],
    [5] + [0] * 69 + [7, 40],  # more experts than lanes
]


@pytest.mark.gpu
@pytest.mark.parametrize("runs", RUNS, ids=lambda r: "-".join(map(str, r[:3])))
@pytest.mark.parametrize("gather,scatter,glu", [(True, False, True), (False, True, False), (True, True, False), (False, False, True)])
def test_runs_of_rows(runs, gather, scatter, glu, monkeypatch):
    monkeypatch.setattr(moe, "stream_gemm_ok", lambda *a: False)  # (few rows per expert would take the streaming kernel)
    torch.manual_seed(len(runs))
    E, N, K, top = len(runs), 512, 256, 2
    R = sum(runs) + sum(runs) % 2
    offsets = torch.tensor([0] + runs).cumsum(0).to(torch.int32)
    order = torch.randperm(R).to(torch.int32)  # the last entry may belong to no expert
    a = torch.randn(R // top if gather else R, K).bfloat16()
    w = torch.randn(E, N, K).bfloat16()
    want = torch.zeros(R, N // 2 if glu else N, dtype=torch.float64)
    for e in range(E):
        r = torch.arange(offsets[e], offsets[e + 1])
        o = order[r].long()
        y = a[o // top if gather else r].double() @ w[e].double().t()
        if glu:
            y = torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:]
        want[o if scatter else r] = y
    wg = (moe.interleave_glu(w) if glu else w).cuda()
    got = moe.grouped_gemm(a.cuda(), wg, order.cuda(), offsets.cuda(), top, gather, scatter, glu).cpu()
    rows = torch.arange(sum(runs))
    rows = order[rows].long() if scatter else rows
    assert torch.isfinite(got[rows]).all()
    # one rounding to bf16 (2^-9 of a value) over fp32 sums of 256 terms and the fast exponential
    err = (got[rows].double() - want[rows]).abs()
    assert (err <= 2 ** -8 * want[rows].abs() + 2 ** -12 * (K if glu else K ** 0.5)).all()
    assert float(err.norm() / want[rows].norm()) < 0.002
