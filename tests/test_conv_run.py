"""The short convolution with its tail update in one launch (csrc/mixers/recurrent.hip, conv_run_kernel) against the PyTorch
form: sequences that begin at every place of a run of eight rows, shorter than the taps and across several runs."""
import pytest
import torch

from dynamo_exp_amd.ops import recurrent as rc


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("taps", [1, 2, 3, 4])
@pytest.mark.parametrize("rows", [[1], [8], [7, 2, 1, 30], [6, 1, 1, 1, 9], [5, 3, 2, 2, 2, 1, 0, 4, 17], [1] * 21, [23, 8, 1, 16, 40],
                                  [3, 4, 5, 6, 7, 9, 10, 11, 1, 2]])
def test_runs_and_tails(rows, taps, dtype):
    torch.manual_seed(len(rows) + taps)
    T, C, n = sum(rows), 1032, len(rows)
    x = torch.randn(T, C + 8).to(dtype)[:, :C]
    w, b = torch.randn(taps, C), torch.randn(C)
    tail0 = torch.randn(n + 2, taps - 1, C).to(dtype)
    slots = torch.randperm(n + 2)[:n].to(torch.int32)
    if n > 3:
        slots[2] = -1  # padding rows
    starts = [(0, 1, 2, 50)[i % 4] for i in range(n)]
    pos = torch.cat([torch.arange(s, s + r) for s, r in zip(starts, rows)])
    seq_rows = torch.tensor([0] + rows).cumsum(0).to(torch.int32)
    row_seq = torch.tensor([i for i, r in enumerate(rows) for _ in range(r)], dtype=torch.int32)

    def run(device):
        tail = tail0.clone().to(device)
        at = [t.to(device) for t in (pos, row_seq, seq_rows, slots)]
        return rc.causal_conv(x.to(device), w.to(device), tail, *at, bias=b.to(device), act="silu").cpu(), tail.cpu()

    (want, tail_want), (got, tail) = run("cpu"), run("cuda")
    assert torch.equal(tail, tail_want)
    live = slots[row_seq.long()] >= 0
    # sums of four products of numbers around one in fp32, silu by the hardware's exponential (2^-21); bf16: its rounding
    tol = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -19
    assert torch.allclose(got[live].float(), want[live].float(), rtol=tol, atol=tol)
    assert bool((got[~live] == 0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("taps", [2, 4])
@pytest.mark.parametrize("first,rows", [
    ([0, 9, 16], [0] * 9 + [1] * 2), ([0, 1, 12], [0] + [1] * 10),                 # the last one's end behind the step
    ([0, 2, 11], [0] * 5 + [1] * 6), ([0, 1, 11], [0] * 3 + [1] * 8),              # rows behind their sequence's end
    ([0, 4, 4, 11], [0] * 4 + [1] * 2 + [2] * 5), ([0, 4, 3, 11], [0] * 3 + [1] * 2 + [2] * 6),  # no rows, or fewer than none
    ([0, 5, 11], [0, -1, 0, 0, 0, 1, -1, 7, 1, 1, 1]),                             # rows of no sequence
    ([-1, 4, 11], [0] * 4 + [1] * 7), ([0, 40, 50], [0] * 8 + [1] * 3)])           # a start outside the step
def test_rows_that_the_bounds_do_not_hold(monkeypatch, first, rows, taps, dtype):
    """Bounds and row numbers that do not fit each other: every row is written, and rows and tails are those of the kernel for any
    size with its update behind it."""
    torch.manual_seed(taps)
    T, C, n = len(rows), 264, len(first) - 1
    x, w = torch.randn(T, C).to(dtype).cuda(), torch.randn(taps, C).cuda()
    tail0 = torch.randn(n + 1, taps - 1, C).to(dtype).cuda()
    at = (torch.arange(T).cuda() + 1, torch.tensor(rows, dtype=torch.int32).cuda(), torch.tensor(first, dtype=torch.int32).cuda(),
          torch.arange(1, n + 1, dtype=torch.int32).cuda())
    tail_want, tail = tail0.clone(), tail0.clone()
    want = rc.conv_rope_cache(x, w, tail_want, at[0], torch.full_like(at[0], -1), *at[1:], 1, 0, C, 0, None, None, None)
    rc.conv_state_update(x, tail_want, at[0], *at[2:])
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **k: empty(*a, **k).fill_(float("nan")))
    got = rc.causal_conv(x, w, tail, *at)
    assert torch.equal(tail, tail_want)
    tol = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -19  # (as in test_runs_and_tails)
    assert torch.allclose(got.float(), want.float(), rtol=tol, atol=tol)
