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
