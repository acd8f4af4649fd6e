"""The expert plan and the routers (csrc/mixers/moe.hip) where their runs of slots, bits of expert numbers and passes over
outputs end."""
from __future__ import annotations

import pytest
import torch

from dynamo_exp_amd.ops import moe


@pytest.mark.gpu
@pytest.mark.parametrize("E", [1, 2, 3, 16, 63, 64, 127, 255, 256, 257, 600])
@pytest.mark.parametrize("T,top", [(1, 1), (1, 8), (9, 7), (64, 16), (65, 16), (1025, 8), (8200, 2)])
def test_plan(E, T, top):
    """Slots in order within an expert; choices that are no expert hold no place."""
    torch.manual_seed(E + T)
    idx = torch.randint(0, E + 2, (T, top), dtype=torch.int32)
    if E > 4:
        idx[T // 2:] = idx[T // 2:] % 3  # most experts end early
    order, offsets = moe.plan(idx.cuda(), E)
    want, want_off = moe.plan(idx, E)
    assert torch.equal(offsets.cpu(), want_off)
    n = int(want_off[-1])
    assert torch.equal(order.cpu()[:n], want[:n])


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 40, 257, 4097])
@pytest.mark.parametrize("n_route,n", [(1, 1), (8, 8), (7, 9), (16, 16), (16, 17), (32, 33), (64, 64)])
@pytest.mark.parametrize("W", [96, 250, 2048])
def test_router(T, n_route, n, W):
    """Passes over 8, 16 and 32 outputs and their remainders, widths that are no multiple of a wave's pieces."""
    torch.manual_seed(T + n + W)
    h, w = torch.randn(T, W).bfloat16(), torch.randn(n, W) * 0.05
    top = min(2, n_route)
    z = h.double() @ w.double().t()
    s = torch.sigmoid(z[:, :n_route])
    idx, wt, gates = moe.router(h.cuda(), w.cuda(), n_route, None, top)
    idx, wt = idx.cpu().long(), wt.cpu().double()
    # true fp32 products and sums of W terms of 0.05: a choice may differ only between scores that close
    tol = 2 ** -22 * W ** 0.5
    assert (s.gather(1, idx) - wt).abs().max() < tol
    assert (s.topk(top, -1).values - wt).abs().max() < tol
    if n > n_route:
        assert (torch.sigmoid(z[:, n_route:]) - gates.cpu().double()).abs().max() < tol
