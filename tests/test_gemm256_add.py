"""y += x w^T on the 256-tile kernel (csrc/kernels/gemm256.hip): whole tiles, a last round cut along K, both together;
and which shapes take it."""
from __future__ import annotations

import pytest
import torch

from dynamo_exp_amd import ops


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,pieces", [
    (1, 256, 128, 1),  # one tile whose K does not divide
    (300, 512, 256, 2), (255, 256, 1408, 11), (257, 768, 2304, 16),  # pieces of one and more pairs of K tiles
    (1100, 4096, 512, 3), (2049, 4096, 384, 0), (4096, 4096, 256, 0),  # 80, 144 and 256 tiles
    (4097, 4096, 640, 5), (16500, 512, 2176, 0),  # a full round and 16; 130 tiles
    (33000, 512, 1152, 9),  # 258: the rest in the last rows
])
def test_add(M, N, K, pieces):
    torch.manual_seed(M)
    x, w = torch.randn(M, K, device="cuda").bfloat16(), (torch.randn(N, K, device="cuda") * 0.1).bfloat16()
    y0 = torch.randn(M, N + 4, device="cuda").bfloat16()
    tiles = -(-M // 256) * (N // 256)
    left = tiles % 256 if pieces else 0
    floats = ops._k().gemm256_add_floats(M, N, K)
    assert floats == left * pieces * 65536
    outs = []
    for _ in range(2):
        y = y0.clone()
        ws = torch.full((max(floats, 1),), float("nan"), device="cuda")
        ops._k().gemm256_add(y.data_ptr(), y.stride(0), x.data_ptr(), K, w.data_ptr(), M, N, K, 16, ws.data_ptr(), ops._stream())
        outs.append(y)
    assert torch.equal(*outs) and torch.equal(outs[0][:, N:], y0[:, N:])
    want = y0[:, :N].double() + x.double() @ w.double().t()
    # one rounding to bf16 (2^-9 relative) over fp32 sums of K terms of 0.1
    err = (outs[0][:, :N].double() - want).abs()
    assert bool((err <= 2 ** -8 * want.abs() + 2 ** -22 * K).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,pieces", [
    (6151, 4096, 256, 0),  # 400 tiles: workgroups with a second whole tile, none cut
    (8200, 4096, 512, 4),  # 512 whole tiles, two a workgroup, then pieces of K of 16
    (12295, 4096, 384, 3),  # 768 and 16: three whole tiles a workgroup
])
def test_add_after_add(M, N, K, pieces):
    """A workgroup that adds several tiles, one after the other: a tile's loads of y and stores lie beside the next one's
    first loads."""
    test_add(M, N, K, pieces)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,left,pieces", [
    (2100, 4096, 13312, 16, 16),  # no whole tile
    (6151, 4096, 13440, 16, 16),  # a round in front; 105 pairs of K tiles in 16 pieces
    (16500, 512, 13312, 2, 16),  # a workgroup without a second piece
    (22728, 512, 14336, 50, 5), (7100, 4096, 16384, 64, 4), (5800, 5120, 25600, 76, 3),
])
def test_add_two_kinds(M, N, K, left, pieces):
    """A last round of more than half of the CUs: 128 tiles in two pieces of K, the others in more."""
    torch.manual_seed(M)
    x, w = torch.randn(M, K, device="cuda").bfloat16(), (torch.randn(N, K, device="cuda") * 0.02).bfloat16()
    y0 = torch.randn(M, N + 4, device="cuda").bfloat16()
    floats = ops._k().gemm256_add_floats(M, N, K)
    assert floats == (128 * 2 + left * pieces) * 65536
    outs = []
    for _ in range(2):
        y = y0.clone()
        ws = torch.full((floats,), float("nan"), device="cuda")
        ops._k().gemm256_add(y.data_ptr(), y.stride(0), x.data_ptr(), K, w.data_ptr(), M, N, K, 16, ws.data_ptr(), ops._stream())
        outs.append(y)
    assert torch.equal(*outs) and torch.equal(outs[0][:, N:], y0[:, N:])
    want = torch.addmm(y0[:, :N].double(), x.double(), w.double().t())
    # as above
    assert bool(((outs[0][:, :N].double() - want).abs() <= 2 ** -8 * want.abs() + 2 ** -22 * K).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M", [500, 1280, 1300, 4200])
def test_linear_add(M):
    """The op on both sides of its rule, and rows whose alignment the kernel does not take."""
    torch.manual_seed(M)
    N, K = 4096, 10240
    x, w = torch.randn(M, K, device="cuda").bfloat16(), (torch.randn(N, K, device="cuda") * 0.02).bfloat16()
    assert ops.deep_add_tiles(M, N, K) == (M != 1300)
    want = x.double() @ w.double().t()
    for y in (torch.randn(M, N, device="cuda").bfloat16(), torch.randn(M * N + 1, device="cuda").bfloat16()[1:].view(M, N),
              torch.randn(N, M, device="cuda").bfloat16().t()):
        exact = y.double() + want
        assert ops.linear_add_(y, x, w) is y
        assert bool(((y.double() - exact).abs() <= 2 ** -8 * exact.abs() + 2 ** -22 * K).all())


@pytest.mark.parametrize("M,N,K,left,pieces", [
    # (no pieces: whole tiles are faster there, or two pieces all that fit)
    (6151, 4096, 10240, 16, 0), (6151, 4096, 11008, 16, 0), (6500, 4096, 11520, 32, 0), (6800, 4096, 12288, 48, 0),
    (7100, 4096, 12288, 64, 0), (3500, 8192, 14336, 64, 0), (7300, 4096, 16384, 80, 0), (7525, 4096, 28672, 96, 0),
    (6151, 4096, 12288, 16, 16), (6500, 4096, 13312, 32, 8), (6800, 4096, 14336, 48, 5), (7100, 4096, 16384, 64, 4),
    (3100, 8192, 28672, 32, 8), (7300, 4096, 28672, 80, 3),
])
def test_rule_of_two_kinds(M, N, K, left, pieces):
    assert -(-M // 256) * (N // 256) % 256 == 128 + left
    assert ops._k().gemm256_add_floats(M, N, K) == (128 * 2 + left * pieces if pieces else 0) * 65536


def test_rule_and_cpu():
    ok = ops.deep_add_tiles
    assert ok(600, 4096, 14336) and ok(6151, 4096, 14336) and ok(384, 4096, 10240)
    for shape in ((383, 4096, 14336), (6151, 4096, 10112), (2000, 4096, 14336), (4096, 4096, 14336), (7936, 4096, 14336)):
        assert not ok(*shape), shape
    y, x, w = torch.randn(384, 256), torch.randn(384, 10240), torch.randn(256, 10240)
    want = torch.addmm(y, x, w.t())
    assert torch.equal(ops.linear_add_(y, x, w), want)
