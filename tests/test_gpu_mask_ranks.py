"""Masks with 1-D terms in 2-D loads, stores and dot operands, against float64.
Memory past the bounds holds NaN (guard values in outputs), so an element that
a mask should have kept out shows. Dot tolerance: an fp32 sum of K products,
K * 2^-24 of the sum of magnitudes."""

import pytest
import torch
from test_mask_ranks_cpu import copy_k, dot_k, three_terms_k

import newt

pytestmark = pytest.mark.gpu
copy, three_terms, dot = newt.jit(copy_k), newt.jit(three_terms_k), newt.jit(dot_k)


def padded(rows, cols, ld, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    flat = torch.full(((rows + 1) * ld,), float("nan"), device="cuda", dtype=dtype)
    v = flat.as_strided((rows, cols), (ld, 1))
    v.copy_(torch.randn(rows, cols, generator=g, device="cuda").to(dtype))
    return v


@pytest.mark.parametrize("BM,BN", [(4, 64), (64, 4), (16, 256)])
@pytest.mark.parametrize("dM,dN,pad", [(0, 0, 0), (1, 0, 8), (1, 1, 1), (3, 3, 13), (2, 4, 0)])
def test_row_kernels(BM, BN, dM, dN, pad):
    M, N = BM - dM, max(1, BN - dN)
    ld = N + pad
    x = padded(M, N, ld, torch.float32, BM)
    for kernel in (copy, three_terms):
        o = torch.full((BM + 1, ld), 7.0, device="cuda")
        print(f"mask ranks {M}x{N} ld {ld} block {BM}x{BN} {kernel.__name__}", flush=True)
        kernel[(1,)](x, o, M, N, ld, FULL=False, BM=BM, BN=BN)
        want = torch.full_like(o, 7.0)
        want[:M, :N] = x * 2.0 if kernel is copy else x
        if kernel is three_terms:
            want[:M, :min(8, N)] = 7.0
        assert torch.equal(o, want)


# (tile, M, N, K, elements added to the 16-byte row strides): whole tiles, k
# tails on and inside a 16-byte run, aligned and odd strides
DOTS = [((64, 64, 64, 8, 3), 24, 63, 205, 0), ((64, 64, 64, 8, 3), 31, 56, 648, 1),
        ((128, 64, 32, 4, 4), 64, 64, 512, 0), ((128, 64, 32, 4, 4), 8, 8, 1032, 0),
        ((32, 64, 128, 4, 2), 31, 56, 648, 0), ((32, 64, 128, 4, 2), 24, 63, 205, 1)]


@pytest.mark.parametrize("tile,M,N,K,odd", DOTS)
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (True, True), (False, True)])
def test_dot_operands(tile, M, N, K, odd, ta, tb):
    BM, BN, BK, waves, stages = tile
    M, N = min(M, BM), min(N, BN)
    a = padded(K, M, BM + 16 + odd, torch.float16, 1).t() if ta \
        else padded(M, K, K // 16 * 16 + 16 + odd, torch.float16, 1)
    b = padded(N, K, K // 16 * 16 + 16 + odd, torch.float16, 2).t() if tb \
        else padded(K, N, BN + 16 + odd, torch.float16, 2)
    o = torch.full((BM, BN), float("nan"), device="cuda")
    print(f"mask ranks dot {M}x{N}x{K} ta={ta} tb={tb} odd={odd} tile {BM}x{BN}x{BK}", flush=True)
    dot[(1,)](a, b, o, M, N, K, *a.stride(), *b.stride(), FULL=False, BM=BM, BN=BN, BK=BK,
              num_warps=waves, num_stages=stages)
    A = torch.zeros(BM, K, device="cuda", dtype=torch.float64)
    B = torch.zeros(K, BN, device="cuda", dtype=torch.float64)
    A[:M], B[:, :N] = a.double(), b.double()
    bound = (K + 2) * 2.0 ** -24 * (A.abs() @ B.abs()) + 1e-30
    assert bool(((o.double() - A @ B).abs() <= bound).all())
