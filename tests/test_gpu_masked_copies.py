"""Ragged tiles of a pipelined dot: where a mask is uniform over 16-byte chunks
and fills with zero, the tile's asynchronous copies run under it (an offset past
the buffer's range writes zeros). Every other mask keeps the register path.
Values past the bounds are NaN in memory, so an unmasked element shows.
Tolerances: an fp32 sum of K products against float64, K * 2^-24 of the sum of
magnitudes."""

import pytest
import torch

import newt
import newt.language as nl

pytestmark = pytest.mark.gpu


@newt.jit
def masked_k(a_ptr, b_ptr, o_ptr, M, N, K, sam, sbk, OTHER: nl.constexpr, BM: nl.constexpr,
             BN: nl.constexpr, BK: nl.constexpr):
    rm, rn, rk = nl.arange(0, BM), nl.arange(0, BN), nl.arange(0, BK)
    pa = a_ptr + rm[:, None] * sam + rk[None, :]
    pb = b_ptr + rk[:, None] * sbk + rn[None, :]
    acc = nl.zeros((BM, BN), dtype=nl.float32)
    for k in range(nl.cdiv(K, BK)):
        a_mask = (rm[:, None] < M) & (rk[None, :] < K - k * BK)
        b_mask = (rk[:, None] < K - k * BK) & (rn[None, :] < N)
        a = nl.load(pa, mask=a_mask, other=OTHER)
        b = nl.load(pb, mask=b_mask, other=0.0)
        acc = nl.dot(a, b, acc)
        pa += BK
        pb += BK * sbk
    nl.store(o_ptr + rm[:, None] * BN + rn[None, :], acc)


def case(M, N, K, lda, ldb, BM, BN, BK, waves, stages, other=0.0, dtype=torch.float16):
    g = torch.Generator(device="cuda").manual_seed(5)

    def padded(rows, cols, ld):
        # NaN everywhere but the [rows, cols] corner, one more row included
        flat = torch.full(((rows + 1) * ld,), float("nan"), device="cuda", dtype=dtype)
        v = flat.as_strided((rows, cols), (ld, 1))
        v.copy_(torch.randn(rows, cols, generator=g, device="cuda").to(dtype))
        return v
    a, b = padded(M, K, lda), padded(K, N, ldb)
    o = torch.full((BM, BN), float("nan"), device="cuda")
    print(f"masked copy {M}x{N}x{K} ld {lda},{ldb} tile {BM}x{BN}x{BK} other={other}", flush=True)
    masked_k[(1,)](a, b, o, M, N, K, lda, ldb, OTHER=other, BM=BM, BN=BN, BK=BK, num_warps=waves,
                   num_stages=stages)
    A = torch.full((BM, -(-K // BK) * BK), other, device="cuda", dtype=torch.float64)
    A[:M, :K] = a.double()
    B = torch.zeros(A.shape[1], BN, device="cuda", dtype=torch.float64)
    B[:K, :N] = b.double()
    bound = (A.shape[1] + 2) * 2.0 ** -24 * (A.abs() @ B.abs()) + 1e-30
    assert bool(((o.double() - A @ B).abs() <= bound).all())


TILES = [(64, 64, 64, 4, 4), (128, 128, 32, 4, 3), (256, 256, 32, 4, 4), (256, 128, 32, 8, 2),
         (16, 32, 128, 4, 4)]


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (7, 24, 200), (63, 56, 648), (16, 32, 1024)])
def test_chunk_uniform_masks(tile, M, N, K):
    BM, BN, BK, waves, stages = tile
    M, N = min(M, BM), min(N, BN)
    case(M, N, K, K + 8, N + 16, BM, BN, BK, waves, stages)


@pytest.mark.parametrize("M,N,K,other", [(7, 21, 205, 0.0), (64, 61, 130, 0.0), (33, 24, 200, 1.5)])
def test_masks_that_split_a_chunk_or_fill_with_a_value(M, N, K, other):
    """16-byte aligned rows whose bounds fall inside a chunk, and a fill that
    zeros would get wrong (the last k-step multiplies it by B's zeros, the rows
    past M by B's values)."""
    case(M, N, K, (K + 15) // 8 * 8, (N + 15) // 8 * 8, 64, 64, 64, 4, 3, other=other)


@pytest.mark.parametrize("lda", [4_210_688, 4_300_800])
@pytest.mark.parametrize("M", [256, 201])
def test_masked_rows_near_two_gib(lda, M):
    """Lane offsets of a 256-row tile that end just below and above 2^31."""
    case(M, 64, 72, lda, 64, 256, 64, 32, 4, 3)


def test_fp32_masked_copies():
    case(50, 60, 100, 104, 64, 64, 64, 16, 4, 4, dtype=torch.float32)


@pytest.mark.parametrize("tile", [(64, 64, 64, 8, 2), (64, 64, 64, 4, 4), (128, 128, 32, 4, 3),
                                  (32, 64, 128, 4, 2)])
@pytest.mark.parametrize("lda,ldb", [(1033, 64), (1040, 65), (1033, 67)])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (13, 9, 65), (31, 63, 1032), (64, 64, 1024),
                                   (63, 7, 700), (64, 8, 832), (5, 15, 513)])
def test_odd_strides(tile, lda, ldb, M, N, K):
    """Rows of an odd stride: tiles loaded into registers several iterations
    ahead at their elements' alignment, whole, cut by the column bound after
    their first chunk (shifted into place) or inside it (element loads), over
    trip counts from none in the branch-free loop to several."""
    BM, BN, BK, waves, stages = tile
    case(min(M, BM), min(N, BN), K, lda, ldb, BM, BN, BK, waves, stages)


@pytest.mark.parametrize("N", [9, 60, 61, 62, 63])
def test_odd_strides_fp32(N):
    """32-bit elements: four to a chunk, bounds that cut one to three off."""
    case(61, N, 260, 261, 67, 64, 64, 16, 4, 4, dtype=torch.float32)
