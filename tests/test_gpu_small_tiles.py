"""Output tiles too small for the workgroup's waves: the waves left over split
k within each k-step and their shares are added after the loop. Each case is
held to the float64 oracle at half an ulp of the output type per element plus
the fp32 accumulation error, as a relative Frobenius norm: 2^-9 for bf16
(2^-9 / sqrt(3) rms of a uniform rounding error, with slack), 2^-12 for fp16,
1e-5 for fp32. Outputs start as NaN, so a tile written short shows."""

import pytest
import torch

import newt
import newt.language as nl

pytestmark = pytest.mark.gpu

BOUND = {torch.bfloat16: 2 ** -9, torch.float16: 2 ** -12, torch.float32: 1e-5}


def operands(M, N, K, ta, tb, dtype):
    g = torch.Generator(device="cuda").manual_seed(M + 3 * N + 7 * K)

    def rnd(*s):
        return (torch.randn(*s, generator=g, device="cuda") * K ** -0.5).to(dtype)
    return (rnd(K, M).t() if ta else rnd(M, K)), (rnd(N, K).t() if tb else rnd(K, N))


def check(M, N, K, ta, tb, dtype, cfg):
    from newt_amd import workloads as W
    a, b = operands(M, N, K, ta, tb, dtype)
    c = torch.full((M, N), float("nan"), device="cuda", dtype=dtype)
    print(f"small tile {M}x{N}x{K} ta={ta} tb={tb} {dtype} {cfg}", flush=True)
    if cfg is None:
        W.matmul(a, b, c)
    else:
        BM, BN, BK, nw, ns = cfg
        W.matmul(a, b, c, config=newt.Config({"BLOCK_M": BM, "BLOCK_N": BN, "BLOCK_K": BK},
                                             num_warps=nw, num_stages=ns))
    ref = a.double() @ b.double().contiguous()
    assert ((c.double() - ref).norm() / ref.norm()).item() <= BOUND[dtype]


@pytest.mark.parametrize("cfg", [(16, 16, 256, 4, 4), (16, 16, 512, 8, 3), (16, 32, 256, 4, 4),
                                 (16, 64, 128, 8, 4), (32, 32, 128, 8, 6), (32, 64, 128, 4, 4),
                                 (64, 64, 128, 8, 3), (16, 16, 64, 2, 2)])
@pytest.mark.parametrize("M,N,K", [(16, 256, 2048), (64, 64, 512), (17, 72, 1032), (1, 130, 264),
                                   (33, 31, 136)])
@pytest.mark.parametrize("tb", [True, False])
def test_waves_split_k(M, N, K, tb, cfg):
    check(M, N, K, False, tb, torch.bfloat16, cfg)


@pytest.mark.parametrize("cfg", [(64, 64, 32, 8, 3), (32, 64, 64, 4, 3), (64, 64, 64, 16, 2)])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)])
@pytest.mark.parametrize("M,N,K", [(128, 64, 256), (65, 60, 100)])
def test_waves_split_k_fp32(M, N, K, ta, tb, cfg):
    check(M, N, K, ta, tb, torch.float32, cfg)


@pytest.mark.parametrize("dtype,cfg", [
    (torch.float16, (64, 64, 64, 8, 3)), (torch.bfloat16, (64, 128, 32, 16, 3)),
    (torch.bfloat16, (64, 128, 64, 16, 2)), (torch.float32, (32, 64, 64, 8, 4)),
    (torch.float32, (64, 64, 32, 8, 4)), (torch.float32, (32, 64, 32, 4, 2))])
@pytest.mark.parametrize("M,N,K", [(128, 128, 512), (70, 131, 1033)])
def test_shares_joined_in_parts(M, N, K, dtype, cfg):
    """Shares of more than one stage's LDS, and of less than one part each."""
    check(M, N, K, False, False, dtype, cfg)


@pytest.mark.parametrize("M,N,K", [(16, 1024, 1024), (1, 512, 768), (100, 1000, 520),
                                   (960, 1024, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_few_tiles_are_tuned_over_small_tiles(M, N, K, dtype):
    from newt_amd import workloads as W
    check(M, N, K, False, True, dtype, None)
    assert any(key[:3] == (M, N, K) for key in W.matmul_tuned_small.timings)


@pytest.mark.parametrize("M,N,K", [(16, 512, 512), (1, 64, 96), (300, 129, 77), (1000, 1024, 40)])
@pytest.mark.parametrize("tb", [True, False])
def test_few_fp32_tiles_are_tuned_over_small_tiles(M, N, K, tb):
    from newt_amd import workloads as W
    check(M, N, K, False, tb, torch.float32, None)
    assert any(key[:3] == (M, N, K) for key in W.matmul_tuned_fp32_small.timings)


@newt.jit
def init_and_two_loops_k(a_ptr, b_ptr, o_ptr, K, FULL, REST, INIT: nl.constexpr,
                         BM: nl.constexpr, BN: nl.constexpr, BK: nl.constexpr):
    rm, rn, rk = nl.arange(0, BM), nl.arange(0, BN), nl.arange(0, BK)
    pa = a_ptr + rm[:, None] * K + rk[None, :]
    pb = b_ptr + rn[None, :] * K + rk[:, None]
    acc = nl.full((BM, BN), INIT, dtype=nl.float32)
    for i in range(FULL):
        a = nl.load(pa)
        b = nl.load(pb)
        acc = nl.dot(a, b, acc)
        pa += BK
        pb += BK
    for j in range(REST):
        a2 = nl.load(pa)
        b2 = nl.load(pb)
        acc = nl.dot(a2, b2, acc)
        pa += BK
        pb += BK
    nl.store(o_ptr + rm[:, None] * BN + rn[None, :], acc)


@pytest.mark.parametrize("full,rest", [(0, 0), (0, 1), (5, 0), (4, 7)])
@pytest.mark.parametrize("waves", [1, 4, 8])
def test_initial_accumulator_counts_once(full, rest, waves):
    """A nonzero initial accumulator and two loops on it (zero trips included):
    each group's share starts from zero but the first's."""
    BM = BN = 16
    BK = 256
    K = (full + rest) * BK
    g = torch.Generator(device="cuda").manual_seed(1)
    a = torch.randn(BM, max(K, 1), generator=g, device="cuda").half()
    b = torch.randn(BN, max(K, 1), generator=g, device="cuda").half()
    o = torch.full((BM, BN), float("nan"), device="cuda")
    init_and_two_loops_k[(1,)](a, b, o, K, full, rest, INIT=3.0, BM=BM, BN=BN, BK=BK,
                               num_warps=waves, num_stages=3)
    want = 3.0 + a[:, :K].double() @ b[:, :K].double().t().contiguous()
    # fp32 sums of K products: error at most K * 2^-24 of the sum of magnitudes
    mags = 3.0 + a[:, :K].double().abs() @ b[:, :K].double().abs().t().contiguous()
    assert bool(((o.double() - want).abs() <= (K + 2) * 2.0 ** -24 * mags).all())
