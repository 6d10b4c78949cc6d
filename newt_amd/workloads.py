"""The five hot-path workloads written in the newt DSL, with host wrappers.

These are user-level kernels exactly as a newt user writes them (the
reference's examples/01-05), extended to the benchmark configurations:
  add_kernel        examples/01_vector_add.py:14-21 (unchanged)
  copy_kernel       no reference counterpart: a streaming copy that measures
                    the HBM ceiling of a kernel compiled by newt (bench.py)
  softmax_kernel    examples/02_fused_softmax.py:15-24 (unchanged)
  layernorm_kernel  examples/03_layernorm.py:13-27 + stores of the saved
                    per-row mean / rstd (config 3 asks for them)
  matmul_kernel     examples/04_matmul.py:14-45 (unchanged body), autotuned over
                    a configuration space re-derived for gfx950
  attention_kernel  examples/05_fused_attention.py:14-48 generalised to
                    [batch, heads, seq, head_dim] with a batch*head grid axis,
                    strides, an optional causal mask with the loop bound trimmed
                    to the diagonal, p cast to V's dtype before P @ V, and the
                    softmax written on exp2 with log2(e) folded into the scale
                    (exp(x) = exp2(x*log2 e): the same softmax, fewer
                    instructions per element), the exponents referred to each
                    row's first-block maximum (no rescale in the main loops;
                    an online-softmax pass for a program where some row's sum
                    passes 2^80 or the accumulator overflows); launched with
                    waves_per_eu=2 so two waves share each SIMD and one
                    wave's softmax runs while the other's MFMAs do
  attention_plain_kernel
                    examples/05_fused_attention.py:14-48 as written there
                    (nl.exp, qk * scale, a where mask), generalised only by the
                    batch*head axis and the causal mask; also the kernel for a
                    scale <= 0
  dt_matmul         examples/deuteron/01_matmul.py (unchanged body): the tile
                    DSL traced to newt and autotuned against its eager oracle
Everything is compiled by newt_amd's compiler to HIP for gfx950.
"""

import functools

import torch

import newt_amd as newt
import newt_amd.language as nl


# ---------------------------------------------------------------------------
# 1. vector add
# ---------------------------------------------------------------------------
@newt.jit
def add_kernel(x_ptr, y_ptr, out_ptr, n, BLOCK: nl.constexpr):
    pid = nl.program_id(0)
    offs = pid * BLOCK + nl.arange(0, BLOCK)
    mask = offs < n
    x = nl.load(x_ptr + offs, mask=mask)
    y = nl.load(y_ptr + offs, mask=mask)
    nl.store(out_ptr + offs, x + y, mask=mask)


def add(x, y, out=None, BLOCK=1024, num_warps=4):
    out = torch.empty_like(x) if out is None else out
    n = x.numel()
    add_kernel[(newt.cdiv(n, BLOCK),)](x, y, out, n, BLOCK=BLOCK, num_warps=num_warps)
    return out


@newt.jit
def copy_kernel(src_ptr, dst_ptr, n, BLOCK: nl.constexpr):
    # a one-read-one-write stream: the HBM ceiling any kernel compiled by
    # newt that reads and writes its bytes once can reach at a given size
    offs = nl.program_id(0) * BLOCK + nl.arange(0, BLOCK)
    mask = offs < n
    nl.store(dst_ptr + offs, nl.load(src_ptr + offs, mask=mask), mask=mask)


def copy(src, dst, BLOCK=2048, num_warps=4):
    # 8 fp32 per thread (two 16-byte loads): the fastest shape measured at
    # 128 MiB and 256 MiB moved (BLOCK 1024-16384, 4-16 waves)
    n = src.numel()
    copy_kernel[(newt.cdiv(n, BLOCK),)](src, dst, n, BLOCK=BLOCK, num_warps=num_warps)
    return dst


# ---------------------------------------------------------------------------
# 2. fused row softmax
# ---------------------------------------------------------------------------
@newt.jit
def softmax_kernel(x_ptr, out_ptr, N, stride, BLOCK_N: nl.constexpr):
    row = nl.program_id(0)
    cols = nl.arange(0, BLOCK_N)
    mask = cols < N
    x = nl.load(x_ptr + row * stride + cols, mask=mask, other=float("-inf"))
    x = x - nl.max(x, axis=0)
    num = nl.exp(x)
    den = nl.sum(num, axis=0)
    nl.store(out_ptr + row * stride + cols, num / den, mask=mask)


def softmax_warps(block_n):
    # one row per workgroup, 16 fp32 values (four 16-byte loads) per thread:
    # enough bytes in flight per wave, and several rows per CU to overlap one
    # row's reductions with another's loads (measured best at 1000..8192 cols)
    return max(2, min(16, block_n // 1024))


@newt.jit
def softmax_rows_kernel(x_ptr, out_ptr, M, N, stride, ROWS: nl.constexpr,
                        BLOCK_N: nl.constexpr):
    # softmax_kernel over ROWS short rows at a time
    rows = nl.program_id(0) * ROWS + nl.arange(0, ROWS)
    cols = nl.arange(0, BLOCK_N)
    mask = (rows[:, None] < M) & (cols[None, :] < N)
    offs = rows[:, None] * stride + cols[None, :]
    x = nl.load(x_ptr + offs, mask=mask, other=float("-inf"))
    x = x - nl.max(x, axis=1)[:, None]
    num = nl.exp(x)
    den = nl.sum(num, axis=1)
    nl.store(out_ptr + offs, num / den[:, None], mask=mask)


def rows_per_program(block_n, itemsize):
    """Rows of a 4-wave program for rows that fit one 16-byte access of a
    wave's lanes (256 fp32 or 512 16-bit columns), 0 for longer or tinier ones
    (less than one access). A row per program leaves most of its lanes idle
    and a launch is bound by the rate at which workgroups start; with as many
    rows as four waves hold, each row's reductions stay within a wave and the
    lanes are full. Against a row per program: softmax fp32 32768x64 9.8 ->
    3.9 us, 32768x128 10.8 -> 5.9 (16.8 MB read and written: 5.7 at the copy's
    rate), 32768x250 16.0 -> 12.3; layernorm fp16 32768x64 13.3 -> 3.2,
    32768x128 13.9 -> 4.5, 8192x500 7.9 -> 6.0, bf16 32768x512 15.8 -> 13.0.
    At 512 fp32 columns (two accesses a lane) both forms are level."""
    if not 16 <= block_n * itemsize <= 1024:
        return 0
    return 4 * 1024 // (block_n * itemsize)


def softmax(x, out=None, num_warps=None):
    M, N = x.shape
    out = torch.empty_like(x) if out is None else out
    BLOCK_N = newt.next_power_of_2(N)
    rows = 0 if num_warps or BLOCK_N > 512 else rows_per_program(BLOCK_N, x.element_size())
    if rows:
        softmax_rows_kernel[(newt.cdiv(M, rows),)](x, out, M, N, x.stride(0), ROWS=rows,
                                                   BLOCK_N=BLOCK_N, num_warps=4)
        return out
    nw = num_warps or softmax_warps(BLOCK_N)
    softmax_kernel[(M,)](x, out, N, x.stride(0), BLOCK_N=BLOCK_N, num_warps=nw)
    return out


# ---------------------------------------------------------------------------
# 3. layernorm forward (+ saved mean / rstd)
# ---------------------------------------------------------------------------
@newt.jit
def layernorm_kernel(x_ptr, w_ptr, b_ptr, out_ptr, mean_ptr, rstd_ptr, N, stride, eps,
                     BLOCK_N: nl.constexpr):
    row = nl.program_id(0)
    cols = nl.arange(0, BLOCK_N)
    mask = cols < N
    x = nl.load(x_ptr + row * stride + cols, mask=mask, other=0.0)
    mean = nl.sum(x, axis=0) / N
    diff = nl.where(mask, x - mean, 0.0)
    var = nl.sum(diff * diff, axis=0) / N
    rstd = nl.rsqrt(var + eps)
    w = nl.load(w_ptr + cols, mask=mask)
    b = nl.load(b_ptr + cols, mask=mask)
    y = (x - mean) * rstd * w + b
    nl.store(out_ptr + row * stride + cols, y, mask=mask)
    nl.store(mean_ptr + row, mean)
    nl.store(rstd_ptr + row, rstd)


@newt.jit
def layernorm_rows_kernel(x_ptr, w_ptr, b_ptr, out_ptr, mean_ptr, rstd_ptr, M, N, stride, eps,
                          ROWS: nl.constexpr, BLOCK_N: nl.constexpr):
    # layernorm_kernel over ROWS short rows at a time
    rows = nl.program_id(0) * ROWS + nl.arange(0, ROWS)
    cols = nl.arange(0, BLOCK_N)
    in_row = cols[None, :] < N
    mask = (rows[:, None] < M) & in_row
    offs = rows[:, None] * stride + cols[None, :]
    x = nl.load(x_ptr + offs, mask=mask, other=0.0)
    mean = nl.sum(x, axis=1) / N
    diff = nl.where(in_row, x - mean[:, None], 0.0)
    var = nl.sum(diff * diff, axis=1) / N
    rstd = nl.rsqrt(var + eps)
    w = nl.load(w_ptr + cols, mask=cols < N)
    b = nl.load(b_ptr + cols, mask=cols < N)
    y = (x - mean[:, None]) * rstd[:, None] * w[None, :] + b[None, :]
    nl.store(out_ptr + offs, y, mask=mask)
    nl.store(mean_ptr + rows, mean, mask=rows < M)
    nl.store(rstd_ptr + rows, rstd, mask=rows < M)


def layernorm(x, w, b, eps=1e-5, out=None, num_warps=None):
    M, N = x.shape
    out = torch.empty_like(x) if out is None else out
    mean = torch.empty(M, device=x.device, dtype=torch.float32)
    rstd = torch.empty(M, device=x.device, dtype=torch.float32)
    BLOCK_N = newt.next_power_of_2(N)
    rows = 0 if num_warps or BLOCK_N > 512 else rows_per_program(BLOCK_N, x.element_size())
    if rows:
        layernorm_rows_kernel[(newt.cdiv(M, rows),)](x, w, b, out, mean, rstd, M, N, x.stride(0),
                                                     eps, ROWS=rows, BLOCK_N=BLOCK_N, num_warps=4)
        return out, mean, rstd
    # 16 fp16 elements (two 16-byte loads) per thread: a 8192-wide row on 8
    # waves measured ~2% faster than on 4 (fewer registers per wave, and the
    # same bytes in flight per CU); 16 waves per row were 20% slower
    nw = num_warps or max(2, min(8, BLOCK_N // 1024))
    layernorm_kernel[(M,)](x, w, b, out, mean, rstd, N, x.stride(0), eps,
                           BLOCK_N=BLOCK_N, num_warps=nw)
    return out, mean, rstd


# ---------------------------------------------------------------------------
# 4. matmul (fp16 / bf16, fp32 accumulate)
# ---------------------------------------------------------------------------
@newt.jit
def matmul_kernel(a_ptr, b_ptr, c_ptr, M, N, K,
                  sam, sak, sbk, sbn, scm, scn,
                  BLOCK_M: nl.constexpr, BLOCK_N: nl.constexpr, BLOCK_K: nl.constexpr):
    pid_m = nl.program_id(0)
    pid_n = nl.program_id(1)
    offs_m = pid_m * BLOCK_M + nl.arange(0, BLOCK_M)
    offs_n = pid_n * BLOCK_N + nl.arange(0, BLOCK_N)
    offs_k = nl.arange(0, BLOCK_K)
    a_ptrs = a_ptr + offs_m[:, None] * sam + offs_k[None, :] * sak
    b_ptrs = b_ptr + offs_k[:, None] * sbk + offs_n[None, :] * sbn
    acc = nl.zeros((BLOCK_M, BLOCK_N), dtype=nl.float32)
    for k in range(nl.cdiv(K, BLOCK_K)):
        a_mask = (offs_m[:, None] < M) & (offs_k[None, :] < K - k * BLOCK_K)
        b_mask = (offs_k[:, None] < K - k * BLOCK_K) & (offs_n[None, :] < N)
        a = nl.load(a_ptrs, mask=a_mask, other=0.0)
        b = nl.load(b_ptrs, mask=b_mask, other=0.0)
        acc = nl.dot(a, b, acc)
        a_ptrs += BLOCK_K * sak
        b_ptrs += BLOCK_K * sbk
    c_ptrs = c_ptr + offs_m[:, None] * scm + offs_n[None, :] * scn
    c_mask = (offs_m[:, None] < M) & (offs_n[None, :] < N)
    nl.store(c_ptrs, acc.to(c_ptr.dtype.element_ty), mask=c_mask)


def operand_layout(sam, sak, sbk, sbn):
    """What of the operands' strides decides which tiles serve them, as a part
    of the tuning key: which dim has unit stride and whether the other keeps
    16-byte rows. One shape in two layouts (x @ w.t() and then dy @ w of a
    square weight, or an odd row stride) has different best tiles: the best of
    bf16 x[16,4096] @ w.t(), 16x16x512 at 6.7 us, takes 18.5 on w itself, where
    16x32x128 takes 11.4; of fp32 512^3, 32x32x64 at 5.9, takes 17.3, where
    32x64x32 takes 7.3."""
    # per stride: 1, a multiple of 8 elements (0) or any other (2)
    return (sam if sam == 1 else sam % 8 and 2, sak if sak == 1 else sak % 8 and 2,
            sbk if sbk == 1 else sbk % 8 and 2, sbn if sbn == 1 else sbn % 8 and 2)


MATMUL_KEY = ["M", "N", "K", operand_layout]


# gfx950 search space: 64-wide waves, 160 KB LDS per CU, 256 CUs. The k-loop is
# software-pipelined num_stages deep through distinct LDS stages, so tiles of
# 256x256 with BLOCK_K=32 and 4 stages (128 KB) give each CU one workgroup:
# 4 waves with a 128x128 MFMA sub-tile each (accumulators in AGPRs; half the
# LDS operand reads per flop of 8 waves) or 8 waves with 128x64; smaller tiles
# keep grids of >= 256 workgroups for smaller problems.
MATMUL_CONFIGS = [
    newt.Config({"BLOCK_M": 256, "BLOCK_N": 256, "BLOCK_K": 32}, num_warps=4, num_stages=4),
    newt.Config({"BLOCK_M": 256, "BLOCK_N": 256, "BLOCK_K": 32}, num_warps=8, num_stages=4),
    newt.Config({"BLOCK_M": 256, "BLOCK_N": 256, "BLOCK_K": 64}, num_warps=8, num_stages=2),
    newt.Config({"BLOCK_M": 256, "BLOCK_N": 256, "BLOCK_K": 32}, num_warps=8, num_stages=3),
    newt.Config({"BLOCK_M": 256, "BLOCK_N": 128, "BLOCK_K": 32}, num_warps=8, num_stages=4),
    newt.Config({"BLOCK_M": 128, "BLOCK_N": 256, "BLOCK_K": 32}, num_warps=8, num_stages=4),
    newt.Config({"BLOCK_M": 128, "BLOCK_N": 128, "BLOCK_K": 64}, num_warps=4, num_stages=3),
    # 2048^3 (one 128x128 tile per CU): 64-deep k-steps with 4 stages (128 KB)
    # measured 813 against 799 TFLOP/s for the 32-deep tile below
    newt.Config({"BLOCK_M": 128, "BLOCK_N": 128, "BLOCK_K": 64}, num_warps=4, num_stages=4),
    newt.Config({"BLOCK_M": 128, "BLOCK_N": 128, "BLOCK_K": 32}, num_warps=4, num_stages=4),
    newt.Config({"BLOCK_M": 64, "BLOCK_N": 128, "BLOCK_K": 64}, num_warps=4, num_stages=3),
    # 64x64 tiles give a 1024^3 problem 256 workgroups (one per CU)
    newt.Config({"BLOCK_M": 64, "BLOCK_N": 64, "BLOCK_K": 64}, num_warps=4, num_stages=4),
    # (64x64x64 on 4 waves with 3 stages left this list: of eight products from
    # 1024x1024x256 to 256x4096x4096 in four layouts each it was ahead of the
    # others in one, odd rows of the latter, 25.3 against 26.1 us.
    # 64x64x128 with 4 stages stays out: with flushed caches, as
    # the tuner times, it wins at 1024^3, where it then runs 7.0 us back to back
    # against 6.0 for the tile above; it gained 9% at 256x4096x4096)
    # two waves per SIMD over a 64x128 tile: bf16 640x2048x2048 (320 such
    # tiles) 12.7 us against 15.1 for 64x64x64 and 15.5 for 128x128x64
    newt.Config({"BLOCK_M": 64, "BLOCK_N": 128, "BLOCK_K": 64}, num_warps=8, num_stages=4),
    # odd strides: tiles that go through registers want few bytes per wave
    # (fp16 2048x2047x2049 32.6 us against 37.1 on 4 waves and 48.6 on 64x64
    # tiles; 1000x1003x777 10.2 against 11.8 on 4 waves)
    newt.Config({"BLOCK_M": 128, "BLOCK_N": 128, "BLOCK_K": 32}, num_warps=8, num_stages=4),
    newt.Config({"BLOCK_M": 64, "BLOCK_N": 64, "BLOCK_K": 64}, num_warps=8, num_stages=3),
]

matmul_tuned = newt.autotune(configs=MATMUL_CONFIGS, key=MATMUL_KEY)(matmul_kernel)

# Products whose 64x64 tiles do not fill the 256 CUs (few rows, few columns or
# small all round) are bound by the bytes that the launch keeps in flight, not
# by MFMAs: a 16-row product reads its long operand once. These tiles are
# small enough for a workgroup per CU, their k-steps deep enough that each CU
# keeps 50-100 KB of copies in flight, and waves that a tile has no rows or
# columns for split k (DotPipeline._join_ksplit). bf16, back to back, against
# the fastest of MATMUL_CONFIGS: x[16,4096] @ w[4096,4096].t() 7.9 against
# 58 us (34 MB: 4.3 TB/s), 64 rows 9.3, 128 rows 12.5; w not transposed 12.1,
# 12.2, 13.9; [32,8192] @ [8192,1024] 8.1 transposed, 18.3 not; 256x256x1024
# 3.6 and 512x1024x1024 5.1 (5.6). 16-wide column tiles serve only a
# transposed w (a tile of whole 16-byte runs along k); from 256 64x64 tiles on
# (256x4096x4096, 1024^3) none of these wins.
MATMUL_CONFIGS_SMALL = [
    newt.Config({"BLOCK_M": 16, "BLOCK_N": 16, "BLOCK_K": 256}, num_warps=4, num_stages=4),
    newt.Config({"BLOCK_M": 16, "BLOCK_N": 16, "BLOCK_K": 512}, num_warps=4, num_stages=4),
    newt.Config({"BLOCK_M": 16, "BLOCK_N": 32, "BLOCK_K": 256}, num_warps=4, num_stages=4),
    newt.Config({"BLOCK_M": 16, "BLOCK_N": 32, "BLOCK_K": 128}, num_warps=4, num_stages=6),
    newt.Config({"BLOCK_M": 16, "BLOCK_N": 64, "BLOCK_K": 128}, num_warps=4, num_stages=4),
    newt.Config({"BLOCK_M": 32, "BLOCK_N": 32, "BLOCK_K": 128}, num_warps=4, num_stages=4),
    newt.Config({"BLOCK_M": 32, "BLOCK_N": 32, "BLOCK_K": 128}, num_warps=4, num_stages=6),
    newt.Config({"BLOCK_M": 32, "BLOCK_N": 64, "BLOCK_K": 128}, num_warps=4, num_stages=4),
    newt.Config({"BLOCK_M": 64, "BLOCK_N": 32, "BLOCK_K": 128}, num_warps=4, num_stages=4),
    newt.Config({"BLOCK_M": 64, "BLOCK_N": 64, "BLOCK_K": 64}, num_warps=4, num_stages=4),
    newt.Config({"BLOCK_M": 64, "BLOCK_N": 64, "BLOCK_K": 128}, num_warps=4, num_stages=4),
    newt.Config({"BLOCK_M": 64, "BLOCK_N": 32, "BLOCK_K": 64}, num_warps=4, num_stages=4),
    newt.Config({"BLOCK_M": 64, "BLOCK_N": 64, "BLOCK_K": 64}, num_warps=8, num_stages=3),
]
matmul_tuned_small = newt.autotune(configs=MATMUL_CONFIGS_SMALL, key=MATMUL_KEY)(matmul_kernel)

# fp32 operands run on the fp32 MFMA (v_mfma_f32_32x32x2_f32, full precision;
# gfx950 has no tf32) through the same pipelined k-loop: 16-deep k-steps keep
# 3-4 fp32 stages within the LDS
MATMUL_CONFIGS_FP32 = [
    newt.Config({"BLOCK_M": 256, "BLOCK_N": 256, "BLOCK_K": 16}, num_warps=8, num_stages=3),
    newt.Config({"BLOCK_M": 256, "BLOCK_N": 128, "BLOCK_K": 16}, num_warps=8, num_stages=4),
    newt.Config({"BLOCK_M": 128, "BLOCK_N": 128, "BLOCK_K": 32}, num_warps=4, num_stages=3),
    newt.Config({"BLOCK_M": 128, "BLOCK_N": 128, "BLOCK_K": 16}, num_warps=4, num_stages=4),
    # two waves per SIMD: 2048^3 118.4 against 119.9 us for the tile above
    newt.Config({"BLOCK_M": 128, "BLOCK_N": 128, "BLOCK_K": 32}, num_warps=8, num_stages=3),
]
matmul_tuned_fp32 = newt.autotune(configs=MATMUL_CONFIGS_FP32, key=MATMUL_KEY)(matmul_kernel)

# fp32 products whose 128x128 tiles do not fill the 256 CUs: the fp32 MFMA is
# slow enough (64 cycles for 32x32x2) that a launch takes as long as its
# busiest CU has MFMAs, so the tile is what divides the work most evenly.
# 1024^3 (64 tiles of 128x128) 61.7 -> 18.6 us on 64x64x32, of 13.7 us of MFMA
# work per CU; 512^3 7.3, x @ w.t() 5.9; [16,4096] @ [4096,4096] 33.2, x @ w.t()
# 19.5 (67 MB; 32x32 tiles serve a transposed w only); 1500x700x1003 33.3.
# From 256 tiles of 128x128 on (2048^3) the larger list is level or ahead.
MATMUL_CONFIGS_FP32_SMALL = [
    newt.Config({"BLOCK_M": 32, "BLOCK_N": 32, "BLOCK_K": 64}, num_warps=4, num_stages=4),
    newt.Config({"BLOCK_M": 32, "BLOCK_N": 64, "BLOCK_K": 32}, num_warps=4, num_stages=4),
    newt.Config({"BLOCK_M": 32, "BLOCK_N": 64, "BLOCK_K": 64}, num_warps=8, num_stages=4),
    newt.Config({"BLOCK_M": 64, "BLOCK_N": 64, "BLOCK_K": 32}, num_warps=4, num_stages=4),
    newt.Config({"BLOCK_M": 64, "BLOCK_N": 64, "BLOCK_K": 32}, num_warps=8, num_stages=4),
    newt.Config({"BLOCK_M": 64, "BLOCK_N": 128, "BLOCK_K": 32}, num_warps=8, num_stages=4),
    newt.Config({"BLOCK_M": 128, "BLOCK_N": 128, "BLOCK_K": 32}, num_warps=8, num_stages=3),
]
matmul_tuned_fp32_small = newt.autotune(configs=MATMUL_CONFIGS_FP32_SMALL,
                                        key=MATMUL_KEY)(matmul_kernel)


def matmul(a, b, c=None, config=None):
    M, K = a.shape
    K2, N = b.shape
    assert K == K2
    c = torch.empty(M, N, device=a.device, dtype=a.dtype) if c is None else c
    args = (a, b, c, M, N, K, *a.stride(), *b.stride(), *c.stride())
    if config is None:
        grid = lambda meta: (newt.cdiv(M, meta["BLOCK_M"]), newt.cdiv(N, meta["BLOCK_N"]))
        if a.dtype == torch.float32:
            few = newt.cdiv(M, 128) * newt.cdiv(N, 128) < 256
            tuned = matmul_tuned_fp32_small if few else matmul_tuned_fp32
        elif newt.cdiv(M, 64) * newt.cdiv(N, 64) < 256:
            tuned = matmul_tuned_small
        else:
            tuned = matmul_tuned
        tuned[grid](*args)
    else:
        grid = (newt.cdiv(M, config.kwargs["BLOCK_M"]), newt.cdiv(N, config.kwargs["BLOCK_N"]))
        matmul_kernel[grid](*args, **config.kwargs, num_warps=config.num_warps,
                            num_stages=config.num_stages)
    return c


# ---------------------------------------------------------------------------
# 5. flash attention forward
# ---------------------------------------------------------------------------
@newt.jit
def attention_kernel(q_ptr, k_ptr, v_ptr, o_ptr, S, H, scale,
                     sqb, sqh, sqm, skb, skh, skn, svb, svh, svn, sob, soh, som,
                     BLOCK_M: nl.constexpr, BLOCK_N: nl.constexpr, D: nl.constexpr,
                     CAUSAL: nl.constexpr):
    pid = nl.program_id(0)
    bh = nl.program_id(1)
    if CAUSAL:
        # Query block i does i + 1 key blocks: each XCD should start its
        # heaviest programs first, so that the last to start are short ones
        # (longest-processing-time-first order, a short tail). Program ids
        # arrive renumbered so that each XCD runs one contiguous range of
        # lin = pid + nqb * bh in increasing order; when the heads split evenly
        # over the 8 XCDs that range is gh whole heads, which it would run one
        # after another, heaviest to lightest within each. The range is taken
        # in groups of grp = 4 heads (all gh when 4 does not divide gh), and
        # within a group its r-th program becomes weight rank r // grp of head
        # r % grp: every head's heaviest block, then every head's next, and so
        # on, with four heads' keys and values in the XCD's L2 at a time. (Any
        # bijection of the programs computes the same result.)
        nqb = nl.num_programs(0)
        nbh = nl.num_programs(1)
        if nbh % 8 == 0:
            gh = nbh // 8
            grp = gh
            if gh % 4 == 0:
                grp = 4
            lin = pid + nqb * bh
            r = lin % (gh * nqb)
            rr = r % (grp * nqb)
            bh = lin // (gh * nqb) * gh + r // (grp * nqb) * grp + rr % grp
            pid = rr // grp
        pid = nqb - 1 - pid
    bi = bh // H
    hi = bh % H
    q_base = q_ptr + bi * sqb + hi * sqh
    k_base = k_ptr + bi * skb + hi * skh
    v_base = v_ptr + bi * svb + hi * svh
    o_base = o_ptr + bi * sob + hi * soh
    offs_m = pid * BLOCK_M + nl.arange(0, BLOCK_M)
    offs_d = nl.arange(0, D)
    qmask = offs_m[:, None] < S
    q = nl.load(q_base + offs_m[:, None] * sqm + offs_d[None, :], mask=qmask, other=0.0)

    qk_scale = scale * 1.4426950408889634  # log2(e): the softmax runs on exp2
    # The exponents share one reference point per row, m_i: the row's maximum
    # over the first key block, fixed for the rest of the row. O = acc / l_i
    # is the same quotient whatever reference point the exponents share, so
    # the loops never rescale acc: p = exp2(qk * s - m_i) only grows past 1
    # where a later score exceeds the first block's maximum. While every p
    # stays below 2^80, l_i stays far inside fp32's range; a row whose sum l_i
    # passes 2^80 (some score 80 or more above that maximum, in log2 units),
    # or an acc that overflowed, sends the program through the online-softmax
    # loop at the end, which rescales at every block. (A rescale inside the
    # main loops costs a cross-wave maximum, a barrier and a branch per key
    # block.)
    m_i = nl.zeros((BLOCK_M,), dtype=nl.float32)
    l_i = nl.zeros((BLOCK_M,), dtype=nl.float32)
    acc = nl.zeros((BLOCK_M, D), dtype=nl.float32)

    # key blocks wholly inside the sequence (and, causal, wholly below the
    # diagonal of every row of this program) need no mask; the ragged tail and
    # the diagonal blocks run in a second, masked loop. Scores stay unscaled:
    # the scale is applied inside the exponent's fma, and the reference is
    # max(qk) * qk_scale (= max(qk * qk_scale): rounding is monotonic).
    full_n = S // BLOCK_N * BLOCK_N
    end_n = S
    if CAUSAL:
        full_n = nl.minimum(full_n, pid * BLOCK_M // BLOCK_N * BLOCK_N)
        end_n = nl.minimum(S, (pid + 1) * BLOCK_M)
    for start_n in range(0, full_n, BLOCK_N):
        offs_n = start_n + nl.arange(0, BLOCK_N)
        k = nl.load(k_base + offs_n[:, None] * skn + offs_d[None, :])
        qk = nl.dot(q, nl.trans(k))
        if start_n == 0:
            m_i = nl.max(qk, axis=1) * qk_scale
        p = nl.exp2(nl.fma(qk, qk_scale, -m_i[:, None]))
        l_i = l_i + nl.sum(p, axis=1)
        v = nl.load(v_base + offs_n[:, None] * svn + offs_d[None, :])
        acc = nl.dot(p.to(v_ptr.dtype.element_ty), v, acc)
    for start_n in range(full_n, end_n, BLOCK_N):
        offs_n = start_n + nl.arange(0, BLOCK_N)
        nmask = offs_n[:, None] < S
        k = nl.load(k_base + offs_n[:, None] * skn + offs_d[None, :], mask=nmask, other=0.0)
        qk = nl.dot(q, nl.trans(k))
        if CAUSAL:
            qk = nl.where((offs_m[:, None] >= offs_n[None, :]) & (offs_n[None, :] < S),
                          qk, float("-inf"))
        else:
            qk = nl.where(offs_n[None, :] < S, qk, float("-inf"))
        # the first key block has key 0 in it, which no row masks: every row's
        # reference is finite (masked scores are -inf, p = exp2(-inf) = 0)
        if start_n == 0:
            m_i = nl.max(qk, axis=1) * qk_scale
        p = nl.exp2(nl.fma(qk, qk_scale, -m_i[:, None]))
        l_i = l_i + nl.sum(p, axis=1)
        v = nl.load(v_base + offs_n[:, None] * svn + offs_d[None, :], mask=nmask, other=0.0)
        acc = nl.dot(p.to(v_ptr.dtype.element_ty), v, acc)

    # acc <= l_i * max|v|: past the first block's maximum, p grows acc by up
    # to 2^80 more than the per-block rescale's p <= 1 does, so for values
    # above ~2^48 acc can overflow where the rescaled sum stays finite.
    # acc * 0 is NaN exactly where acc holds an inf or NaN (no fast-math:
    # the product is not folded), which makes `peak` NaN and sends the
    # program through the rescaling pass too.
    peak = nl.max(l_i) + nl.sum(acc * 0.0)
    if not (peak <= 1.2089258196146292e24):  # 2^80: start again with a rescale per block
        m_i = nl.full((BLOCK_M,), float("-inf"), dtype=nl.float32)
        l_i = nl.zeros((BLOCK_M,), dtype=nl.float32)
        acc = nl.zeros((BLOCK_M, D), dtype=nl.float32)
        for start_n in range(0, end_n, BLOCK_N):
            offs_n = start_n + nl.arange(0, BLOCK_N)
            nmask = offs_n[:, None] < S
            k = nl.load(k_base + offs_n[:, None] * skn + offs_d[None, :], mask=nmask, other=0.0)
            qk = nl.dot(q, nl.trans(k))
            if CAUSAL:
                qk = nl.where((offs_m[:, None] >= offs_n[None, :]) & (offs_n[None, :] < S),
                              qk, float("-inf"))
            else:
                qk = nl.where(offs_n[None, :] < S, qk, float("-inf"))
            m_new = nl.maximum(m_i, nl.max(qk, axis=1) * qk_scale)
            alpha = nl.exp2(m_i - m_new)
            p = nl.exp2(nl.fma(qk, qk_scale, -m_new[:, None]))
            l_i = l_i * alpha + nl.sum(p, axis=1)
            acc = acc * alpha[:, None]
            v = nl.load(v_base + offs_n[:, None] * svn + offs_d[None, :], mask=nmask, other=0.0)
            acc = nl.dot(p.to(v_ptr.dtype.element_ty), v, acc)
            m_i = m_new

    # one reciprocal per row and a multiply per element instead of a division
    # per element (an IEEE fp32 division is ~10 instructions); the two differ
    # by at most an ulp of fp32, far below the bf16 rounding of the output
    acc = acc * (1.0 / l_i)[:, None]
    nl.store(o_base + offs_m[:, None] * som + offs_d[None, :], acc.to(o_ptr.dtype.element_ty),
             mask=qmask)


@newt.jit
def attention_plain_kernel(q_ptr, k_ptr, v_ptr, o_ptr, S, H, scale,
                           sqb, sqh, sqm, skb, skh, skn, svb, svh, svn, sob, soh, som,
                           BLOCK_M: nl.constexpr, BLOCK_N: nl.constexpr, D: nl.constexpr,
                           CAUSAL: nl.constexpr):
    # examples/05_fused_attention.py:14-48 as written there (one key loop,
    # nl.exp, qk * scale, a where mask, p cast to V's dtype), generalised only
    # by the batch*head grid axis and the causal mask with its loop bound
    pid = nl.program_id(0)
    bh = nl.program_id(1)
    bi = bh // H
    hi = bh % H
    q_base = q_ptr + bi * sqb + hi * sqh
    k_base = k_ptr + bi * skb + hi * skh
    v_base = v_ptr + bi * svb + hi * svh
    o_base = o_ptr + bi * sob + hi * soh
    offs_m = pid * BLOCK_M + nl.arange(0, BLOCK_M)
    offs_d = nl.arange(0, D)
    qmask = offs_m[:, None] < S
    q = nl.load(q_base + offs_m[:, None] * sqm + offs_d[None, :], mask=qmask, other=0.0)

    m_i = nl.full((BLOCK_M,), float("-inf"), dtype=nl.float32)
    l_i = nl.zeros((BLOCK_M,), dtype=nl.float32)
    acc = nl.zeros((BLOCK_M, D), dtype=nl.float32)

    end_n = S
    if CAUSAL:
        end_n = nl.minimum(S, (pid + 1) * BLOCK_M)
    for start_n in range(0, end_n, BLOCK_N):
        offs_n = start_n + nl.arange(0, BLOCK_N)
        nmask = offs_n[:, None] < S
        k = nl.load(k_base + offs_n[:, None] * skn + offs_d[None, :], mask=nmask, other=0.0)
        qk = nl.dot(q, nl.trans(k)) * scale
        if CAUSAL:
            qk = nl.where((offs_n[None, :] < S) & (offs_m[:, None] >= offs_n[None, :]),
                          qk, float("-inf"))
        else:
            qk = nl.where(offs_n[None, :] < S, qk, float("-inf"))
        m_new = nl.maximum(m_i, nl.max(qk, axis=1))
        alpha = nl.exp(m_i - m_new)
        p = nl.exp(qk - m_new[:, None])
        l_i = l_i * alpha + nl.sum(p, axis=1)
        acc = acc * alpha[:, None]
        v = nl.load(v_base + offs_n[:, None] * svn + offs_d[None, :], mask=nmask, other=0.0)
        acc = nl.dot(p.to(v_ptr.dtype.element_ty), v, acc)
        m_i = m_new

    acc = acc / l_i[:, None]
    nl.store(o_base + offs_m[:, None] * som + offs_d[None, :], acc, mask=qmask)


@functools.lru_cache(maxsize=1024)
def attention_tile(S, heads, D, causal):
    """(query rows, waves) of a program of the default kernel at 64-key blocks.

    256 rows on 8 waves share each K and V block between the most rows, but
    one such workgroup takes a whole CU: a launch wants a multiple of 256 of
    them. 128 rows on 4 waves run two to a CU, in half the steps and 2-6%
    slower per row (1-2% faster at head dim 64); 128 rows on 8 waves and 64 on
    4 keep 16 rows per wave and so read K and V twice as often, which costs
    15-25% where the chip is full anyway but fills four SIMDs with the fewest
    rows. Lines drawn from bf16 sweeps of 256 to 4096 keys over 96 to 1024
    programs of 256 rows (us, [heads, S]; 256x8 / 128x8 / 128x4 / 64x4):
      not causal, D 128: [24, 1024] 30.7 / 21.1 / 22.1 / 22.7, [40, 1024] 31.4 /
      39.7 / 34.1 / 35.0, [68, 1024] 63.0 / 58.8 / 52.8 / 53.8, [100, 1024] 63.6 /
      79.1 / 66.7 / 73.0: the costs below are rounds of the 256 CUs, measured in
      full rounds of 256 rows;
      causal, D 128 (the programs of a head differ in length, so more of them
      also balance better): [32, 1024] 33.4 / 22.0 / 24.3 / 18.8, [64, 1024] 35.6 /
      29.7 / 36.6 / 31.8, [112, 1024] 52.9 / 57.5 / 49.7 / 52.0, [40, 2048] 58.7 /
      62.4 / 52.2 / 59.8, [64, 2048] 76.1 / 87.4 / 80.0 / 90.0, [80, 2048] 104 / 114 /
      96 / 112, [128, 2048] 166 / 188 / 168 / 192;
      heads that the 8 XCDs share evenly, S from 2048 (256x8 / 128x4), up to two
      rounds: [32, 2816] 75.5 / 71.1, [16, 5888] 144 / 133, [16, 6144] 150 / 147,
      [24, 4096] 104 / 106, [40, 2560] 75.8 / 79.3, [32, 3328] 89.0 / 96.5, [24, 4608]
      122 / 132, [16, 7168] 178 / 198, [40, 3072] 98.6 / 102, [48, 2560] 87.6 / 87.8,
      [64, 2048] 75.4 / 79.6, [16, 8192] 228 / 245, [40, 3328] 121 / 113, [24, 5632] 179 /
      177; with an odd number of heads per XCD in 8 or 9 blocks [56, 2048] 75.2 /
      72.7, [56, 2304] 87.8 / 83.3, [40, 2304] 64.3 / 65.9; from four rounds on
      [128, 2048] 156 / 155, [64, 4096] 275 / 267, [128, 4096] 547 / 547, [32, 8192] 475 /
      490;
      other heads: [47, 2048] 89 / 83, [49, 2048] 108 / 89, [63, 2048] 111 / 101,
      [65, 2048] 119 / 108, [31, 4096] 185 / 170, [33, 4096] 196 / 176, [129, 2048]
      206 / 180, [125, 4096] 604 / 558, [65, 8192] 1080 / 1047;
      causal, D 64: [64, 1024] 24.3 / 24.2 / 23.6 / 20.2, [256, 1024] 74.2 / 64.2 /
      60.7 / 58.7, [64, 2048] 52.1 / 53.9 / 50.0 / 55.9, [32, 2048] 41.9 / 32.6 /
      30.1 / 28.3."""
    def rounds(rows):
        return newt.cdiv(newt.cdiv(S, rows) * heads, 256)

    programs = newt.cdiv(S, 256) * heads
    if not causal:
        if D > 64:
            cost = {(256, 8): 0.88 * rounds(256) + 0.02, (128, 8): 0.58 * rounds(128),
                    (128, 4): max(0.45 * rounds(128) + 0.1, 0.61),
                    (64, 4): 0.29 * rounds(64) + 0.06}
        else:
            cost = {(256, 8): rounds(256), (128, 4): rounds(128) / 2.04,
                    (64, 4): rounds(64) / 3.72}
        return min(cost, key=cost.get)
    if D <= 64:
        return (64, 4) if S <= 1024 or rounds(128) < 4 else (128, 4)
    if programs <= 256:
        return (128, 8) if programs > 160 and S > 512 else (64, 4)
    # long sequences whose heads divide over the 8 XCDs: a launch of up to two
    # rounds lasts as long as its longest program, which 256 rows run in less
    # once the rest fills three quarters of that time; from four rounds on it
    # balances by the number of programs. In between, and where an XCD holds a
    # part of a head, the halves on 4 waves fill the last round better. 256-wide
    # heads do not fit 256 rows' registers ([64, 2048] 987 / 221)
    if D <= 128 and S >= 2048 and heads % 8 == 0 and (
            programs >= 1024 or (376 < programs <= 512 and (heads % 16 == 0 or S > 2304))):
        return 256, 8
    return 128, 4


def attention(q, k, v, causal=False, scale=None, out=None, BLOCK_M=None, BLOCK_N=64,
              num_warps=None, num_stages=2, waves_per_eu=2, plain=False):
    """Flash attention forward over [B, H, S, D] tensors (unit stride along D).

    plain=True launches attention_plain_kernel (the examples/05 form). A
    scale <= 0 always does: the default kernel folds the scale into the
    exponent and takes max(qk) * scale as the row maximum, which holds only
    for a positive scale.

    Default tiles: 32 query rows per wave, two waves per SIMD, 256-row
    programs on 8 waves (one workgroup per CU shares each K and V block
    between all 8 waves); causal too, where two 128-row workgroups per CU
    measured 2-3% slower. A launch of the default kernel too small for that
    takes attention_tile's."""
    B, H, S, D = q.shape
    scale = D ** -0.5 if scale is None else float(scale)
    plain = plain or not scale > 0
    if (BLOCK_M is None and num_warps is None and not plain
            and (BLOCK_N, num_stages, waves_per_eu) == (64, 2, 2)):
        BLOCK_M, num_warps = attention_tile(S, B * H, D, causal)
    if BLOCK_M is None:
        BLOCK_M = 256
    if num_warps is None:
        num_warps = BLOCK_M // 32
    out = torch.empty_like(q) if out is None else out
    sq, sk, sv, so = q.stride(), k.stride(), v.stride(), out.stride()
    if not sq[3] == sk[3] == sv[3] == 1:
        raise ValueError("attention: q, k and v need unit stride along head_dim")
    if so[3] != 1:
        raise ValueError("attention: out needs unit stride along head_dim")
    kernel = attention_plain_kernel if plain else attention_kernel
    kernel[(newt.cdiv(S, BLOCK_M), B * H)](
        q, k, v, out, S, H, scale, *sq[:3], *sk[:3], *sv[:3], *so[:3],
        BLOCK_M=BLOCK_M, BLOCK_N=BLOCK_N, D=D, CAUSAL=causal, num_warps=num_warps,
        num_stages=num_stages, waves_per_eu=waves_per_eu)
    return out


# ---------------------------------------------------------------------------
# 6. deuteron matmul (examples/deuteron/01_matmul.py, unchanged body)
# ---------------------------------------------------------------------------
from . import deuteron as dt  # noqa: E402


@dt.kernel
def dt_matmul(x, y, out):
    for tile_m, tile_n in dt.tile([x.shape[0], y.shape[1]]):
        acc = dt.zeros([tile_m, tile_n], dtype=dt.float32)
        for tile_k in dt.tile(x.shape[1]):
            acc += x[tile_m, tile_k] @ y[tile_k, tile_n]
        out[tile_m, tile_n] = acc
