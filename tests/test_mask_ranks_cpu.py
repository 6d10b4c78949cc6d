"""Masks whose terms differ in rank: `(rows[:, None] < M) & (cols < N)` is
`(rows[:, None] < M) & (cols[None, :] < N)`, so both forms compile to the same
source, in loads, stores, `where` and the operands of a pipelined dot (either
operand, either storage order, the ragged k among the terms)."""

import pytest
from test_codegen_cpu import A16, D16, F16P, F32P, compile_source

import newt_amd.language as nl
from newt_amd.compiler import types as tp


def copy_k(x_ptr, o_ptr, M, N, stride, FULL: nl.constexpr, BM: nl.constexpr, BN: nl.constexpr):
    rows, cols = nl.arange(0, BM), nl.arange(0, BN)
    if FULL:
        mask = (rows[:, None] < M) & (cols[None, :] < N)
    else:
        mask = (rows[:, None] < M) & (cols < N)
    offs = rows[:, None] * stride + cols[None, :]
    x = nl.load(x_ptr + offs, mask=mask, other=0.0)
    x = nl.where(mask, x * 2.0, 1.0)
    nl.store(o_ptr + offs, x, mask=mask)


def three_terms_k(x_ptr, o_ptr, M, N, stride, FULL: nl.constexpr, BM: nl.constexpr,
                  BN: nl.constexpr):
    rows, cols = nl.arange(0, BM), nl.arange(0, BN)
    if FULL:
        mask = ((cols[None, :] >= 8) & (cols[None, :] < N)) & (rows[:, None] < M)
    else:
        mask = ((cols >= 8) & (cols < N)) & (rows[:, None] < M)
    offs = rows[:, None] * stride + cols[None, :]
    nl.store(o_ptr + offs, nl.load(x_ptr + offs, mask=mask, other=1.0), mask=mask)


def dot_k(a_ptr, b_ptr, o_ptr, M, N, K, sam, sak, sbk, sbn, FULL: nl.constexpr, BM: nl.constexpr,
          BN: nl.constexpr, BK: nl.constexpr):
    rm, rn, rk = nl.arange(0, BM), nl.arange(0, BN), nl.arange(0, BK)
    acc = nl.zeros((BM, BN), dtype=nl.float32)
    for k in range(nl.cdiv(K, BK)):
        left = K - k * BK
        if FULL:
            a_mask = (rm[:, None] < M) & (rk[None, :] < left)
            b_mask = (rn[None, :] < N) & (rk[:, None] < left)
        else:
            a_mask = (rm[:, None] < M) & (rk < left)
            b_mask = (rn < N) & (rk[:, None] < left)
        a = nl.load(a_ptr + rm[:, None] * sam + (k * BK + rk[None, :]) * sak, mask=a_mask, other=0.0)
        b = nl.load(b_ptr + (k * BK + rk[:, None]) * sbk + rn[None, :] * sbn, mask=b_mask, other=0.0)
        acc = nl.dot(a, b, acc)
    nl.store(o_ptr + rm[:, None] * BN + rn[None, :], acc)


@pytest.mark.parametrize("kernel", [copy_k, three_terms_k])
@pytest.mark.parametrize("BM,BN", [(4, 64), (64, 4), (16, 256)])
@pytest.mark.parametrize("facts", [{}, D16])
def test_row_kernels(kernel, BM, BN, facts):
    args = {"x_ptr": (F32P, A16), "o_ptr": (F32P, A16), "M": tp.int32, "N": (tp.int32, facts),
            "stride": (tp.int32, facts)}
    got, want = (compile_source(kernel, args, {"FULL": full, "BM": BM, "BN": BN})
                 for full in (False, True))
    assert got == want
    assert f"(-N) + {BN - 1})" in got[0]     # the column bound over the columns' extent


ONE = {"eq1": True}


@pytest.mark.parametrize("a_strides", [(D16, ONE), (ONE, D16), ({}, ONE)])
@pytest.mark.parametrize("b_strides", [(D16, ONE), (ONE, D16), ({}, ONE)])
@pytest.mark.parametrize("tile", [(64, 64, 64, 8, 3), (128, 64, 32, 4, 4), (32, 64, 128, 4, 2)])
def test_dot_operands(tile, a_strides, b_strides):
    BM, BN, BK, waves, stages = tile
    i = tp.int32
    args = {"a_ptr": (F16P, A16), "b_ptr": (F16P, A16), "o_ptr": (F32P, A16), "M": i,
            "N": (i, D16), "K": (i, D16), "sam": (i, a_strides[0]), "sak": (i, a_strides[1]),
            "sbk": (i, b_strides[0]), "sbn": (i, b_strides[1])}
    got, want = (compile_source(dot_k, args, {"FULL": full, "BM": BM, "BN": BN, "BK": BK}, waves,
                                stages) for full in (False, True))
    assert got == want
