"""NEWT_BARE_BARRIER=1: the barrier without a fence publishes asynchronous
copies only, so a branch-free loop that writes a tile to LDS from registers
(loaded ahead, or written after the MFMAs) keeps the fenced barrier."""

import re

import pytest
from test_codegen_cpu import A16, D16, F16P, compile_source, isa

from newt_amd import workloads as W
from newt_amd.compiler import types as tp

ONE = {"eq1": True}


def matmul(a_facts, sam, sak, sbk, sbn, tile):
    i = tp.int32
    BM, BN, BK, waves, stages = tile
    args = {"a_ptr": (F16P, a_facts), "b_ptr": (F16P, A16), "c_ptr": (F16P, A16), "M": i, "N": i,
            "K": i, "sam": (i, sam), "sak": (i, sak), "sbk": (i, sbk), "sbn": (i, sbn),
            "scm": (i, D16), "scn": (i, ONE)}
    return compile_source(W.matmul_kernel, args, {"BLOCK_M": BM, "BLOCK_N": BN, "BLOCK_K": BK},
                          waves, stages)[0]


# tiles loaded ahead; written late with 2 and with 4 stages (a strided operand)
FROM_REGISTERS = [(({}, {}, ONE, {}, ONE), (64, 64, 64, 8, 3)),
                  (({}, {}, ONE, {}, ONE), (64, 64, 64, 4, 2)),
                  ((A16, D16, {}, D16, ONE), (64, 64, 64, 4, 2)),
                  ((A16, D16, {}, D16, ONE), (128, 128, 32, 4, 4))]


@pytest.mark.parametrize("facts,tile", FROM_REGISTERS)
def test_tiles_written_from_registers_are_fenced(monkeypatch, facts, tile):
    monkeypatch.setenv("NEWT_BARE_BARRIER", "1")
    src = matmul(*facts, tile)
    assert "__syncthreads" in src and "barrier_nofence" not in src
    # no wave arrives at a barrier with an LDS write of its own still in flight
    pending = False
    for ln in isa(src).splitlines():
        if re.search(r"\bds_write", ln):
            pending = True
        elif "s_waitcnt" in ln and "lgkmcnt(0)" in ln:
            pending = False
        elif re.search(r"\bs_barrier\b", ln):
            assert not pending
    assert "ds_write" in isa(src)


def test_copied_tiles_take_the_bare_barrier(monkeypatch):
    monkeypatch.setenv("NEWT_BARE_BARRIER", "1")
    assert "barrier_nofence" in matmul(A16, D16, ONE, D16, ONE, (128, 128, 32, 4, 3))
