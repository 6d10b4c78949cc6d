"""The 256-byte and longer LDS rows of deep k-steps (small output tiles keep
few rows and many k per stage), under the bank model of test_lds_layout_cpu."""

import re
import subprocess

import pytest
import test_lds_layout_cpu as lds
from test_codegen_cpu import A16, D16, compile_source

from newt_amd import workloads as W
from newt_amd.compiler import types as tp


def test_long_k_major_rows_are_bijective_and_conflict_free(tmp_path):
    src, exe = tmp_path / "lds.cpp", tmp_path / "lds"
    checks = "".join(f"check_k<{kd}, {mi}>();" for kd in (128, 256, 512) for mi in (16, 32))
    src.write_text(re.sub(r"int main\(\) \{.*", "int main() {" + checks + "}", lds.HARNESS,
                          flags=re.S))
    subprocess.run([lds.HIPCC, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O1",
                    "-I", lds.HEADER_DIR, str(src), "-o", str(exe)], check=True,
                   capture_output=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    rows = [line.split() for line in out.splitlines()]
    assert len(rows) == 6
    for f in rows:
        assert f[-2:] == ["1", "1"], f


@pytest.mark.parametrize("dtype,tile,stages_kb", [
    ("float16", (64, 64, 64, 8, 3), 48), ("bfloat16", (16, 16, 512, 4, 4), 128),
    ("float32", (64, 64, 32, 8, 4), 64), ("float32", (32, 64, 64, 8, 4), 96),
    ("float32", (32, 64, 32, 4, 4), 48)])
def test_joining_k_shares_takes_no_lds_of_its_own(dtype, tile, stages_kb):
    """A loop whose waves split k joins their shares through a stage's LDS, so
    the kernel holds its stages alone."""
    ptr, i, one = tp.pointer_type(getattr(tp, dtype)), tp.int32, {"eq1": True}
    BM, BN, BK, waves, stages = tile
    args = {"a_ptr": (ptr, A16), "b_ptr": (ptr, A16), "c_ptr": (ptr, A16), "M": i, "N": i, "K": i,
            "sam": (i, D16), "sak": (i, one), "sbk": (i, one), "sbn": (i, D16), "scm": (i, D16),
            "scn": (i, one)}
    src, lds = compile_source(W.matmul_kernel, args, {"BLOCK_M": BM, "BLOCK_N": BN, "BLOCK_K": BK},
                              waves, stages)
    assert "newt::join_k_groups" in src
    assert lds == stages_kb * 1024
