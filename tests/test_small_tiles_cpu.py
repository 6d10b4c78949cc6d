"""The 256-byte and longer LDS rows of deep k-steps (small output tiles keep
few rows and many k per stage), under the bank model of test_lds_layout_cpu."""

import re
import subprocess

import test_lds_layout_cpu as lds


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
