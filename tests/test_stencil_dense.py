"""The bounded x pass evaluates closure rows with dense per-column weights of
f(q) - f(0).  Host-only check (tests/native/stencil_dense_check.cpp): they give
the row-by-row stencils of src/dfbydx.f:116-228 and src/d2fdx2.f:116-260 to
rounding on all 11 row kinds, and the interior rows with working-precision
coefficients are the same sums."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not present")
def test_dense_rows_equal_switch_form(tmp_path):
    exe = tmp_path / "stencil_dense_check"
    src = os.path.join(HERE, "native", "stencil_dense_check.cpp")
    r = subprocess.run([HIPCC, "-O2", "-std=c++17", "-ffp-contract=off", "-I", os.path.join(ROOT, "include"),
                        "-I", os.path.join(ROOT, "senga-versiona_amd", "csrc"), src, "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
    assert r.stdout.count(" ok") == 12
