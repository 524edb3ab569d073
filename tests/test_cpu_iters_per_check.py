"""Iterations enqueued between completion tests (gpu_solver.cpp,
iterations_ahead): a value that the caller sets is kept whatever the
convergence; only the default looks ahead, never below itself, past half of the
iterations left or past 32."""
import ctypes
import math
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
sys.path.insert(0, str(ROOT))

SHIM = r"""
#include "apxchol_amd/csrc/host/gpu_solver.hpp"
extern "C" int ahead(int every, double residual, long iterations, double tol) {
    return apxchol_amd::iterations_ahead(every, residual, iterations, tol);
}
"""


@pytest.fixture(scope="module")
def ahead(tmp_path_factory):
    from apxchol_amd import build as b
    if not b.LIB.exists():
        pytest.fail(f"{b.LIB} is missing: build it first")
    tmp = tmp_path_factory.mktemp("ahead")
    src, so = tmp / "shim.cpp", tmp / "shim.so"
    src.write_text(SHIM)
    r = subprocess.run([str(b.ROCM / "llvm" / "bin" / "clang++"), *b.HOST_FLAGS, "-shared", f"-I{ROOT}", str(src),
                        "-o", str(so), f"-L{b.LIB.parent}", "-lapxchol_amd", f"-Wl,-rpath,{b.LIB.parent}"],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    f = ctypes.CDLL(str(so)).ahead
    f.argtypes = [ctypes.c_int, ctypes.c_double, ctypes.c_long, ctypes.c_double]
    return f


@pytest.mark.parametrize("residual", [0.9, 1e-1, 1e-3, 1e-7, 1e-9, 2.0, math.nan, math.inf])
@pytest.mark.parametrize("iterations", [0, 1, 2, 10, 40, 1000])
def test_set_values_are_kept_and_the_default_looks_ahead(ahead, residual, iterations):
    tol = 1e-8
    for every in (1, 3, 4, 8, 50):
        assert ahead(every, residual, iterations, tol) == every
    n = ahead(2, residual, iterations, tol)
    assert 2 <= n <= 32
    if tol < residual < 1.0 and iterations > 0:
        left = math.log(tol / residual) / math.log(residual) * iterations
        assert n <= max(2, 0.5 * left + 1e-9)
    else:
        assert n == 2


def test_the_default_does_look_ahead(ahead):
    assert ahead(2, 1e-2, 10, 1e-8) == 15      # 30 left at 0.2 digits each
    assert ahead(2, 1e-1, 40, 1e-8) == 32
