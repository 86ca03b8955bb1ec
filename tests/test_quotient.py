"""CPU: the quotients by constants of dba_amd/csrc/mathf64.h (Model B's logarithms over
r_x, r_y, r_z), compiled as plain C++.

Bar: the correctly rounded quotient, bit for bit, as a division gives it. The product
with the reciprocal alone, which is one rounding more, has to fail the same bar."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

WRAP = r"""
#include "mathf64.h"
extern "C" void t_quot(const double* a, const double* b, double* q, double* any, long n) {
    for (long i = 0; i < n; i++) {
        q[i] = dba::quotient(a[i], b[i], 1.0 / b[i]);
        any[i] = dba::quotient_any(a[i], b[i], 1.0 / b[i]);
    }
}
"""


@pytest.fixture(scope="module")
def quot(tmp_path_factory):
    d = tmp_path_factory.mktemp("quotient")
    (d / "w.cpp").write_text(WRAP)
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-fPIC", "-shared", "-I",
                    os.path.join(ROOT, "dba_amd", "csrc"), "-o", str(d / "w.so"), str(d / "w.cpp")], check=True)
    lib = ctypes.CDLL(str(d / "w.so"))
    P = ctypes.POINTER(ctypes.c_double)

    def f(a, b):
        a, b = (np.ascontiguousarray(v, dtype=np.float64) for v in np.broadcast_arrays(a, b))
        q, any_ = np.empty_like(a), np.empty_like(a)
        lib.t_quot(*(v.ctypes.data_as(P) for v in (a, b, q, any_)), ctypes.c_long(a.size))
        return q, any_
    return f


def test_quotient_rounds_to_nearest(quot):
    rng = np.random.default_rng(3)
    n = 300_000
    a = np.concatenate([np.log(rng.uniform(1e-12, 1.0, n)), rng.uniform(0.0, 5.0, n),
                        np.nextafter(1.0, 2.0) ** np.arange(8), [0.0, 745.13, 2.0 ** -53]])
    bs = np.concatenate([np.arange(1.0, 130.0), 1.0 - rng.uniform(0.0, 0.999, 40), rng.uniform(0.01, 2000.0, 40),
                         [np.nextafter(1.0, 0.0), np.nextafter(2.0, 0.0), np.nextafter(1.0, 2.0), 1e-3, 1e6, -3.0]])
    worse = 0
    for b in bs:
        q, any_ = quot(a, b)
        assert np.array_equal(q, a / b), b
        assert np.array_equal(any_, a / b), b
        worse += int((a * (1.0 / b) != a / b).sum())
    assert worse > 0


def test_quotient_of_no_finite_value(quot):
    a = np.array([np.inf, -np.inf, np.nan, -np.inf])
    _, q = quot(a, np.array([3.0, 7.0, 3.0, -2.0]))
    assert q[0] == np.inf and q[1] == -np.inf and np.isnan(q[2]) and q[3] == np.inf
