"""The host eigensolver of the Davidson driver (csrc/sym_eigh.hpp), compiled as it stands with g++:
couplings whose squares leave the normal range, graded, degenerate, zero and denormal matrices, and
matrices that are not finite.

Tolerance: Householder reduction and QR steps are backward stable; the residual |A V - V w| and
|V^T V - 1| of an m x m problem stay within a few m units of rounding of |A|.  64 m eps covers m up to 256."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def eigh(tmp_path_factory):
    d = tmp_path_factory.mktemp("eigh")
    src, so = d / "e.cpp", d / "e.so"
    src.write_text('#include "sym_eigh.hpp"\n#include <cstring>\n'
                   'extern "C" int eigh(int m, const double *a, double *w, double *v) {\n'
                   '    std::vector<double> W, V;\n'
                   '    if (!hipotf::sym_eigh(m, std::vector<double>(a, a + m * m), W, V)) return 0;\n'
                   '    std::memcpy(w, W.data(), m * 8);\n    std::memcpy(v, V.data(), m * m * 8);\n    return 1;\n}\n')
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "binsim_amd", "csrc"),
                    str(src), "-o", str(so)], check=True)
    f = C.CDLL(str(so)).eigh
    dp = C.POINTER(C.c_double)

    def call(a):
        a = np.ascontiguousarray(a, dtype=np.float64)
        m = len(a)
        w, v = np.full(m, np.nan), np.full((m, m), np.nan)
        ok = f(m, a.ctypes.data_as(dp), w.ctypes.data_as(dp), v.ctypes.data_as(dp))
        return ok, w, v
    return call


def _check(a, ok, w, v):
    m, s = len(a), np.frexp(np.abs(a).max())[1]
    a, w, eps = np.ldexp(a, -s), np.ldexp(w, -s), 64 * len(a) * np.finfo(float).eps
    assert ok and np.all(np.diff(w) >= 0.0)
    assert np.max(np.abs(a @ v - v * w)) <= eps
    assert np.max(np.abs(v.T @ v - np.eye(m))) <= eps


def _sym(rng, m):
    a = rng.standard_normal((m, m))
    return a + a.T


@pytest.mark.parametrize("t", [0.0, 5e-324, 1e-310, 1e-200, 1e-163, 1e-162, 1e-161, 1e-160, 1e-158, 1e-155, 1e-154,
                               1e-150, 1e-100, 1e-17])
def test_tiny_couplings(eigh, t):
    a = np.array([[1.0, 0.0, t], [0.0, 2.0, 0.1], [t, 0.1, 3.0]])
    _check(a, *eigh(a))
    b = np.diag(-np.arange(1.0, 7.0)) + t * (1.0 - np.eye(6))
    _check(b, *eigh(b))


@pytest.mark.parametrize("m", [1, 2, 3, 4, 17, 64, 256])
def test_ordinary_graded_and_degenerate_matrices(eigh, m):
    rng = np.random.default_rng(m)
    q = np.linalg.qr(rng.standard_normal((m, m)))[0]
    for a in (_sym(rng, m), np.zeros((m, m)), np.eye(m), (q * np.arange(m)) @ q.T, (q * (np.arange(m) // 3)) @ q.T,
              _sym(rng, m) * np.outer(g := 10.0 ** -np.linspace(0, 12, m), g), 1e-200 * _sym(rng, m), 1e-310 * _sym(rng, m),
              1e150 * _sym(rng, m), np.ones((m, m)),
              np.outer(q[0], q[0]), np.outer(q[0], q[0]) + 1e-300 * _sym(rng, m)):
        a = 0.5 * (a + a.T)
        _check(a, *eigh(a))


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_not_finite(eigh, bad):
    a = _sym(np.random.default_rng(1), 5)
    a[1, 3] = a[3, 1] = bad
    assert eigh(a)[0] == 0
