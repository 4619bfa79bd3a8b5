"""The eigensolver of a persymmetric tridiagonal matrix by its even and odd
halves (dopamine-fdm_amd/csrc/symtri_eigen.h), built with g++: eigenvalues
against LAPACK, the eigen identity, orthonormality and exact parity, on the
z-wall operators of uniform and stretched ducts."""
from __future__ import annotations

import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest
import scipy.linalg

from oracle import ref_numpy as R

HDR = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dopamine-fdm_amd", "csrc")
SRC = r'''
#include "symtri_eigen.h"
extern "C" int eig(int n, const double* d, const double* e, double* lam, double* v) {
    std::vector<long double> dl(d, d + n), el(e, e + (n > 1 ? n - 1 : 1));
    std::vector<double> dd, vv;
    if (!dfp::symtri_eigen_sym(n, dl, el, dd, vv)) return 1;
    for (int i = 0; i < n; ++i) lam[i] = dd[i];
    for (size_t i = 0; i < vv.size(); ++i) v[i] = vv[i];
    return 0;
}
'''


@pytest.mark.skipif(not shutil.which("g++"), reason="no g++")
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 16, 33, 130])
@pytest.mark.parametrize("alpha", [0.0, 2.0])
def test_halves_match_lapack(n, alpha, tmp_path):
    (tmp_path / "e.cpp").write_text(SRC)
    so = str(tmp_path / "libe.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", HDR, str(tmp_path / "e.cpp"), "-o", so],
                   check=True)
    lib = ctypes.CDLL(so)
    dp = ctypes.POINTER(ctypes.c_double)
    g = R.duct_grid(4, 3, n, 1.0, alpha)
    D = R.dyy_matrix(g.z, g.zg)
    w = g.z[1:] - g.z[:-1]
    d = np.ascontiguousarray(np.diag(D))
    e = np.array([1.0 / ((g.zg[k + 1] - g.zg[k]) * np.sqrt(w[k - 1] * w[k])) for k in range(1, n)] or [0.0])
    lam, v = np.zeros(n), np.zeros(n * n)
    assert lib.eig(n, *(a.ctypes.data_as(dp) for a in (d, e, lam, v))) == 0
    v = v.reshape((n, n), order="F")
    S = np.diag(d) + (np.diag(e, 1) + np.diag(e, -1) if n > 1 else 0.0)
    scale = np.max(np.abs(S))
    ref = scipy.linalg.eigvalsh(S)
    assert np.max(np.abs(np.sort(lam) - ref)) <= 1e-13 * n * scale
    assert np.max(np.abs(S @ v - v * lam)) <= 1e-13 * n * scale
    assert np.max(np.abs(v.T @ v - np.eye(n))) <= 1e-13 * n
    h = (n + 1) // 2
    assert np.array_equal(v[::-1, :h], v[:, :h]) and np.array_equal(v[::-1, h:], -v[:, h:])
