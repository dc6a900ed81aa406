"""CPU: the tridiagonal eigensolver of the projection kernels, compiled for the
host, on spectra in which a whole group of eigenvalues is equal.

Bounds: the eigenvalues are bisected to 2 eps ||T|| and the Sturm counts are
those of a matrix within a few eps ||T||, ||T|| <= 4 (Gershgorin), so 64 eps
holds with room; reducing a dense matrix first moves them by d eps.  The
projection U+ is Lipschitz in U with constant 1, so 100 d eps max|l| leaves room
for the vectors.
"""
import ctypes

import numpy as np
import pytest

from native_host import build

EPS = np.finfo(float).eps
P = ctypes.POINTER(ctypes.c_double)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return build("tri_eigen_host", tmp_path_factory)


def _ptr(a):
    return a.ctypes.data_as(P)


def _values(lib, dd, ee, prev=None):
    d = len(dd)
    dd, ee, lam = np.ascontiguousarray(dd), np.append(ee, 0.0), np.zeros(d)
    bad = lib.tri_values_host(d, _ptr(dd), _ptr(ee), None if prev is None else _ptr(np.ascontiguousarray(prev)), _ptr(lam))
    assert bad == 0
    return lam


def _tridiagonal(w, rng, zeros):
    """A tridiagonal matrix of the given spectrum: its eigenvalues on the
    diagonal (zeros), or a dense matrix reduced by Householder steps."""
    if zeros:
        return rng.permutation(w), np.zeros(len(w) - 1)
    from scipy.linalg import hessenberg
    Q = np.linalg.qr(rng.standard_normal((len(w), len(w))))[0]
    A = (Q * w) @ Q.T
    T = hessenberg(0.5 * (A + A.T))
    return np.diag(T).copy(), 0.5 * (np.diag(T, 1) + np.diag(T, -1))


def _spectrum(kind, d, rng):
    if kind == "ends":       # one eigenvalue at each end, two large groups between
        return np.concatenate([[2.0, -2.0], np.ones(d // 2), np.zeros(d - 2 - d // 2)])
    if kind == "integers":
        w = rng.integers(-2, 2, d).astype(float)
        w[0] = 2.0
        return w
    if kind == "one positive":  # after a zero block: many zero, many negative
        return np.concatenate([[1.0], np.zeros(d // 2), -rng.uniform(0.1, 1.0, d - 1 - d // 2)])
    return np.concatenate([np.zeros((2 * d) // 3), rng.uniform(-1.0, 1.0, d - (2 * d) // 3)])  # mostly zero


@pytest.mark.parametrize("d", [17, 33, 64, 65, 128, 224, 257, 300, 417])
@pytest.mark.parametrize("kind", ["ends", "integers", "one positive", "mostly zero"])
def test_eigenvalues_of_degenerate_spectra(lib, kind, d):
    rng = np.random.default_rng([d, len(kind)])
    for rep in range(2):
        w = _spectrum(kind, d, rng)
        dd, ee = _tridiagonal(w, rng, rep == 0)
        for prev in (None, np.zeros(d + 1), np.append(np.sort(w) + 1e-3, 1e-3), np.append(np.zeros(d), 1e-2)):
            lam = _values(lib, dd, ee, prev)
            err = np.abs(np.sort(lam) - np.sort(w)).max()
            assert err <= (64 if rep == 0 else 64 + 4 * d) * EPS, (kind, d, rep, prev is None, err)


@pytest.mark.parametrize("d", [17, 64, 100])
@pytest.mark.parametrize("kind", ["ends", "integers", "one positive", "mostly zero"])
def test_projection_of_degenerate_spectra(lib, kind, d):
    rng = np.random.default_rng([d, 7, len(kind)])
    for zeros in (True, False):
        w = _spectrum(kind, d, rng)
        dd, ee = _tridiagonal(w, rng, zeros)
        lam = _values(lib, dd, ee, np.zeros(d + 1))
        S, xs = np.zeros((d, d)), np.zeros(d)
        assert lib.tri_vectors_host(d, _ptr(np.ascontiguousarray(dd)), _ptr(np.append(ee, 0.0)), _ptr(lam), _ptr(S), _ptr(xs)) == 0
        V = S / np.sqrt(xs)
        T = np.diag(dd) + np.diag(ee, 1) + np.diag(ee, -1)
        lw, lv = np.linalg.eigh(T)
        err = np.abs((V * np.maximum(lam, 0.0)) @ V.T - (lv * np.maximum(lw, 0.0)) @ lv.T).max()
        assert err <= 100 * d * EPS * 2.0, (kind, d, zeros, err)
