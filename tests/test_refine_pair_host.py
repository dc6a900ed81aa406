"""CPU: the pair corrections of the warm-started refinement, compiled for the
host."""
import ctypes

import numpy as np
import pytest

from native_host import build

P = ctypes.POINTER(ctypes.c_double)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    lib = build("refine_pair_host", tmp_path_factory)
    lib.refine_step_host.restype = ctypes.c_double
    return lib


def _step(lib, U, X):
    d = len(U)
    U, X, E = np.ascontiguousarray(U), np.array(X, order="C"), np.zeros((d, d))
    me = lib.refine_step_host(d, U.ctypes.data_as(P), X.ctypes.data_as(P), E.ctypes.data_as(P), ctypes.c_double(1e-8))
    return X, E, me


def test_equal_estimates_rotate(lib):
    """From X = I the estimates are the diagonal: pairs with the same diagonal
    element and a coupling turn by 45 degrees, (i, j) and (j, i) to opposite
    sides, and the iteration converges."""
    U = np.diag([1.0, 1.0, -0.5, -0.5, 0.25])
    U[0, 1] = U[1, 0] = 0.3
    U[2, 3] = U[3, 2] = -0.2
    X, E, me = _step(lib, U, np.eye(5))
    assert me == 1.0
    assert np.array_equal(np.triu(E, 1), -np.tril(E, -1).T)
    for _ in range(3):
        X, E, me = _step(lib, U, X)
    assert me < 1e-12
    w, V = np.linalg.eigh(U)
    l = np.einsum("ij,ik,kj->j", X, U, X)
    assert np.abs((X * np.maximum(l, 0.0)) @ X.T - (V * np.maximum(w, 0.0)) @ V.T).max() < 1e-14


@pytest.mark.parametrize("g", [1e-8, 1e-7])
def test_coupling_of_a_close_pair_leaves_out_the_overlap(lib, g):
    """x_i . x_j = g with U = 0.7 I on both: s = 0.7 g, and nothing is left once
    the step has made them orthogonal; a true coupling stays."""
    left = ctypes.c_double()
    assert lib.pair_host(ctypes.c_double(0.7), ctypes.c_double(0.7), ctypes.c_double(g), ctypes.c_double(0.7 * g),
                         ctypes.c_double(1e-8), ctypes.byref(left)) == 1
    assert abs(left.value) < 1e-22
    lib.pair_host(ctypes.c_double(0.7), ctypes.c_double(0.7), ctypes.c_double(g), ctypes.c_double(0.7 * g + 5e-9),
                  ctypes.c_double(1e-8), ctypes.byref(left))
    assert abs(left.value - 5e-9) < 1e-21
