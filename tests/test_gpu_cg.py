"""GPU: the conjugate gradients of one outer iteration, at sizes on both sides of
the line between the CG in one workgroup (registers and LDS) and the CG in two
launches a step, against the residual computed in numpy.

The stopping rule bounds the recursive residual by 0.003 ||rhs|| in the first
iteration; the true one drifts from it by rounding only, about steps x
eps x cond of the steps taken, well below 1e-9 ||rhs||.
"""
import numpy as np
import pytest

from hilbert_amd.batch import Batch, Problem, options
from hilbert_amd.integrals import synthetic_integrals
from hilbert_amd.structure import Structure

pytestmark = pytest.mark.gpu

NEVER = dict(e_convergence=1e-14, r_convergence=1e-13, maxiter=1000000)
# (orbitals, irreps): 1 x 1 blocks, rows of several pieces, 96 slices and a few
# more, long rows, T2
CASES = [(1, 1, False), (2, 1, False), (3, 2, False), (4, 1, False), (5, 1, False), (6, 4, False), (7, 4, False),
         (7, 8, False), (8, 8, False), (10, 8, False), (12, 4, False), (3, 1, True), (4, 2, True)]


def _numpy_steps(A, rhs, tol):
    r = rhs.copy()
    p, rr, n = r.copy(), r @ r, 0
    while rr > tol * tol * (rhs @ rhs):
        q = A.T @ p
        al = rr / (q @ q)
        r = r - al * (A @ q)
        new = r @ r
        p, rr, n = r + new / rr * p, new, n + 1
    return n


@pytest.mark.parametrize("n,nirrep,t2", CASES)
def test_first_cg_reaches_its_tolerance(n, nirrep, t2):
    irr = [k * nirrep // n for k in range(n)] if nirrep > 1 else None
    na, nb = (n + 1) // 2, n // 2
    A, b = Structure(n, na, nb, irr, nirrep, t2=t2).matrix()
    p = Problem(n, na, nb, irr, nirrep, t2=t2)
    # alone, and twice in one batch with a larger instance, whose CG is the other kind
    for items in ([p], [p, Problem(9, 5, 4, None, 1), p]):
        B = Batch(items, options(**NEVER))
        for i, q in enumerate(items):
            h, g = synthetic_integrals(q.nmo, 2 * q.nmo + 3, 7, irreps=q.irreps)
            B.set_integrals(i, h, g)
        x0, c, mu = B.x(0), B.c(0), B.mu(0)
        rhs = A @ c + mu * (b - A @ x0)
        B.solve(1)
        y = B.y(0)
        res = np.linalg.norm(rhs - A @ (A.T @ y)) / np.linalg.norm(rhs)
        steps = _numpy_steps(A, rhs, 0.003)
        assert res <= 0.003 + 1e-9, (n, res)
        assert abs(B.status(0)["iiter"] - steps) <= 1, (B.status(0)["iiter"], steps)
        if len(items) > 1:
            assert np.array_equal(y, B.y(2)) and np.array_equal(y, alone)
        alone = y
        B.close()
