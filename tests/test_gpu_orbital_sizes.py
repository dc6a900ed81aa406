"""The orbital step's kernels at the edges of their tiles: 16 x 16 and 64 x 64
product tiles, 64-slice rows of the gather, the exponential below and above
128 orbitals, results of up to 32 x 32 and above.

Tolerances: an element sums at most no^2 nq < 1e5 products, so its rounding
stays below 1e5 eps = 2e-11 of the largest partial sum in the worst case and
near sqrt(1e5) eps = 7e-14 in the mean; 1e-11 relative to the largest element
is the bound the other orbital tests use.
"""
import numpy as np
import pytest

from hilbert_amd.batch import Batch, Problem, options
from hilbert_amd.integrals import synthetic_df
from oracle import orbopt as oo
from oracle.pyoracle import OracleProblem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nfull,ncore,n,nq", [(5, 1, 4, 5), (16, 12, 4, 63), (17, 12, 5, 64), (65, 28, 4, 65),
                                               (128, 29, 4, 129), (130, 12, 4, 136)])
def test_orbital_step_matches_oracle_at_tile_edges(nfull, ncore, n, nq):
    rng = np.random.default_rng(7000 + nfull)
    h, qmo, _ = synthetic_df(nfull, nq, rng)
    core = np.arange(ncore, dtype=np.int32)
    active = np.arange(ncore, ncore + n, dtype=np.int32)
    B = Batch([Problem(n, 2, 2)], options())
    B.set_guess_hf(0)
    B.set_df_integrals(0, h, qmo, core, active)
    pairs, g, H = B.orbital_gradient(0)
    x = B.x(0)
    B.optimize_orbitals(0, maxiter=1)
    U, h_gpu, q_gpu = B.df_orbitals(0)
    B.close()
    P = OracleProblem(n, 2, 2, [0] * n, 1)
    D1, d = oo.spatial_rdms(P, x)
    D, dd = oo.occupied_rdms(D1, d, ncore)
    occ = list(core) + [int(active[u]) for u in oo.pitzer_order([0] * n)]
    opairs = oo.rotation_pairs(nfull, core, active, None)
    assert np.array_equal(pairs, opairs)
    Bd = oo.unpack_df(qmo, nfull)
    go, Ho = oo.gradient_hessian(h, Bd, D, dd, occ, opairs)
    print(nfull, "max |dg|", np.abs(g - go).max(), "max |dH|", np.abs(H - Ho).max(), flush=True)
    assert np.abs(g - go).max() <= 1e-11 * max(1.0, np.abs(go).max())
    assert np.abs(H - Ho).max() <= 1e-11 * max(1.0, np.abs(Ho).max())
    _, _, Uo, _ = oo.optimize_orbitals(h, Bd, D, dd, occ, opairs, maxiter=1)
    # the step is -g / max(|H|, 1e-2), so small H magnify the roundings of g and
    # H checked above: exp(K + dK) differs from exp(K) by at most ||dK||_2 <=
    # ||dK||_1 (both antisymmetric), twice that for a step taken in two parts
    dk = np.zeros((nfull, nfull))
    dk[pairs[:, 0], pairs[:, 1]] = np.abs(g / np.maximum(np.abs(H), 1e-2) - go / np.maximum(np.abs(Ho), 1e-2))
    bound = 1e-12 + 2.0 * (dk + dk.T).sum(axis=0).max()
    print(nfull, "max |dU|", np.abs(U - Uo).max(), "bound", bound, flush=True)
    assert np.abs(U - Uo).max() <= bound
    # exp(K) is squared log2(2 ||K||_1) times, and each time doubles an error
    # that begins near eps
    kappa = np.zeros((nfull, nfull))
    kappa[pairs[:, 0], pairs[:, 1]] = np.abs(go) / np.maximum(np.abs(Ho), 1e-2)
    orth = 1e-12 + 4.0 * np.finfo(float).eps * (kappa + kappa.T).sum(axis=0).max()
    assert np.abs(U.T @ U - np.eye(nfull)).max() <= orth
    # the integrals rotated by the U that was returned: two products of nfull terms
    assert np.abs(h_gpu - U.T @ h @ U).max() <= 1e-12 * max(1.0, np.abs(h).max())
    B2 = np.einsum("pi,Qpq,qj->Qij", U, Bd, U, optimize=True)
    assert np.abs(q_gpu - oo.pack_df(B2)).max() <= 1e-12 * max(1.0, np.abs(Bd).max())
