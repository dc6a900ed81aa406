"""GPU: the PSD projection of single blocks against LAPACK, at the sizes where
its kernels change (16-row tiles, size classes) and for the spectra that decide
between refinement and eigensolver.

The caller-map solver with a zero map projects U = mu x - c, so a sequence of
U is projected with whatever eigenvectors the call before left: a first block
without any, then steps small enough to refine, then one too large.

Bound: U+ is Lipschitz in U with constant 1, so a backward-stable projection is
within a small multiple of d eps max|l| of the exact one; eps d 100 (1.4e-12 at
d = 64) leaves room for the eigensolver's clusters, whose vectors are
orthogonal to about 1e-5 / gap eps.
"""
import time

import numpy as np
import pytest
import scipy.linalg

from hilbert_amd.batch import options
from hilbert_amd.sdp import BPSDPSolver

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def _positive_part(U):
    w, V = np.linalg.eigh(U)
    return (V * np.maximum(w, 0.0)) @ V.T


def _spectrum(kind, d, rng):
    w = rng.uniform(-1.0, 1.0, d)
    if kind == "degenerate":            # repeated eigenvalues on both sides of zero
        w = np.round(w * 2.0) / 2.0 + 0.25
    elif kind == "zero":                # most of the spectrum at zero
        w[: (2 * d) // 3] = 0.0
    elif kind == "positive":
        w = np.abs(w) + 0.1
    elif kind == "negative":
        w = -np.abs(w) - 0.1
    return w


def _sequence(kind, d, rng):
    """Blocks that a solve would meet one after the other."""
    Q = np.linalg.qr(rng.standard_normal((d, d)))[0]
    U = (Q * _spectrum(kind, d, rng)) @ Q.T
    out = [U]
    for step in (1e-2, 1e-3, 1e-5, 1e-9, 0.0, 1e-7):
        G = rng.standard_normal((d, d)) / np.sqrt(d)
        U = U + step * (G + G.T)
        out.append(U)
    Q = np.linalg.qr(rng.standard_normal((d, d)))[0]
    out.append((Q * _spectrum(kind, d, rng)) @ Q.T)  # nothing in common with the one before
    out.append(np.zeros((d, d)))
    out.append(out[1])
    return out


SMALL = [1, 2, 3, 4, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64]


@pytest.mark.parametrize("kind", ["plain", "degenerate", "zero", "positive", "negative"])
@pytest.mark.parametrize("dims", [SMALL, [5, 16, 1], [20, 32, 7]], ids=["to64", "to16", "to32"])
def test_projection_sequence(kind, dims):
    _check(kind, dims)


@pytest.mark.parametrize("kind", ["plain", "positive", "negative"])
@pytest.mark.parametrize("dims", [[65, 96, 97, 128], [129, 192, 193, 224], [225, 256, 257], [2, 300, 64, 417]],
                         ids=["to128", "to224", "to257", "mixed"])
def test_projection_sequence_large(kind, dims):
    _check(kind, dims)


def _turning_sequence(kind, d, rng):
    """A spectrum with groups of equal (or nearly equal) eigenvalues whose
    eigenvectors turn a little from block to block: the refinement meets
    clusters whose columns are not orthogonal yet."""
    w = rng.uniform(-1.0, 1.0, d)
    third = max(1, d // 3)
    w[:third] = 0.7
    w[third:2 * third] = -0.4 if kind != "zero" else 0.0
    if kind == "spread":                # apart by less than the cluster threshold
        w[:third] += 1e-9 * rng.uniform(-1.0, 1.0, third)
    Q = np.linalg.qr(rng.standard_normal((d, d)))[0]
    out = []
    for angle in (0.0, 1e-3, 1e-4, 3e-5, 1e-5, 3e-6, 1e-6, 1e-7, 0.0):
        K = angle * rng.standard_normal((d, d)) / np.sqrt(d)
        Q = Q @ scipy.linalg.expm(K - K.T)
        U = (Q * w) @ Q.T
        out.append(0.5 * (U + U.T))
    return out


@pytest.mark.parametrize("kind", ["equal", "spread", "zero"])
@pytest.mark.parametrize("dims", [[3, 6, 9, 16], [17, 33, 48, 64], [65, 96, 160, 224], [230, 288]],
                         ids=["to16", "to64", "to224", "to288"])
def test_projection_while_clusters_turn(kind, dims):
    # a step is accepted with corrections of up to 2e-7 (3e-8 up to 64 rows) and
    # leaves their square, d of which add up in an element
    rng = np.random.default_rng([len(dims), len(kind), 2])
    _check_sequences(kind, dims, [_turning_sequence(kind, d, rng) for d in dims],
                     extra=lambda d: d * (2e-7 if d > 64 else 3e-8) ** 2)


def _degenerate_sequence(kind, d, rng):
    """Blocks whose eigenvalues are equal in large groups, diagonal and turned,
    some of them after a zero block (whose eigenvalues are the guess then)."""
    def spectrum():
        if kind == "ends":          # one eigenvalue at each end, two groups between
            w = np.zeros(d)
            w[1:1 + d // 2] = 1.0
            w[0] = 2.0
            w[-1] = -2.0 if d > 2 else w[-1]
        elif kind == "integers":    # the cost of a caller's map, say
            w = rng.integers(-2, 2, d).astype(float)
            w[0] = 2.0
        elif kind == "one":         # one positive, many zero, many negative
            w = -rng.uniform(0.1, 1.0, d)
            w[: (d + 1) // 2] = 0.0
            w[0] = 1.0
        else:                       # low rank
            w = np.zeros(d)
            w[: max(1, d // 20)] = rng.uniform(0.5, 1.0, max(1, d // 20))
        return rng.permutation(w)

    def turned(w):
        Q = np.linalg.qr(rng.standard_normal((d, d)))[0]
        U = (Q * w) @ Q.T
        return 0.5 * (U + U.T)

    return [np.diag(spectrum()), np.zeros((d, d)), turned(spectrum()), np.zeros((d, d)), np.diag(spectrum()),
            turned(spectrum())]


@pytest.mark.parametrize("kind", ["ends", "integers", "one", "rank"])
@pytest.mark.parametrize("dims", [SMALL, [13, 14, 15, 16] * 8, [17, 31, 32, 33, 47, 48, 49, 63, 64],
                                  [65, 96, 128, 224], [225, 257, 300, 417]],
                         ids=["small", "to16", "to64", "to224", "to417"])
def test_projection_of_degenerate_blocks(kind, dims):
    rng = np.random.default_rng([len(dims), len(kind), 1])
    _check_sequences(kind, dims, [_degenerate_sequence(kind, d, rng) for d in dims])


def test_cluster_of_a_large_block_is_shared():
    """397 equal eigenvalues of 417: 80 ms with a workgroup orthogonalising their
    vectors; one thread (some 300 000 dependent column passes) takes above ten
    seconds."""
    d, rng = 417, np.random.default_rng(5)
    U = _degenerate_sequence("rank", d, rng)[2]
    S = BPSDPSolver(d * d, 1, options(e_convergence=1e-30, r_convergence=1e-30, maxiter=10 ** 6))
    S.set_mu(1.0)
    for cost in (np.eye(d), -U):  # the first call also sets up
        t0 = time.perf_counter()
        S.solve(np.zeros(d * d), np.zeros(1), cost.ravel(), [d], 1, lambda u: np.zeros(1), lambda y: np.zeros(d * d))
        seconds = time.perf_counter() - t0
    S.close()
    assert seconds < 2.0, seconds


def _check(kind, dims):
    rng = np.random.default_rng([len(dims), len(kind)])
    _check_sequences(kind, dims, [_sequence(kind, d, rng) for d in dims])


def _check_sequences(kind, dims, seqs, extra=lambda d: 0.0):
    n = sum(d * d for d in dims)
    S = BPSDPSolver(n, 1, options(e_convergence=1e-30, r_convergence=1e-30, maxiter=10 ** 6))
    zero_a = lambda u: np.zeros(1)
    zero_at = lambda y: np.zeros(n)
    S.set_mu(1.0)
    for k in range(len(seqs[0])):
        U = [s[k] for s in seqs]
        x = np.zeros(n)
        c = -np.concatenate([u.ravel() for u in U])
        S.solve(x, np.zeros(1), c, dims, 1, zero_a, zero_at)
        mu = S.get_mu()
        assert S.status()["status_bits"] == 0
        off = 0
        for d, u in zip(dims, U):
            scale = max(np.abs(np.linalg.eigvalsh(u)).max(), 1e-300)
            err = np.abs(mu * x[off:off + d * d].reshape(d, d) - _positive_part(u)).max() / scale
            assert err < 100 * EPS * max(d, 10) + extra(d), (kind, k, d, err)
            off += d * d
    S.close()
