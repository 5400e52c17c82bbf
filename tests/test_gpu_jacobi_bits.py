"""Projected-matrix eigensolver, bit for bit against its definition: a cyclic
Jacobi iteration in round-robin order that rotates all columns of a round and
then all rows, and orders the result by a selection sort.  Restarts carry the
rounding on, so the sign of a block solver's eigenvector depends on it."""
import numpy as np
import pytest

import spined
from spined import internal


def _wave_sum(v):
    """Sum of 64 values by halving."""
    v = v.copy()
    for off in (32, 16, 8, 4, 2, 1):
        v[:off] = v[:off] + v[off:2 * off]
    return v[0]


def _total(values, mp):
    """Sum over the matrix by 256 threads, strided, then waves in order."""
    lanes = np.zeros(256)
    flat = np.zeros(-(-mp * mp // 256) * 256)
    flat[:mp * mp] = values.ravel()
    for part in flat.reshape(-1, 256):
        lanes = lanes + part
    w = [_wave_sum(lanes[64 * i:64 * i + 64]) for i in range(4)]
    return (w[0] + w[1]) + (w[2] + w[3])


def _jacobi(T, sweeps=40):
    m = len(T)
    mp = m + (m & 1)
    A = np.zeros((mp, mp))
    A[:m, :m] = 0.5 * (T + T.T)
    V = np.eye(mp)
    diagonal = np.eye(mp, dtype=bool)
    for _ in range(sweeps):
        off = _total(np.where(diagonal, 0.0, A * A), mp)
        dia = _total(np.where(diagonal, A * A, 0.0), mp)
        if off <= 1e-30 * (dia + off) or off == 0.0:
            break
        for step in range(mp - 1):
            player = [0] + [1 + (pos - 1 + step) % (mp - 1) for pos in range(1, mp)]
            pairs = [sorted((player[k], player[mp - 1 - k])) for k in range(mp // 2)]
            P, Q = np.array(pairs).T
            apq = A[P, Q]
            some = apq != 0.0
            tau = (A[Q, Q] - A[P, P]) / (2.0 * np.where(some, apq, 1.0))
            t = np.where(tau >= 0.0, 1.0, -1.0) / (np.abs(tau) + np.sqrt(1.0 + tau * tau))
            c = np.where(some, 1.0 / np.sqrt(1.0 + t * t), 1.0)
            s = np.where(some, t * (1.0 / np.sqrt(1.0 + t * t)), 0.0)
            for M in (A, V):
                a, b = M[:, P], M[:, Q]
                M[:, P], M[:, Q] = c * a - s * b, s * a + c * b
            a, b = A[P], A[Q]
            A[P], A[Q] = c[:, None] * a - s[:, None] * b, s[:, None] * a + c[:, None] * b
    d = np.diag(A)
    order = list(range(m))
    for i in range(m):
        best = i
        for j in range(i + 1, m):
            if d[order[j]] < d[order[best]]:
                best = j
        order[i], order[best] = order[best], order[i]
    return d[order], V[:m, order].T


def _matrix(kind, m):
    rng = np.random.default_rng(1000 + m)
    if kind == "dense":
        a = rng.normal(size=(m, m))
        return 0.5 * (a + a.T)
    if kind == "restart":  # kept Ritz values, their couplings, new Lanczos steps
        a = np.diag(np.sort(rng.uniform(-40, -20, m)))
        k = m // 2
        a[:k, k] = a[k, :k] = rng.normal(size=k) * 1e-3
        for j in range(k, m - 1):
            a[j, j + 1] = a[j + 1, j] = rng.uniform(3, 9)
        return a
    # equal eigenvalues that no rotation touches
    return np.diag(np.array([2.0, 2.0, 1.0, 3.0, 1.0, 2.0] * 11)[:m])


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 2, 8, 23, 24, 31, 32, 33, 64])
@pytest.mark.parametrize("kind", ["dense", "restart", "equal"])
def test_bits(kind, m):
    T = _matrix(kind, m)
    evals, vecs = internal.debug_eigh(T)
    ref_evals, ref_vecs = _jacobi(T)
    np.testing.assert_array_equal(evals, ref_evals)
    np.testing.assert_array_equal(vecs, ref_vecs)


@pytest.mark.parametrize("m", [2, 23, 64])
def test_definition_is_an_eigensolver(m):
    T = _matrix("dense", m)
    e, v = _jacobi(T)
    assert np.max(np.abs(T @ v.T - v.T * e)) <= 1e-13 * m * np.max(np.abs(T))
    np.testing.assert_allclose(e, np.linalg.eigvalsh(T), atol=1e-13 * m)


def test_size_is_checked():
    with pytest.raises(Exception):
        internal.debug_eigh(np.eye(65))
    with pytest.raises(ValueError):
        internal.debug_eigh(np.ones((2, 3)))
