"""Matvecs of solves of small sectors (below 2^20 rows).  Far from convergence the
estimates are looked at between cycles only: ordinary solves take the matvecs of
a check at every fourth step, and a start vector that exhausts its Krylov space
inside a cycle goes on to the end of it."""
import numpy as np
import pytest

import spined
from helpers import engine, ring
from spined import internal, lattice, solver

pytestmark = pytest.mark.gpu

CYCLE = 24  # basis size of one level


@pytest.mark.parametrize("n,levels,precision,matvecs", [
    (14, 1, "fp64", 29), (16, 1, "fp64", 37), (18, 1, "fp64", 41), (20, 1, "fp64", 49),
    (24, 1, "fp64", 53), (16, 4, "fp64", 62), (20, 4, "fp64", 78), (24, 4, "fp64", 96),
    (16, 1, "mixed", 41), (20, 1, "mixed", 57)])
def test_same_as_every_fourth_step(n, levels, precision, matvecs):
    # Delta and the seed of the solves recorded with a check at every fourth step
    delta = float(np.random.default_rng(1).uniform(0.5, 1.5))
    _, op = engine(ring(n, k=0, p=0, z=1, matrix=lattice.xxz_matrix(delta)))
    r = solver.eigsh(op, k=levels, tol=1e-10, precision=precision, seed=1)
    assert r.status == 0
    assert r.stats["matvecs"] == matvecs


@pytest.mark.parametrize("few", [1, 2, 3, 7, 9, 11])
def test_short_krylov_space(few):
    _, op = engine(ring(18, k=0, p=0, z=1))
    D = internal.get_number_states(op.basis)
    H = spined.apply(op, np.asfortranarray(np.eye(D)))
    e, v = np.linalg.eigh(0.5 * (H + H.T))
    r = solver.eigsh(op, k=1, tol=1e-10, start_vector=v[:, :few].sum(axis=1))
    assert r.status == 0 and abs(r.evals[0] - e[0]) <= 2e-10 * abs(e[0])
    # the cycle, the steps after the breakdown once more, one for the residual
    assert r.stats["matvecs"] <= CYCLE + (CYCLE - few) + 1
