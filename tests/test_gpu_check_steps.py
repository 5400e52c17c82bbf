"""Matvecs of solves of sectors below 2^20 rows are those of a convergence check at
every fourth step: recorded with such a solver, for sectors on both sides of the
size from which checks far from convergence are left out (4,096 rows), and for
start vectors that exhaust their Krylov space inside a cycle."""
import numpy as np
import pytest

import spined
from helpers import Spec, engine, ring
from spined import internal, lattice, solver

pytestmark = pytest.mark.gpu


def _system(kind, n, w, seed):
    # Delta and the seed of the recorded solves
    delta = float(np.random.default_rng(seed).uniform(0.5, 1.5))
    m, z = lattice.xxz_matrix(delta), 1 if 2 * w == n else None
    if kind == "square":
        side = int(round(n ** 0.5))
        return engine(Spec(n, w, z, lattice.square_symmetries(side), [(m, lattice.square_bonds(side))]))[1]
    return engine(ring(n, k=0, p=0, z=z, w=w, matrix=m))[1]


@pytest.mark.parametrize("kind,n,w,seed,levels,precision,basis,matvecs", [
    ("ring", 13, 6, 0, 1, "fp64", 40, 37), ("ring", 14, 6, 0, 1, "mixed", 0, 33),
    ("ring", 14, 6, 0, 1, "fp64", 40, 29), ("ring", 14, 7, 0, 1, "mixed", 0, 33),
    ("ring", 14, 7, 1, 1, "fp64", 0, 29), ("ring", 16, 8, 0, 1, "fp64", 40, 37),
    ("ring", 16, 8, 1, 4, "fp64", 0, 62), ("ring", 18, 8, 2, 1, "fp64", 40, 37),
    ("square", 16, 8, 0, 1, "mixed", 0, 37), ("square", 16, 7, 1, 1, "mixed", 0, 33),
    ("square", 16, 6, 2, 1, "fp64", 40, 29), ("ring", 20, 10, 1, 4, "fp64", 0, 78),
    ("ring", 22, 11, 1, 1, "fp64", 0, 49), ("ring", 24, 12, 1, 1, "fp64", 40, 53),
    ("ring", 24, 12, 1, 4, "fp64", 0, 96)])
def test_same_as_every_fourth_step(kind, n, w, seed, levels, precision, basis, matvecs):
    op = _system(kind, n, w, seed)
    r = solver.eigsh(op, k=levels, tol=1e-10, precision=precision, seed=seed, max_basis_size=basis)
    assert r.status == 0
    assert r.stats["matvecs"] == matvecs


# steps of the Krylov space, matvecs; of one to three steps the breakdown is read
# at the first check and the steps to it are taken again
@pytest.mark.parametrize("few,matvecs", [(1, 8), (2, 7), (3, 6), (7, 13), (9, 18), (11, 17)])
def test_short_krylov_space(few, matvecs):
    _, op = engine(ring(18, k=0, p=0, z=1))
    D = internal.get_number_states(op.basis)
    H = spined.apply(op, np.asfortranarray(np.eye(D)))
    e, v = np.linalg.eigh(0.5 * (H + H.T))
    r = solver.eigsh(op, k=1, tol=1e-10, start_vector=v[:, :few].sum(axis=1))
    assert r.status == 0 and abs(r.evals[0] - e[0]) <= 2e-10 * abs(e[0])
    # eigenvectors of the host's LAPACK: its rounding moves a breakdown by a check
    assert r.stats["matvecs"] <= matvecs + 4
