"""Orthogonalisation sums over any number of basis vectors: the Ritz pairs of a
sector against the oracle at basis sizes on both sides of the kernels' widths
(8, 16, 24, 32 vectors, one more and one fewer), with a row count that leaves
lanes and workgroups partly empty."""
import numpy as np
import pytest

from helpers import Spec, engine, oracle
from spined import lattice, solver


@pytest.mark.gpu
@pytest.mark.parametrize("basis", [7, 8, 9, 15, 16, 17, 24, 25, 31, 32])
def test_basis_widths(basis):
    n = 14
    spec = Spec(n, 7, 1, lattice.ring_symmetries(n, 0, 0), [(lattice.HEISENBERG, lattice.ring_bonds(n))])
    b, op = engine(spec)
    o = oracle(spec)
    H = np.column_stack([o.matvec(e) for e in np.eye(o.dimension)])
    ref = np.linalg.eigvalsh((H + H.T) / 2)[0]
    r = solver.eigsh(op, k=1, tol=1e-10, seed=3, max_basis_size=basis)
    # a residual of 1e-10 |theta| bounds the eigenvalue's error by as much
    assert abs(r.evals[0] - ref) <= 2e-10 * abs(ref)
