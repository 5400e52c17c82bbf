"""Batches of more than 65,536 instances: small symmetry-free sectors with
and without the split row gather, the latter's tables for the few that use it."""
import numpy as np
import pytest

import spined
from spined import batch, internal, lattice

pytestmark = pytest.mark.gpu


def _op(n, delta):
    basis = spined.mk_basis(spined.mk_group([]), n, n // 2, 1)
    spined.build_basis(basis)
    J = np.random.default_rng(n).uniform(0.8, 1.2, n)
    return spined.mk_operator(basis, [spined.mk_interaction(lattice.xxz_matrix(delta, J[b]), [[b, (b + 1) % n]])
                                      for b in range(n)])


def test_many_instances():
    small = _op(8, 0.4)                          # 35 rows: row by row
    large = [_op(12, d) for d in (0.3, 0.9)]     # 462 rows: one group each
    assert internal.get_number_states(small.basis) == 35
    ref = [spined.eigsh(op, k=1, tol=1e-11, want_vectors=False).evals[0] for op in [small] + large]
    count = (1 << 16) + 8
    r = batch.batch_eigsh([small] * count + large * 4, tol=1e-9)
    assert r["status"] == 0
    # a residual of 1e-9 puts an energy far closer than 1e-10
    want = np.array([ref[0]] * count + ref[1:] * 4)
    assert np.max(np.abs(r["evals"] - want)) <= 1e-10 * np.max(np.abs(want))
    # no split instance at all, and nothing but
    assert abs(batch.batch_eigsh([small], tol=1e-9)["evals"][0] - ref[0]) <= 1e-10 * abs(ref[0])
    e = batch.batch_eigsh(large, tol=1e-9)["evals"]
    assert np.max(np.abs(e - np.array(ref[1:]))) <= 1e-10 * np.max(np.abs(e))
