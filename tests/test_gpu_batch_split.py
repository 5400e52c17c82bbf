"""Batched solver with the split row gather at its edges: one group (12 sites),
a few (14, 16), bonds in mixed order, and team sizes from one workgroup to the
largest; each ground energy against the single solver's to 1e-10 (both solve
to a residual of 1e-9, so the energies are far closer)."""
import numpy as np
import pytest

import spined
from spined import batch, lattice

pytestmark = pytest.mark.gpu


def _op(n, w, z, bonds, rng):
    basis = spined.mk_basis(spined.mk_group([]), n, w, z)
    spined.build_basis(basis)
    return spined.mk_operator(basis, [spined.mk_interaction(lattice.xxz_matrix(0.5, j), [b])
                                      for j, b in zip(rng.uniform(0.8, 1.2, len(bonds)), bonds)])


@pytest.mark.parametrize("rows,team", [(None, None), (1024, 128), (32768, 1)])
def test_batch_split_edges(monkeypatch, rows, team):
    if rows:
        monkeypatch.setenv("SPINED_BATCH_ROWS_PER_MEMBER", str(rows))
        monkeypatch.setenv("SPINED_BATCH_MAX_TEAM", str(team))
    rng = np.random.default_rng(11)
    ops = []
    for n, w, z in ((12, 6, 1), (12, 6, -1), (13, 6, None), (14, 7, 1), (16, 8, -1), (16, 8, None),
                    (18, 9, 1), (20, 10, 1), (20, 3, None)):
        order = rng.permutation(n)
        ops.append(_op(n, w, z, lattice.ring_bonds(n), rng))
        ops.append(_op(n, w, z, [lattice.ring_bonds(n)[k] for k in order], rng))
    print("rows", rows, "team", team, flush=True)
    r = batch.batch_eigsh(ops, tol=1e-9)
    assert r["status"] == 0
    for op, e in zip(ops, r["evals"]):
        s = spined.eigsh(op, k=1, tol=1e-10, want_vectors=False)
        assert s.status == 0
        assert abs(e - s.evals[0]) <= 1e-10 * max(1.0, abs(s.evals[0]))
