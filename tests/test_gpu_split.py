"""Split row gather of symmetry-free weight sectors (split.hpp) against the
gather cache (bit for bit) and, on sampled rows, against H x written out with
integer arithmetic here; bonds inside the low part, inside the high part and
across the cut, in mixed order, with and without the flip."""
import numpy as np
import pytest

import spined
from spined import lattice

pytestmark = pytest.mark.gpu


def _bonds(n, kind, rng):
    if kind == "ring":
        return lattice.ring_bonds(n)
    pairs = [[i, j] for i in range(n) for j in range(n) if i != j]
    return [pairs[k] for k in rng.choice(len(pairs), 40, replace=False)]


# 23 sites: the smallest that takes the path; 26 at and below half filling;
# 27 has the deeper cut
CASES = [(23, 11, None, "ring"), (24, 12, 1, "ring"), (24, 12, -1, "mixed"), (25, 13, None, "mixed"),
         (26, 13, 1, "mixed"), (26, 9, None, "ring"), (27, 13, None, "ring")]


@pytest.mark.parametrize("n,w,z,kind", CASES)
def test_split_matvec(n, w, z, kind):
    print("case", n, w, z, kind, flush=True)
    rng = np.random.default_rng(n * 100 + w)
    basis = spined.mk_basis(spined.mk_group([]), n, w, z)
    spined.build_basis(basis)
    bonds = _bonds(n, kind, rng)
    J = rng.uniform(0.5, 1.5, len(bonds))
    J[1] = 0.0
    delta = rng.uniform(-1, 1, len(bonds))
    ms = [lattice.xxz_matrix(d, j) for d, j in zip(delta, J)]
    op = spined.mk_operator(basis, [spined.mk_interaction(m, [b]) for m, b in zip(ms, bonds)])
    D = spined.get_number_states(basis)
    assert D >= 1 << 20
    x = rng.uniform(-1, 1, D)
    out = {}
    for mode in (-1, 1):
        spined.set_gather_cache(op, mode)
        out[mode] = [spined.apply(op, x), spined.apply(op, x.astype(np.float32))]
        # the automatic mode takes the split path where its groups are large
        if mode == -1 and not (n == 26 and w == 9):
            assert spined.gather_cache(op) == 0
    np.testing.assert_array_equal(out[-1][0], out[1][0])
    np.testing.assert_array_equal(out[-1][1], out[1][1])
    reps = spined.basis_get_states(basis)
    full = np.uint64((1 << n) - 1)
    scale = np.max(np.abs(out[1][0]))
    for i in np.concatenate([[0, 1, D - 1], rng.integers(0, D, 200)]):
        r, y = reps[i], 0.0
        for m, (a, b) in zip(ms, bonds):
            anti = ((int(r) >> a) ^ (int(r) >> b)) & 1
            y += (m[1][1] if anti else m[0][0]) * x[i]
            if anti:
                t = r ^ np.uint64((1 << a) | (1 << b))
                sign = 1.0
                if z and (int(t) >> (n - 1)) & 1:
                    t, sign = full ^ t, float(z)
                y += sign * m[1][2] * x[np.searchsorted(reps, t)]
        assert abs(y - out[-1][0][i]) <= 1e-13 * scale


def test_split_solve_matches_cache():
    basis = spined.mk_basis(spined.mk_group([]), 24, 12, 1)
    spined.build_basis(basis)
    J = np.random.default_rng(3).uniform(0.8, 1.2, 24)
    op = spined.mk_operator(basis, [spined.mk_interaction(lattice.xxz_matrix(0.6, J[b]), [[b, (b + 1) % 24]])
                                    for b in range(24)])
    e = []
    for mode in (-1, 1):
        spined.set_gather_cache(op, mode)
        r = spined.eigsh(op, k=1, tol=1e-10, want_vectors=False)
        assert r.status == 0
        e.append((r.evals[0], r.stats["matvecs"]))
    assert e[0] == e[1]
