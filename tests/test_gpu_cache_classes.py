"""An operator of more coefficient classes than the gather cache numbers: served by
the matrix-free kernels in every mode, asked for or not."""
import numpy as np
import pytest

import spined
from spined import internal, lattice

pytestmark = pytest.mark.gpu


def test_too_many_classes_stay_matrix_free():
    n, terms = 12, 5500
    # bonds across the ring, one strength per term: six units each, and twelve
    # phases per strength
    across = [[i, i + n // 2] for i in range(n // 2)]
    assert 6 * terms <= 65535 and 12 * terms > 65536
    J = np.random.default_rng(1).uniform(0.5, 1.5, terms)
    basis = spined.mk_basis(spined.mk_group([spined.mk_symmetry([(i + 1) % n for i in range(n)], 1)]), n, 6, None)
    spined.build_basis(basis)
    ops = [spined.mk_operator(basis, [spined.mk_interaction(lattice.xxz_matrix(0.5, j), across) for j in strengths])
           for strengths in (J, [J.sum()])]
    D = internal.get_number_states(basis)
    assert D > 64  # smaller bases have no automatic cache
    rng = np.random.default_rng(2)
    x = rng.normal(size=D) + 1j * rng.normal(size=D)
    # one bond of the summed strength: the same operator to rounding
    ref = spined.apply(ops[1], x)
    for mode in (-1, 1, 0):
        internal.set_gather_cache(ops[0], mode)
        for _ in range(3):
            y = spined.apply(ops[0], x)
            # sums of 5,500 terms of both signs: eps times terms times their size
            assert np.max(np.abs(y - ref)) <= 2e-16 * terms * J.sum() * np.max(np.abs(x))
            assert internal.gather_cache(ops[0]) == 0 and internal.debug_matvec_path(ops[0]) == 0
