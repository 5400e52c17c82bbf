"""Row-key orbits of tori (representative test and scans that look only at the
translations with the least row on top) against the scan over every element's
program and the oracle, on the CPU."""
import numpy as np
import pytest

import pyoracle as O
import spined
from test_abi_cpu import _torus_gens


@pytest.mark.parametrize("l1,l2,kx,ky,z,points", [
    (5, 2, 0, 0, None, 1),   # five-bit rows: row keys only with point elements
    (5, 2, 0, 0, 1, 2),
    (6, 2, 3, 0, -1, 1),
    (6, 2, 2, 1, None, 1),   # complex phases
    (7, 2, 0, 1, 1, 2),
    (8, 2, 0, 0, 1, 2),      # the longest rows with keys
    (8, 2, 4, 1, -1, 1),
    (9, 2, 0, 0, 1, 2),      # beyond them: the scan
])
def test_every_state_of_a_torus(l1, l2, kx, ky, z, points):
    n = l1 * l2
    gens = _torus_gens(l1, l2, kx, ky, points == 2)
    b = spined.mk_basis(spined.mk_group([spined.mk_symmetry(p, s) for p, s in gens]), n, None, z)
    assert spined.torus_shape(b)[0] in (l1, l2)
    # all-equal rows, empty rows and their complements included: every state
    st = np.arange(1 << n, dtype=np.uint64)
    key, scan = spined.debug_orbit(b, st, 0), spined.debug_orbit(b, st, 2)
    for q in (0, 2, 3):
        np.testing.assert_array_equal(key[q], scan[q])
    np.testing.assert_array_equal(spined.debug_orbit(b, st, 3)[0], scan[0])
    v = key[3].astype(bool)
    np.testing.assert_array_equal(key[1][v], scan[1][v])
    o = O.System(n, None, z, gens)
    for x in range(0, 1 << n, 257):
        r = o.orbit(x)
        assert (key[0][x], key[2][x], key[3][x]) == (r[0], r[2], r[3])


@pytest.mark.gpu
@pytest.mark.parametrize("l1,l2,kx,ky,z,reflect", [
    (3, 4, 0, 0, 1, True), (4, 4, 1, 2, None, False), (5, 3, 0, 0, None, True), (6, 3, 3, 0, -1, False),
    (7, 2, 0, 1, None, False), (8, 2, 0, 0, 1, True), (8, 2, 4, 1, -1, False)])
def test_build_by_row_keys(l1, l2, kx, ky, z, reflect):
    """The representative test keeps exactly the oracle's basis."""
    n = l1 * l2
    gens = _torus_gens(l1, l2, kx, ky, reflect)
    w = n // 2 if n % 2 == 0 else None
    b = spined.mk_basis(spined.mk_group([spined.mk_symmetry(p, s) for p, s in gens]), n, w, z)
    spined.build_basis(b)
    ref = O.System(n, w, z, gens)
    ref.build()
    np.testing.assert_array_equal(spined.basis_get_states(b), ref.basis()[0])
