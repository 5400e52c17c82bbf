"""Row schedule of complex operators: built when their gather cache is due and
not before (one tile is 4096 rows), with the same sums at every use."""
import numpy as np
import pytest

import spined
from spined import internal
from helpers import engine, ring

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,rows_of_a_tile", [(16, 1, False), (18, 5, False), (20, 3, True)])
def test_schedule_comes_with_the_cache(n, k, rows_of_a_tile):
    basis, op = engine(ring(n, k=k, p=None, z=None, name="ring"))
    D = internal.get_number_states(basis)
    assert (D >= 4096) == rows_of_a_tile
    x = np.random.default_rng(n).normal(size=(2, D))
    x = x[0] + 1j * x[1]
    _, plain = engine(ring(n, k=k, p=None, z=None, name="ring"))
    internal.set_gather_cache(plain, 0)
    ref = spined.apply(plain, x)
    for use in (1, 2, 3):
        np.testing.assert_array_equal(spined.apply(op, x), ref)
        assert internal.gather_cache(op) == (1 if use > 1 else 0)
        assert internal.schedule(op) == (1 if rows_of_a_tile and use > 1 else 0)
    # asked for, it is built at the first use
    _, asked = engine(ring(n, k=k, p=None, z=None, name="ring"))
    internal.set_schedule(asked, 1)
    np.testing.assert_array_equal(spined.apply(asked, x), ref)
    assert internal.schedule(asked) == 1
