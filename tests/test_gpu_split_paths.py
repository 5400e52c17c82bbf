"""Which kernels serve symmetry-free sectors: the split row gather by itself, the
orbit and index kernels with the gather cache turned off, the cache when asked
for, and the same bits from all three."""
import numpy as np
import pytest

import spined
from spined import internal, lattice

pytestmark = pytest.mark.gpu


def _system(n, w, z, seed):
    """Bonds between random sites, and the ring's in order, of random strengths."""
    rng = np.random.default_rng(seed)
    basis = spined.mk_basis(spined.mk_group([]), n, w, z)
    spined.build_basis(basis)
    pairs = [[i, j] for i in range(n) for j in range(n) if i != j]
    bonds = [pairs[k] for k in rng.choice(len(pairs), 30, replace=False)] + lattice.ring_bonds(n)
    terms = [spined.mk_interaction(lattice.xxz_matrix(d, j), [b])
             for b, d, j in zip(bonds, rng.uniform(-1, 1, len(bonds)), rng.uniform(0.5, 1.5, len(bonds)))]
    return spined.mk_operator(basis, terms), rng


# shallow and deep cut (12 and 13 low sites), with and without the flip, weights
# away from half filling that still take the path
@pytest.mark.parametrize("n,w,z", [(24, 12, -1), (26, 11, None), (27, 13, None), (28, 14, -1), (28, 14, 1)])
def test_paths_agree(n, w, z):
    print("case", n, w, z, flush=True)
    op, rng = _system(n, w, z, n * 10 + w)
    x = rng.uniform(-1, 1, internal.get_number_states(op.basis))
    for dtype in (np.float64, np.float32):
        xt = x.astype(dtype)
        out = {}
        for mode, path in ((-1, 2), (0, 0), (1, 1)):
            internal.set_gather_cache(op, mode)
            out[mode] = spined.apply(op, xt)
            assert internal.debug_matvec_path(op) == path
        np.testing.assert_array_equal(out[0], out[-1])
        np.testing.assert_array_equal(out[0], out[1])
        internal.set_gather_cache(op, 0)  # drops the cache
