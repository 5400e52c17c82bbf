"""Gather cache beyond one real vector of a bond operator: complex sectors and
complex matrices, operators of many bonds or templates, coefficient classes
that do not fit in the entries, partly filled tiles of the row schedule.  The
cached sums must equal the matrix-free ones bit for bit; when an automatic
cache is built."""
import numpy as np
import pytest

import spined
from spined import lattice
from helpers import Spec, engine, ring

pytestmark = pytest.mark.gpu


def _disordered(spec, seed):
    rng = np.random.default_rng(seed)
    n = spec.n
    spec.terms = [(lattice.xxz_matrix(0.7, J), [[b, (b + 1) % n]])
                  for b, J in enumerate(rng.uniform(0.8, 1.2, n))]
    spec.name += "_disordered"
    return spec


def _all_pairs(n, name):
    pairs = [[i, j] for i in range(n) for j in range(i + 1, n)]
    s = ring(n, k=0, p=0, z=1 if n % 2 == 0 else None, name=name)
    s.terms = [(lattice.HEISENBERG, pairs)]
    return s


def _three_site(n):
    rng = np.random.default_rng(3)
    m = rng.normal(size=(8, 8)) + 1j * rng.normal(size=(8, 8))
    s = ring(n, k=1, p=None, z=None, w=None, name="ring%d_k1_three_site" % n)
    s.terms = [((m + m.conj().T).tolist(), [[i, (i + 1) % n, (i + 2) % n] for i in range(n)])]
    return s


def _dm(n):
    # Dzyaloshinskii-Moriya bonds: complex matrix elements
    s = ring(n, k=3, p=None, z=None, name="ring%d_k3_dm" % n)
    m = np.zeros((4, 4), dtype=complex)
    m[1, 2], m[2, 1] = 0.4j, -0.4j
    s.terms.append((m.tolist(), [[i, (i + 1) % n] for i in range(n)]))
    return s


CASES = [
    ring(18, k=5, p=None, z=None, name="ring18_k5"),
    ring(16, k=3, p=None, z=-1, name="ring16_k3_z-"),
    _dm(14),
    _three_site(9),
    _all_pairs(18, "ring18_all_pairs"),          # 153 bonds
    _all_pairs(25, "ring25_all_pairs"),          # 300 bonds, five tiles and a part
    ring(24, k=0, p=0, z=1, name="ring24"),      # seven tiles and a part
    Spec(12, 6, None, [([(i + 4) % 12 for i in range(12)], 1)],
         [(lattice.HEISENBERG, lattice.ring_bonds(12))], "ring12_translation_by_4_k1"),
    _disordered(ring(16, k=None, p=None, z=1, name="chain16"), 5),
]


def _vector(D, dtype, seed):
    rng = np.random.default_rng(seed)
    x = rng.uniform(-1, 1, D)
    if np.dtype(dtype).kind == "c":
        x = x + 1j * rng.uniform(-1, 1, D)
    return x.astype(dtype)


def _same(op, D, dtypes):
    for dt in dtypes:
        x = _vector(D, dt, 7)
        spined.set_gather_cache(op, 0)
        y0 = spined.apply(op, x)
        spined.set_gather_cache(op, 1)
        y1 = spined.apply(op, x)
        assert spined.gather_cache(op) == 1
        np.testing.assert_array_equal(y1, y0)
        spined.set_gather_cache(op, 0)


@pytest.mark.parametrize("spec", CASES, ids=lambda s: s.name)
def test_cached_equals_matrix_free(spec):
    print("case", spec.name, flush=True)
    basis, op = engine(spec)
    D = spined.get_number_states(basis)
    real = (np.float64, np.float32) if op.is_real else ()
    for mode in (-1, 0):
        spined.set_schedule(op, mode)
        _same(op, D, real + (np.complex128, np.complex64))


def test_classes_beside_the_entries():
    """30 couplings x 30 momenta and 23 index bits exceed an entry."""
    spec = _disordered(ring(30, k=7, p=None, z=None, name="ring30_k7"), 9)
    basis, op = engine(spec)
    _same(op, spined.get_number_states(basis), (np.complex128,))


def test_automatic_cache_of_small_bases():
    basis, op = engine(ring(20, k=0, p=0, z=1))
    D = spined.get_number_states(basis)
    x = _vector(D, np.float64, 1)
    y = [spined.apply(op, x)]
    assert spined.gather_cache(op) == 0  # a single application: none
    for _ in range(2):
        y.append(spined.apply(op, x))
        assert spined.gather_cache(op) == 1
    np.testing.assert_array_equal(y[0], y[1])
    np.testing.assert_array_equal(y[0], y[2])
    # a tiny basis never
    b2, op2 = engine(ring(10, k=0, p=0, z=1))
    x2 = _vector(spined.get_number_states(b2), np.float64, 2)
    for _ in range(3):
        spined.apply(op2, x2)
    assert spined.gather_cache(op2) == 0
