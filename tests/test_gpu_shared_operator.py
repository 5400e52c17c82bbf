"""One fresh operator applied by several threads at once: the first calls build
its gather cache and row schedule between them, and every result, during that
and later, has the bits of the matrix-free kernels."""
import threading

import numpy as np
import pytest

import spined
from spined import internal, lattice
from helpers import Spec, engine, ring

pytestmark = pytest.mark.gpu

# a momentum sector of several schedule tiles, and a real operator of more bonds
# than the matrix-free kernels schedule rows for
PAIRS = [[i, j] for i in range(22) for j in range(i + 1, 22)]
CASES = {
    "complex": ring(20, k=3, p=None, z=None, name="ring"),
    "bonds": Spec(22, 11, 1, lattice.ring_symmetries(22, 0, 0), [(lattice.xxz_matrix(0.7), PAIRS)]),
}


@pytest.mark.parametrize("kind", list(CASES))
def test_threads_share_a_fresh_operator(kind):
    spec = CASES[kind]
    basis, plain = engine(spec)
    D = internal.get_number_states(basis)
    assert 4096 <= D < 1 << 20
    rng = np.random.default_rng(5)
    X = rng.normal(size=(4, D, 9)) + (1j * rng.normal(size=(4, D, 9)) if kind == "complex" else 0.0)
    X = [np.asfortranarray(x) for x in X]
    internal.set_gather_cache(plain, 0)
    Y = [spined.apply(plain, x) for x in X]
    E = [spined.expectation(plain, x) for x in X]
    for round_ in range(6):
        op = spined.mk_operator(basis, [spined.mk_interaction(m, s) for m, s in spec.terms])
        gate = threading.Barrier(4)
        bad = []

        def work(i):
            gate.wait()
            for use in range(3):
                if not np.array_equal(spined.apply(op, X[i]), Y[i]):
                    bad.append(("apply", round_, i, use))
                if not np.array_equal(spined.expectation(op, X[i]), E[i]):
                    bad.append(("expectation", round_, i, use))

        threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not bad
        assert internal.gather_cache(op) == 1 and internal.schedule(op) == 1


def test_threads_make_the_first_call_together():
    """The tables of an operator are uploaded once, whoever comes first."""
    basis, plain = engine(ring(14, k=0, p=0, z=1))
    D = internal.get_number_states(basis)
    X = np.random.default_rng(9).normal(size=(6, D))
    Y = [spined.apply(plain, x) for x in X]
    bad = []
    for round_ in range(40):
        spec = ring(14, k=0, p=0, z=1)
        op = spined.mk_operator(basis, [spined.mk_interaction(m, s) for m, s in spec.terms])
        gate = threading.Barrier(len(X))

        def work(i):
            gate.wait()
            if not np.array_equal(spined.apply(op, X[i]), Y[i]):
                bad.append((round_, i))

        threads = [threading.Thread(target=work, args=(i,)) for i in range(len(X))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    assert not bad
