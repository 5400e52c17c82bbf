"""Small device blocks handed on between calls: threads that apply operators of
different sizes at the same time, objects dropped while their last work is in
flight, and a release of the pool in between all leave the results unchanged."""
import threading

import numpy as np
import pytest

import spined
from helpers import engine, ring

pytestmark = pytest.mark.gpu


def test_threads_share_small_blocks():
    specs = [ring(n, k=0, p=0, z=1) for n in (12, 16, 18, 20)]
    made = [engine(s) for s in specs]
    rng = np.random.default_rng(2)
    X = [np.asfortranarray(rng.uniform(-1, 1, (spined.get_number_states(b), c)))
         for (b, _), c in zip(made, (1, 3, 2, 5))]
    Y = [spined.apply(op, x) for (_, op), x in zip(made, X)]
    E = [spined.expectation(op, x) for (_, op), x in zip(made, X)]
    bad = []

    def work(i):
        for rep in range(20):
            _, op = engine(specs[i]) if rep % 5 == 4 else made[i]
            if not np.array_equal(spined.apply(op, X[i]), Y[i]):
                bad.append(("apply", i, rep))
            if not np.array_equal(spined.expectation(op, X[i]), E[i]):
                bad.append(("expectation", i, rep))
            if i == 0 and rep % 7 == 3:
                spined.release_device_pool()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    spined.release_device_pool()
