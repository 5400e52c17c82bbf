"""With device memory filled to less than the gather cache's reserve, operators run
matrix-free and allocate nothing for a cache that cannot fit."""
import numpy as np
import pytest
import torch

import spined
from spined import internal
from spined.device import DeviceArray
from helpers import engine, ring

pytestmark = pytest.mark.gpu


def test_no_cache_tables_below_the_reserve():
    specs = [ring(20, k=3, p=None, z=None, name="ring"), ring(20, k=0, p=0, z=1)]
    made = []
    for spec in specs:
        basis, plain = engine(spec)
        op = spined.mk_operator(basis, [spined.mk_interaction(m, s) for m, s in spec.terms])
        internal.set_gather_cache(plain, 0)
        x = np.random.default_rng(3).normal(size=internal.get_number_states(basis))
        x = x if plain.is_real else x + 1j * x[::-1]
        made.append((op, x, spined.apply(plain, x)))
    spined.release_device_pool()
    free, _ = torch.cuda.mem_get_info()
    fill = DeviceArray(free - (3 << 30), np.uint8)
    try:
        assert torch.cuda.mem_get_info()[0] < 4 << 30
        for op, x, ref in made:
            for _ in range(3):
                np.testing.assert_array_equal(spined.apply(op, x), ref)
                assert internal.gather_cache(op) == 0
        # a complex operator's row schedule comes with its cache
        assert internal.schedule(made[0][0]) == 0
    finally:
        del fill
    for op, x, ref in made:
        np.testing.assert_array_equal(spined.apply(op, x), ref)
        assert internal.gather_cache(op) == 1
