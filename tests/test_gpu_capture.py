"""Device matvecs recorded by a stream capture: what is not built yet is not built
there, and replays have the bits of eager calls."""
import numpy as np
import pytest
import torch

import spined
from spined import _lib, internal, lattice
from spined.device import DeviceArray
from helpers import engine, ring

pytestmark = pytest.mark.gpu


def _capture(op, x, y, code):
    stream = torch.cuda.ExternalStream(_lib.load().spined_stream())
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        graph.capture_begin(capture_error_mode="relaxed")
        try:
            internal.matvec_device(op, x, y, code)
        finally:
            graph.capture_end()
    return graph, stream


def _replays(op, graph, stream, x, y, code, draw):
    """Replays against eager calls, with other work and a wait in between."""
    for _ in range(4):
        x.copy_(draw())
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            graph.replay()
        torch.cuda.synchronize()
        got = y.clone()
        y.zero_()
        torch.cuda.synchronize()
        internal.matvec_device(op, x, y, code)
        torch.cuda.synchronize()
        assert torch.equal(got, y)


def test_split_tables_are_not_built_under_capture():
    n = 23
    basis = spined.mk_basis(spined.mk_group([]), n, 11, None)
    spined.build_basis(basis)
    J = np.random.default_rng(1).uniform(0.8, 1.2, n)
    op = spined.mk_operator(basis, [spined.mk_interaction(lattice.xxz_matrix(0.5, J[b]), [[b, (b + 1) % n]])
                                    for b in range(n)])
    D = internal.get_number_states(basis)
    x = torch.randn(1, D, dtype=torch.float64, device="cuda")
    y = torch.empty_like(x)
    torch.cuda.synchronize()
    internal.set_gather_cache(op, 0)  # uploads the operator, builds no tables
    internal.matvec_device(op, x, y, 1)
    internal.set_gather_cache(op, -1)
    graph, stream = _capture(op, x, y, 1)
    assert internal.debug_matvec_path(op) == 0
    _replays(op, graph, stream, x, y, 1, lambda: torch.randn_like(x))
    assert internal.debug_matvec_path(op) == 2
    # recorded with the tables there
    graph, stream = _capture(op, x, y, 1)
    assert internal.debug_matvec_path(op) == 2
    _replays(op, graph, stream, x, y, 1, lambda: torch.randn_like(x))


@pytest.mark.parametrize("n,k,code", [(20, 0, 1), (20, 3, 3)])
def test_recorded_cache_outlives_a_refused_allocation(n, k, code):
    basis, op = engine(ring(n, k=k, p=None if k else 0, z=None if k else 1))
    other = spined.mk_operator(basis, [spined.mk_interaction(lattice.xxz_matrix(0.3), lattice.ring_bonds(n))])
    D = internal.get_number_states(basis)
    x = torch.randn(1, D, dtype=torch.complex128 if k else torch.float64, device="cuda")
    y = torch.empty_like(x)
    torch.cuda.synchronize()
    for o in (op, other):
        for _ in range(2):
            internal.matvec_device(o, x, y, code)
        assert internal.gather_cache(o) == 1
    graph, stream = _capture(op, x, y, code)
    with pytest.raises(Exception):
        DeviceArray(1 << 50, np.uint8)  # refused: the library gives its caches back
    assert internal.gather_cache(other) == 0
    assert internal.gather_cache(op) == 1
    _replays(op, graph, stream, x, y, code, lambda: torch.randn_like(x))
    del graph
    internal.set_gather_cache(op, 0)  # at the owner's word
    assert internal.gather_cache(op) == 0
