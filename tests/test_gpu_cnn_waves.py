"""Training kernels of the start-vector network where positions and taps are
dealt to waves: fewer positions than waves, remainders, the largest size of the
several-wave forward pass and the first beyond it, partly filled groups of 16
samples.  Against the FP64 oracle with the bounds of BF16 operands (2^-8
relative each, three layers deep: 5e-2 of the gradient's norm)."""
import numpy as np
import pytest

import pyoracle
from spined import learned

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,count", [(5, 17), (7, 40), (9, 16), (30, 33), (42, 17), (43, 17), (64, 20)])
def test_gradient_at_wave_edges(n, count):
    print("case", n, count, flush=True)
    rng = np.random.default_rng(1000 + n)
    p = learned.init_params(4)
    p[learned.NPARAMS - 34:] = rng.normal(0, 0.3, 34)
    model = learned.CNN(params=p)
    states = np.array([sum(1 << int(i) for i in rng.choice(n, n // 2, replace=False))
                       for _ in range(count)], dtype=np.uint64)
    ga, gt = rng.normal(size=count), rng.normal(size=count)
    g = model.gradient(n, states, ga, gt).astype(np.float64)
    rg = pyoracle.cnn_backward(p.astype(np.float64), n, states, ga, gt)
    assert np.linalg.norm(g - rg) <= 5e-2 * np.linalg.norm(rg)
    a, t, _, _ = model.forward(n, states, store=True)
    ra, rt = pyoracle.cnn_forward(p.astype(np.float64), n, states)
    assert np.max(np.abs(a.numpy() - ra)) <= 2e-2 * (np.max(np.abs(ra)) + 1.0)
    assert np.max(np.abs(t.numpy() - rt)) <= 2e-2 * (np.max(np.abs(rt)) + 1.0)


def test_steps_of_changing_size_share_buffers():
    """A model whose kept buffers served other sizes takes the step of a fresh one."""
    rng = np.random.default_rng(5)
    used, steps = learned.CNN(seed=2), []
    for n, count in ((12, 100), (20, 30), (8, 200), (20, 17)):
        states = np.array([sum(1 << int(i) for i in rng.choice(n, n // 2, replace=False))
                           for _ in range(count)], dtype=np.uint64)
        steps.append((n, states, rng.normal(size=count), np.ones(count)))
    for s in steps[:-1]:
        used.train_step(*s, lr=1e-3)
    fresh = learned.CNN(params=used.params())
    used.set_params(fresh.params())
    g = [m.gradient(steps[-1][0], steps[-1][1], steps[-1][2], steps[-1][3]) for m in (used, fresh)]
    np.testing.assert_array_equal(g[0], g[1])
    losses = [m.train_step(*steps[-1], lr=1e-3) for m in (used, fresh)]
    assert losses[0] == losses[1]
