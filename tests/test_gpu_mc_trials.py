"""The trial kernel of the Monte Carlo path against the oracle, bit for bit:
each model's list of site pairs, sizes at the edges of a wave, of the threads'
molecules and of the largest system taken, and coordinates so far out that the
image shift does not fit the list's 16 bits."""
import numpy as np
import pytest

from genesis6_amd import g6
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu


def start(n, L, seed):
    rng = np.random.default_rng(seed)
    k = int(np.ceil(n ** (1 / 3)))
    grid = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    com = (grid + 0.5) * (L / k) + rng.uniform(-0.2, 0.2, (n, 3))
    q = rng.normal(size=(n, 4))
    q /= np.linalg.norm(q, axis=1)[:, None]
    q[q[:, 0] < 0] *= -1
    return com, q


@pytest.mark.parametrize("model,n,far", [
    ("TIP4P", 2, 0), ("TIP4P", 64, 0), ("SPCE", 65, 0), ("TIP5P", 511, 0), ("NVDE", 513, 0),
    ("OPLSMEOH", 216, 0), ("ST2", 100, 0), ("TIP4P", 1025, 0), ("TIP4P", 1535, 0), ("TIP4P", 216, 40000),
])
def test_trials_equal_the_oracle(model, n, far):
    L = max(20.0, 3.2 * n ** (1 / 3) + 0.1)
    com, q = start(n, L, n + far)
    com[::3, 1] += far * L
    print("mc trials", model, n, far, flush=True)
    s = g6.System(getattr(g6, model), n, L, 9.0, 0.5, 0.002)
    s.upload(com, q)
    s.mc_begin(300.0, 17, 0.2, 1.0)
    o = O.MCRun(getattr(O, model), com, q.T.copy(), L, 9.0, 0.5, 300.0, 17, 0.2, 1.0)
    for trials in (70, 33):  # past a staged chunk, and on from there
        assert s.mc_trials(trials) == o.trials(trials)
    c, qq, d, rt, e = s.mc_state()
    np.testing.assert_array_equal(c, o.com)
    np.testing.assert_array_equal(qq.T, o.quat)
    np.testing.assert_array_equal(d, o.delta)
    np.testing.assert_array_equal(rt, o.rtr)
    # the sums run in other orders: n terms a trial of the energies' size
    bound = 2.0 ** -52 * (n + 103) * max(1.0, np.abs(o.ep).max(), abs(o.epsum[0]))
    assert abs(e - o.epsum[0]) <= bound
    s.close()


def test_the_largest_system():
    """1535 molecules are taken (above), one more is refused."""
    com, q = start(1536, 37.0, 3)
    s = g6.System(g6.TIP4P, 1536, 37.0, 9.0, 0.5, 0.002)
    s.upload(com, q)
    with pytest.raises(g6.G6Error):
        s.mc_begin(300.0, 17, 0.2, 1.0)
    s.close()
