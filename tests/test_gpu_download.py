"""The state's download in pieces of 131,072 doubles (53 n in all): what was
uploaded, bit for bit, where it ends at, before and behind a piece's edge, and
from several threads at once."""
import threading

import numpy as np
import pytest

from genesis6_amd import g6

pytestmark = pytest.mark.gpu


def state(n, seed):
    rng = np.random.default_rng(seed)
    return [rng.normal(size=s) for s in ((n, 3), (5, 4, n), (5, 3, n), (5, 3, n))]


def handle(n, st):
    s = g6.System(g6.TIP4P, n, 60.0, 9.0, 0.5, 0.002)
    s.upload(st[0], None, dx=st[2], w=st[3], quat=st[1])
    return s


def same(s, st):
    return all(np.array_equal(a, b) for a, b in zip(s.download(), st))


@pytest.mark.parametrize("n", [2, 2473, 2474, 4947, 8289])
def test_download_returns_the_upload(n):
    print("download", n, flush=True)
    st = state(n, n)
    s = handle(n, st)
    assert same(s, st) and same(s, st)
    s.close()


def test_threads_take_turns():
    print("download, four threads", flush=True)
    sts = [state(n, n) for n in (64, 2474, 3000, 4947)]
    hs = [handle(len(st[0]), st) for st in sts]
    ok = [False] * 4

    def run(k):
        ok[k] = all(same(hs[k], sts[k]) for _ in range(5))

    ts = [threading.Thread(target=run, args=(k,)) for k in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert all(ok)
    for h in hs:
        h.close()
