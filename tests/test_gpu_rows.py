"""The row build of the MD force kernel: rows from a scan of every molecule
and rows from the cell lists hold the oracle's pairs and give the same
trajectory."""
import os

import numpy as np
import pytest

from genesis6_amd import g6
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu


def system(n, L, rc, skin, prec, scan_max):
    old = os.environ.get("G6_SCAN_MAX")
    os.environ["G6_SCAN_MAX"] = str(scan_max)
    try:
        s = g6.System(g6.TIP4P, n, L, rc, 0.5, 0.002, prec=prec, skin=skin)
    finally:
        if old is None:
            del os.environ["G6_SCAN_MAX"]
        else:
            os.environ["G6_SCAN_MAX"] = old
    com, q = g6.lattice_start(n, L, 31 + n)
    # off the lattice, and some molecules boxes away (unwrapped COMs)
    com += np.random.default_rng(n).normal(0.0, 0.05, com.shape)
    com[::7] += L * np.random.default_rng(n + 1).integers(-3, 4, com[::7].shape)
    s.upload(com, q)
    s.vreset(300.0, 5)
    return s, com


# around a wave (64) and a pass (256) of the scan; one, two and three windows
# of 4096 indices in the sort of the cell rows
@pytest.mark.parametrize("n,skin,prec", [(63, 1.0, g6.FP64), (65, 0.0, g6.FP64),
                                         (256, 1.0, g6.FP32), (257, 0.5, g6.FP64),
                                         (1000, 0.0, g6.FP32), (4097, 1.0, g6.FP32),
                                         (8500, 1.0, g6.FP64)])
def test_scan_and_cell_rows(n, skin, prec):
    L = (n / 0.0334) ** (1.0 / 3.0)
    rc = min(8.5, 0.5 * L - skin - 0.01)
    out = []
    for scan_max in (0, 1 << 20):
        s, com = system(n, L, rc, skin, prec, scan_max)
        print("rows n %d skin %g scan_max %d" % (n, skin, scan_max), flush=True)
        _, _, th = s.eval_forces()
        s.step(12)
        out.append((th, s.download(), s.thermo()))
        s.close()
    for k, radius in ((14, rc), (15, rc + skin)):
        pairs = len(O.pairlist(com, L, radius, radius)[1])
        assert out[0][0][k] == pairs and out[1][0][k] == pairs, (k, pairs)
    for a, b in zip(out[0][1], out[1][1]):
        assert np.array_equal(a, b)
    assert np.array_equal(out[0][2], out[1][2])
