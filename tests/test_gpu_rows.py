"""The forms of the MD step on the rows: rows from a scan of every molecule
and rows from the cell lists hold the oracle's pairs and give the same
trajectory, and so do one kernel per step and two."""
import os

import numpy as np
import pytest

from genesis6_amd import g6
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu


def system(n, L, rc, skin, prec, model=g6.TIP4P, grid=None, **env):
    old = {k: os.environ.get(k) for k in env}
    os.environ.update({k: str(v) for k, v in env.items()})
    try:
        s = g6.System(model, n, L, rc, 0.5, 0.002, prec=prec, skin=skin)
    finally:
        for k, v in old.items():
            if v is None:
                del os.environ[k]
            else:
                os.environ[k] = v
    com, q = g6.lattice_start(n, np.max(L), 31 + n)
    com *= np.asarray(L) / np.max(L)
    if grid is not None:  # an axis' share of the molecules by its length
        com = np.stack(np.meshgrid(*[np.arange(k) + 0.5 for k in grid], indexing="ij"), -1)
        com = com.reshape(-1, 3) * (np.asarray(L) / grid)
    # off the lattice, and some molecules boxes away (unwrapped COMs)
    com += np.random.default_rng(n).normal(0.0, 0.05, com.shape)
    com[::7] += L * np.random.default_rng(n + 1).integers(-3, 4, com[::7].shape)
    s.upload(com, q)
    s.vreset(300.0, 5)
    return s, com


# around a wave (64) and a pass (256) of the scan; one, two and three windows
# of 4096 indices in the sort of the cell rows, and windows too many for the
# rows' entries (the other sort)
@pytest.mark.parametrize("n,skin,prec", [(63, 1.0, g6.FP64), (65, 0.0, g6.FP64),
                                         (256, 1.0, g6.FP32), (257, 0.5, g6.FP64),
                                         (1000, 0.0, g6.FP32), (4097, 1.0, g6.FP32),
                                         (8500, 1.0, g6.FP64), (25003, 0.0, g6.FP64)])
def test_scan_and_cell_rows(n, skin, prec):
    L = (n / 0.0334) ** (1.0 / 3.0)
    rc = min(8.5, 0.5 * L - skin - 0.01)
    out = []
    for scan_max in (0, 1 << 20):
        s, com = system(n, L, rc, skin, prec, G6_SCAN_MAX=scan_max)
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


def brute_pairs(com, L, r):
    """Minimum-image pairs within r."""
    d = com[:, None, :] - com[None, :, :]
    d -= np.asarray(L) * np.round(d / np.asarray(L))
    return int((np.triu((d * d).sum(-1) < r * r, 1)).sum())


# cells of unequal counts per axis: 6 x 9 x 4 (an axis below the five cells of
# the stencil, two above) and 2 x 5 x 11 (two cells across an axis); under the
# barostat the box, and with it the stencil's pruning, moves with every step
@pytest.mark.parametrize("L,rc,skin", [((28.0, 41.0, 17.3), 8.0, 0.5),
                                       ((13.4, 30.1, 60.5), 4.9, 0.5)])
@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("prec", [g6.FP64, g6.FP32])
def test_scan_and_cell_rows_in_other_boxes(L, rc, skin, mode, prec):
    grid = [int(e / 3.1) for e in L]
    n = int(np.prod(grid))
    out = []
    for env in (dict(G6_SCAN_MAX=1 << 20), dict(G6_SCAN_MAX=0),
                dict(G6_SCAN_MAX=0, G6_STEP_MAX=0)):
        s, com = system(n, np.array(L), rc, skin, prec, grid=grid, **env)
        print("rows in a box of", L, "mode", mode, env, flush=True)
        s.set_nose(300.0, 7.5e5)
        if mode:
            s.set_andersen(1.0, 1e-3, mode=mode)
        _, _, th = s.eval_forces()
        s.step(3)
        s.step(60)
        out.append([th, s.thermo(), s.box3(), *s.download()])
        s.close()
    for k, r in ((14, rc), (15, rc + skin)):
        assert out[0][0][k] == brute_pairs(com, L, r)
    if mode:
        assert not np.array_equal(out[0][2], L)
    for other in out[1:]:
        for a, b in zip(out[0], other):
            assert np.array_equal(a, b)


# blocks of four molecules with one to four of them; a thousand kinetic
# energies and more (four per thread); boxes, thermostat, models of three to
# six sites; calls of one, two and several steps between other calls
@pytest.mark.parametrize("n,model,prec,skin,nose,ortho", [
    (2, g6.TIP4P, g6.FP64, 0.0, True, False), (65, g6.TIP5P, g6.FP32, 0.5, True, False),
    (127, g6.SPCE, g6.FP64, 1.0, False, True), (216, g6.NVDE, g6.FP32, 0.0, True, False),
    (510, g6.ST2, g6.FP64, 1.0, True, True), (4101, g6.TIP4P, g6.FP32, 1.0, True, False)])
def test_one_kernel_and_two_kernel_steps(n, model, prec, skin, nose, ortho):
    L = (n / 0.0334) ** (1.0 / 3.0) if n > 2 else 12.0
    rc = min(8.5, 0.45 * L - skin - 0.01)
    box = np.array([L, 1.1 * L, L]) if ortho else L
    out = []
    for step_max in (1 << 30, 0):
        s, _ = system(n, box, rc, skin, prec, model, G6_STEP_MAX=step_max)
        if nose:
            s.set_nose(300.0, 7.5e5)
        print("steps n %d model %d step_max %d" % (n, model, step_max), flush=True)
        got = []
        for k in (1, 2, 1, 7, 50):
            s.step(k)
            got += [s.thermo(), s.nose(), *s.download()]
            if k == 7:
                got += list(s.eval_forces())
                if nose:
                    s.set_temperature(320.0)
        out.append(got)
        s.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


# only a call's last close forms the thermo record; the listed pairs [15] are
# of the call's last row build
@pytest.mark.parametrize("n,prec,skin,env", [
    (217, g6.FP64, 0.0, {}), (1000, g6.FP32, 1.0, {}), (4101, g6.FP32, 0.3, {"G6_STEP_MAX": 0}),
    (6201, g6.FP32, 0.3, {}), (1024, g6.FP32, 1.0, {"G6_TILE_MIN": 0})])
@pytest.mark.parametrize("nose", [True, False])
def test_a_call_of_many_steps_and_many_calls(n, prec, skin, env, nose):
    L = (n / 0.0334) ** (1.0 / 3.0)
    out = []
    print("calls n %d skin %g" % (n, skin), env, flush=True)
    for calls in ([60], [1] * 60):
        s, _ = system(n, L, min(8.5, 0.45 * L - skin - 0.01), skin, prec, **env)
        assert s.md_kernel()[0] == ("G6_TILE_MIN" in env)
        if nose:
            s.set_nose(300.0, 7.5e5)
        for k in calls:
            s.step(k)
        assert s.md_kernel()[0] == ("G6_TILE_MIN" in env)
        out.append([s.thermo(), s.nose(), *s.download()])
        s.close()
    assert out[0][0][15] > 0
    for a, b in zip(*out):
        assert np.array_equal(a, b)
