"""Constant-pressure MD with the Andersen barostat on the GPU against the
reference MD driver (tests/golden/md_tip4p_216_npt.npz, written by
tests/golden/make_npt_md.py): the Fortran driver g6md runs the reference's
decks and logs its @LOGD rows; the pair-list skin keeps the interacting set
while the box moves; the restart carries the barostat (@PCN5)."""
import os
import subprocess
import tempfile

import numpy as np
import pytest

from genesis6_amd import g6
from oracle import pyoracle as O
from tests.golden.configs import parse_logd
from tests.test_gpu_restart import same_restart

pytestmark = pytest.mark.gpu
EXE = os.path.abspath(os.path.join(os.path.dirname(__file__), "..", "genesis6_amd", "lib",
                                   "g6md"))


def run_g6md(deck, *args):
    with tempfile.TemporaryDirectory() as d:
        r = subprocess.run([EXE] + list(args), input=deck, capture_output=True, text=True,
                           timeout=120, cwd=d)
        assert r.returncode == 0, r.stderr
        with open(os.path.join(d, "fort.13"), "rb") as f:
            return parse_logd(r.stdout), f.read()


@pytest.mark.parametrize("name", ["npt", "nph"])
def test_andersen_log_matches_reference_driver(golden, name):
    f = golden("md_tip4p_216_npt")
    print("g6md fp64", name, flush=True)
    got, f13 = run_g6md(str(f["deck_" + name]), "fp64")
    ref = f["logd_" + name]
    assert got.shape == ref.shape
    np.testing.assert_array_equal(got[:, 0], ref[:, 0])
    # T, P, V, ep, ek, Nose, Andersen energies, H
    for col, tol in [(1, 1e-10), (2, 1e-6), (3, 1e-12), (4, 1e-9), (5, 1e-10), (10, 1e-12),
                     (11, 1e-6), (12, 1e-10)]:
        err = np.abs(got[:, col] - ref[:, col]).max() / (np.abs(ref[:, col]).max() + 1e-300)
        print("  column %d: %.2e" % (col, err))
        assert err <= tol, (col, err)
    if name == "npt":
        same_restart(f13, f["fort13_npt"].tobytes(), 216)


@pytest.mark.parametrize("mid", [g6.SPCE, g6.NVDE, g6.TIP5P])
def test_andersen_other_models_follow_the_oracle(golden, mid):
    """The barostat with the other rigid models (the Andersen step does not
    depend on the model): 30 FP64 steps of @PCN4 1 1.0 1e-4 with the Nose
    thermostat against the oracle's step (pinned bit for bit to the
    reference driver for TIP4P): T, P, V and H at every step."""
    g = golden("md_tip4p_216_nve1000")
    L, rc, taper, dt = float(g["L"]), float(g["rc"]), float(g["taper"]), float(g["dt"])
    print("andersen model", mid, flush=True)
    s = g6.System(mid, 216, L, rc, taper, dt, prec=g6.FP64)
    md = O.MDRun(mid, g["com"], g["quat"].T.copy(), L, rc, taper, dt, nose=(300.0, 7.5e5, 0.0))
    try:
        s.upload(g["com"], g["quat"])
        s.set_nose(300.0, 7.5e5)
        s.vreset(300.0, 4246)
        s.set_andersen(1.0, 1e-4)
        md.set_andersen(1.0, 1e-4)
        md.vreset(300.0, 4246)
        for k in range(30):
            s.step(1)
            md.step()
            th = s.thermo()
            assert abs(th[3] - md.s.temperature) <= 1e-11 * md.s.temperature, k
            assert abs(th[25] - md.s.pressure) <= 1e-8 * max(1.0, abs(md.s.pressure)), k
            assert abs(th[26] - md.s.volume) <= 1e-13 * md.s.volume, k
            assert abs(th[13] - md.hamiltonian()) <= 1e-11 * abs(md.hamiltonian()), k
        assert abs(s.box() - md.s.L) <= 1e-13 * md.s.L
    finally:
        s.close()


def test_skin_keeps_the_interacting_set_while_the_box_moves(golden):
    """FP64 with a 1 A skin against no skin under a light barostat (the box
    edge moves by about 0.1 A in 300 steps): the same interacting pairs at
    every step, so the same trajectory bit for bit."""
    g = golden("md_tip4p_216_nve1000")
    runs = []
    for skin in (0.0, 1.0):
        s = g6.System(g6.TIP4P, 216, float(g["L"]), float(g["rc"]), float(g["taper"]),
                      float(g["dt"]), prec=g6.FP64, skin=skin)
        try:
            s.upload(g["com"], g["quat"])
            s.set_nose(300.0, 7.5e5)
            s.vreset(300.0, 4246)
            s.set_andersen(1.0, 2e-6)
            rows = []
            for _ in range(30):
                s.step(10)
                th = s.thermo()
                rows.append([th[14], th[26], th[0], th[13]])
            runs.append((np.array(rows), s.download()[0], s.box()))
        finally:
            s.close()
    (a, ca, La), (b, cb, Lb) = runs
    print("box %.6f -> %.6f, pairs %d..%d" % (float(g["L"]), La, a[:, 0].min(), a[:, 0].max()))
    assert abs(La - float(g["L"])) > 0.05           # the box did move
    np.testing.assert_array_equal(a, b)
    np.testing.assert_array_equal(ca, cb)
    assert La == Lb


def test_fp32_follows_fp64_under_the_barostat(golden):
    """FP32 pair arithmetic with the skin against FP64: the volume and the
    temperature follow the FP64 run over 50 steps."""
    f = golden("md_tip4p_216_npt")
    a, _ = run_g6md(str(f["deck_npt"]), "fp64")
    b, _ = run_g6md(str(f["deck_npt"]), "fp32", "1.0")
    assert np.abs(b[:, 3] / a[:, 3] - 1).max() < 1e-6
    assert np.abs(b[:, 1] / a[:, 1] - 1).max() < 1e-4


def baro_start(n, L, rc, pex, mass, skin=1.0, dt=0.001, tiles=False, **env):
    """A hot lattice start under the barostat; env is read at g6_init."""
    old = {k: os.environ.get(k) for k in env}
    os.environ.update({k: str(v) for k, v in env.items()})
    try:
        s = g6.System(g6.TIP4P, n, L, rc, 0.5, dt, prec=g6.FP32, skin=skin)
    finally:
        for k, v in old.items():
            if v is None:
                del os.environ[k]
            else:
                os.environ[k] = v
    com, q = g6.lattice_start(n, L, 9)
    s.upload(com, q)
    s.set_nose(1500.0, 1500.0 * 2500.0)
    s.vreset(1500.0, 9)
    if not tiles:
        s.set_andersen(pex, mass)
    return s


def same_run(s, f, steps=3):
    """Both handles step on alike: every bit of state and thermo but the
    listed-pair count [15], which depends on when rows were last built."""
    for _ in range(steps):
        s.step(1)
        f.step(1)
        a, b = s.thermo(), f.thermo()
        assert a[14] == b[14], (a[14], b[14])
        np.testing.assert_array_equal(np.delete(a, 15), np.delete(b, 15))
    for x, y in zip(s.download(), f.download()):
        np.testing.assert_array_equal(x, y)
    assert s.box() == f.box()


# the call that fails runs far enough that its last rows are of other
# positions: a cell list of 8 residents overflows once the lattice has melted;
# a box with 0.05 A to spare above its grid's smallest edge is pressed past it
@pytest.mark.parametrize("kw", [
    dict(n=1024, L=31.289, rc=8.5, pex=1.0, mass=1e-2, G6_CELL_CAP=9),
    dict(n=160, L=19.05, rc=8.5, pex=2e4, mass=1e-2)], ids=["cells", "box"])
def test_a_failed_barostat_call_leaves_no_rows_behind(kw):
    print("failed barostat call", kw, flush=True)
    s, f = baro_start(**kw), baro_start(**kw)
    s.step(2)  # rows, which a small displacement would keep
    f.step(2)
    before = s.download()
    with pytest.raises(g6.G6Error):
        s.step(400)
    for x, y in zip(before, s.download()):
        np.testing.assert_array_equal(x, y)
    same_run(s, f)
    s.close()
    f.close()


def test_the_barostat_after_the_tiles_builds_its_rows():
    """A system that stepped on the cell tiles has no rows of both directions
    yet: the barostat's first step builds them."""
    kw = dict(n=1024, L=31.289, rc=9.0, pex=1.0, mass=1e-4)
    print("barostat after the tiles", flush=True)
    s = baro_start(tiles=True, G6_TILE_MIN=0, **kw)
    assert s.md_kernel()[0] == 1
    s.step(20)
    com, quat, dx, w = s.download()
    f = baro_start(tiles=True, G6_TILES=0, **kw)
    f.upload(com, None, dx=dx, w=w, quat=quat)
    z = s.nose()
    f.set_nose(z[0], z[1] / 0.001, z[2], z[3:8], z[8])
    np.testing.assert_array_equal(f.nose(), z)
    for h in (s, f):
        h.set_andersen(1.0, 1e-4)
    same_run(s, f)
    s.close()
    f.close()


def test_the_fixed_box_after_the_barostat_builds_its_rows():
    """Mode 0 gives the handle its first box back: the rows of the barostat's
    last box are not kept for it."""
    kw = dict(n=1024, L=31.289, rc=8.5, pex=1.0, mass=1e-5, G6_CELL_CAP=30)
    print("fixed box after the barostat", flush=True)
    s = baro_start(**kw)
    s.step(120)
    assert s.box() > 31.289 + 0.5
    s.set_andersen(1.0, 1e-4, mode=0)
    com, quat, dx, w = s.download()
    f = baro_start(tiles=True, **kw)
    f.upload(com, None, dx=dx, w=w, quat=quat)
    z = s.nose()
    f.set_nose(z[0], z[1] / 0.001, z[2], z[3:8], z[8])
    np.testing.assert_array_equal(f.nose(), z)
    same_run(s, f)
    s.close()
    f.close()
