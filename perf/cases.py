"""Performance cases: the work a simulation program has this library do.

Every case starts from a liquid (a short damped run from a random lattice,
made here with plain torch and repeated k times along each axis), so that the
library meets liquid densities, forces and neighbour counts.  The kinds:

  md       g6.System.step of one system, then its thermo record and state: a
           log interval of an MD run.  From 216 molecules (launches count) over
           the usual few thousand to 65,536; FP64 and FP32 pairs; rows rebuilt
           every step (skin 0, the reference's list) or kept with a skin; NVE,
           Nose NVT, and the Andersen barostat.  FP32 intervals are short: the
           rounding of the pair forces grows with every step.
  ladder   g6.Ladder.step of replica-exchange ladders (every replica in one
           launch), the thermo records and the states.
  mixture  g6.Mixture.step of water with methanol.
  mc       one sweep of mc2's single-molecule trials.
  npt      NPT Monte Carlo with volume and block moves; with K > 0 screened by
           the surrogate network (delayed acceptance).
  train    epochs of surrogate training on host feature rows.

exact() is the same calculation in plain torch and numpy, in 64 bits.
"""
import functools
import math

import numpy as np
import torch

from genesis6_amd import g6

DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64 = torch.float64
COULOMB = 4.184 * 332.17752 * 100.0  # e^2/A in the internal energy unit (10 J/mol)
RGAS = 6.0225e23 * 1.380066e-23
I2J, J2K = 10.0, 0.120273
DENSITY = 1024 / 31.289 ** 3         # molecules per A^3 at 1.0 g/cm3
LADDERS = [(256, 20.266), (512, 25.088), (1024, 31.289), (2048, 38.786)]
REPEAT = {256: (256, 1), 512: (512, 1), 1024: (1024, 1), 2048: (256, 2)}


# ---- the cases -------------------------------------------------------------

def listed():
    return [
        # the smallest system, the reference's own method: rows rebuilt every
        # step, FP64, NVE; a step is a few launches of a few wavefronts
        dict(name="md-tip4p-216-fp64", kind="md", model="tip4p", m=216, k=1, L=18.626, rc=8.5,
             fp64=True, skin=0.0, nose=False, baro=False, steps=100),
        # constant pressure: the box changes every step
        dict(name="md-spce-1000-npt", kind="md", model="spce", m=1000, k=1, L=31.04, rc=8.5,
             fp64=True, skin=1.0, nose=True, baro=True, steps=50),
        # the benchmark's system in both precisions
        dict(name="md-tip4p-4096-fp32", kind="md", model="tip4p", m=512, k=2, L=49.669, rc=9.0,
             fp64=False, skin=1.8, nose=True, baro=False, steps=40),
        dict(name="md-tip4p-4096-fp64", kind="md", model="tip4p", m=512, k=2, L=49.669, rc=9.0,
             fp64=True, skin=1.8, nose=True, baro=False, steps=100),
        # an odd count, between the two force kernels' ranges, five-site water
        dict(name="md-st2-8289-fp32", kind="md", model="st2", m=307, k=3, L=62.82, rc=9.0,
             fp64=False, skin=1.0, nose=True, baro=False, steps=40),
        # a large system: the force kernel's throughput
        dict(name="md-tip5p-65536-fp32", kind="md", model="tip5p", m=1024, k=4, L=125.157, rc=9.0,
             fp64=False, skin=1.0, nose=True, baro=False, steps=40),
        # replica exchange: four ladders of 16 temperatures
        dict(name="ladder-64", kind="ladder", first=0, count=4, rungs=16, skin=1.0, steps=40),
        # two components
        dict(name="mixture-4096-fp32", kind="mixture", water=448, meoh=64, k=2, fp64=False,
             skin=1.0, steps=40),
        # Monte Carlo: one sweep of trials; 100 collective moves; 20 rounds of
        # 32 screened proposals
        dict(name="mc-tip4p-1024", kind="mc", n=1024, trials=1024),
        dict(name="npt-tip4p-1024", kind="npt", n=1024, moves=100, K=0),
        dict(name="npt-da-tip4p-1024", kind="npt", n=1024, moves=20, K=32),
        # the surrogate's training, two epochs over 256 configurations
        dict(name="train-262144", kind="train", rows=262144, batch=4096, epochs=2),
    ]


def draw(rng):
    kind = rng.choice(["md", "md", "md", "md", "md", "ladder", "mixture", "mc", "npt", "npt",
                       "train"])
    if kind == "md":
        model = rng.choice(["tip4p", "tip5p", "st2", "spce"])
        fp64 = rng.random() < 0.4
        if rng.random() < 0.15:
            # the barostat moves the box: edges between two cell counts of the
            # grid (cells of at least (rc + skin) / 2), as a run has to choose
            L = round(4.75 * (rng.randint(4, 6) + rng.uniform(0.4, 0.8)), 3)
            return dict(kind="md", model=model, m=int(DENSITY * L ** 3), k=1, L=L, rc=8.5,
                        fp64=fp64, skin=1.0, nose=True, baro=True, steps=rng.randint(20, 40))
        n = math.exp(rng.uniform(math.log(200), math.log(12000 if fp64 else 40000)))
        k = 1 if n < 800 else rng.choice([2, 3]) if n < 8000 else rng.choice([3, 4])
        m = max(200, int(n / k ** 3))
        L = round((m / DENSITY / rng.uniform(0.92, 1.05)) ** (1 / 3) * k, 3)
        skin = 0.0 if m * k ** 3 < 2000 and rng.random() < 0.4 else round(rng.uniform(0.8, 1.8), 1)
        # rc + skin <= L / 2
        rc = min(9.0, math.floor(10 * (L / 2 - skin - 0.05)) / 10)
        return dict(kind="md", model=model, m=m, k=k, L=L, rc=rc, fp64=fp64, skin=skin,
                    nose=rng.random() < 0.8, baro=False, steps=rng.randint(20, 40))
    if kind == "ladder":
        first = rng.randint(0, 3)
        return dict(kind="ladder", first=first, count=rng.randint(1, 4 - first),
                    rungs=rng.randint(3, 13), skin=1.0, steps=rng.randint(20, 40))
    if kind == "mixture":
        return dict(kind="mixture", water=rng.randint(230, 500), meoh=rng.randint(20, 130),
                    k=rng.choice([1, 2]), fp64=rng.random() < 0.5, skin=1.0,
                    steps=rng.randint(20, 40))
    if kind == "mc":
        n = int(math.exp(rng.uniform(math.log(216), math.log(1400))))
        return dict(kind="mc", n=n, trials=rng.randint(200, 1200))
    if kind == "npt":
        K = rng.choice([0, 8, 16, 32])
        return dict(kind="npt", n=int(math.exp(rng.uniform(math.log(500), math.log(1200)))),
                    moves=rng.randint(10, 20) if K else rng.randint(40, 120), K=K)
    rows = int(math.exp(rng.uniform(math.log(20000), math.log(260000))))
    return dict(kind="train", rows=rows, batch=rng.choice([1024, 2048, 4096]), epochs=2)


def molecules(c):
    if c["kind"] == "md":
        return c["m"] * c["k"] ** 3
    if c["kind"] == "mixture":
        return (c["water"] + c["meoh"]) * c["k"] ** 3
    return sum(n for n, _ in chosen(c)) * c["rungs"]


def chosen(c):
    return LADDERS[c["first"]:c["first"] + c["count"]]


def work(c):
    """Floating-point operations of the pairs within rc, each once; the state
    (or the training rows) read once and written once per pass."""
    pair = dict(tip4p=257, tip5p=404, st2=416, spce=257)
    if c["kind"] in ("md", "ladder", "mixture"):
        n = molecules(c)
        rc = c.get("rc", 9.0 if c["kind"] == "ladder" else 8.5)
        pairs = 0.5 * n * DENSITY * 4 / 3 * math.pi * rc ** 3
        return dict(bytes=n * 53 * 8 * 2,
                    flops=c["steps"] * pairs * pair[c.get("model", "tip4p")])
    near = DENSITY * 4 / 3 * math.pi * 9.0 ** 3
    if c["kind"] == "mc":
        return dict(bytes=c["n"] * 9 * 8 * 2,
                    flops=c["trials"] * near * 10 * 12)
    if c["kind"] == "npt":
        block, vol = 36.0, c["n"] / 2
        exact_ = c["moves"] * (27 / 28 * block + vol / 28) if not c["K"] else c["moves"] * vol / 2
        rows = 0 if not c["K"] else c["moves"] * c["K"] * (27 / 28 * 150 + c["n"] / 28)
        return dict(bytes=c["n"] * 7 * 8 * 2,
                    flops=exact_ * near * 10 * 12 + rows * (12416 + 340 * 45))
    steps = c["epochs"] * (c["rows"] // c["batch"])
    return dict(bytes=c["rows"] * 33 * 4, flops=steps * c["batch"] * 12416 * 3)


def tolerance(c):
    if c["kind"] in ("mc", "npt"):
        # the chain in FP64: the same decisions, sums in another order
        return dict(rel=1e-12, max=1e-10)
    if c["kind"] == "train":
        # BF16 roundings of gradients and weights, through Adam: 0.7e-3 to
        # 1.4e-3 from the same training in 64 bits after two passes
        return dict(rel=5e-3, max=0.12)
    if c.get("fp64"):
        # 0.9e-11 after 200 steps (the angular velocities, furthest off)
        return dict(rel=5e-11, max=1e-9)
    # FP32 pair arithmetic: 1e-6 after 50 steps and 1.2e-5 after 100, growing
    # as neighbouring trajectories part; two passes are at most 80 steps
    return dict(rel=6e-5, max=1e-2)


# ---- rigid molecules in plain torch -----------------------------------------

def _model(name):
    """Body-frame sites, charges, LJ eps (kJ/mol) and sigma (A), masses."""
    rad = math.pi / 180.0

    def water(theta, oh, zshift_mass=18.0):
        y, z = oh * math.sin(0.5 * theta * rad), oh * math.cos(0.5 * theta * rad)
        return y, z, z * 2.0 / zshift_mass
    st2 = None
    if name == "tip4p":
        y, z, s = 0.756950327263661182, 0.520784245882928820, 0.0
        sites = [(0, 0, -0.0650980307353661025), (0, 0, 0.0849019692646338919), (0, y, z),
                 (0, -y, z)]
        q, mass = [0.0, -1.04, 0.52, 0.52], [16.0, 0.0, 1.0, 1.0]
        eps, sig = [0.15504166666666666 * 4.184, 0, 0, 0], [3.15357794197649532, 0, 0, 0]
    elif name in ("tip5p", "st2"):
        theta, oh, ol = (109.47, 1.0, 0.8) if name == "st2" else (104.52, 0.9572, 0.70)
        y, z, s = water(theta, oh)
        x, zl = ol * math.sin(0.5 * 109.47 * rad), -ol * math.cos(0.5 * 109.47 * rad)
        sites = [(0, 0, -s), (0, y, z - s), (0, -y, z - s), (x, 0, zl - s), (-x, 0, zl - s)]
        mass = [16.0, 1.0, 1.0, 0.0, 0.0]
        if name == "st2":
            e, qh = float(np.float32(0.52605e-21)) * 6.0225e23 * 1e-3, float(np.float32(0.2357))
            eps, sig, st2 = [e, 0, 0, 0, 0], [3.1, 0, 0, 0, 0], (2.0160, 3.1287)
        else:
            qh = 0.2410
            eps, sig = [0.6694, 0, 0, 0, 0], [3.12, 0, 0, 0, 0]
        q = [0.0, qh, qh, -qh, -qh]
    elif name == "spce":
        y, z, s = water(109.5, 1.0)
        sites = [(0, 0, -s), (0, y, z - s), (0, -y, z - s)]
        q, mass = [-0.8476, 0.4238, 0.4238], [16.0, 1.0, 1.0]
        eps, sig = [78.208 / 0.120273 * 1e-3, 0, 0], [3.166, 0, 0]
    else:  # OPLS methanol, united-atom
        sites = [(0.0133, 0.7666, 0), (-0.0634, -0.6559, 0), (0.8152, -1.0042, 0)]
        q, mass = [0.265, -0.700, 0.435], [15.0, 16.0, 1.0]
        eps, sig = [0.207 * 4.184, 0.170 * 4.184, 0], [3.775, 3.070, 0]
    b, w = np.array(sites, float), np.array(mass)
    inertia = [float((w * (b[:, (a + 1) % 3] ** 2 + b[:, (a + 2) % 3] ** 2)).sum())
               for a in range(3)]
    return dict(sites=torch.tensor(b, dtype=F64, device=DEV), q=q, eps=eps, sig=sig,
                mass=float(w.sum()), inertia=torch.tensor(inertia, dtype=F64, device=DEV),
                st2=st2)


def matrices(q):
    """Body to lab rotation (..., 3, 3) of quaternions q (..., 4)."""
    a, b, c, d = q.unbind(-1)
    return torch.stack([
        a * a + b * b - c * c - d * d, -2 * (a * d + b * c), 2 * (b * d - a * c),
        2 * (a * d - b * c), a * a + c * c - b * b - d * d, -2 * (a * b + c * d),
        2 * (a * c + b * d), 2 * (a * b - c * d), a * a + d * d - b * b - c * c,
    ], -1).reshape(q.shape[:-1] + (3, 3))


def offsets(mod, q):
    return torch.matmul(mod["sites"], matrices(q).transpose(-1, -2).contiguous())


def candidates(xi, xj, L, r, same):
    """Padded rows idx (B, ni, w) of the j within r of each i, and their mask."""
    B, ni, _ = xi.shape
    nj = xj.shape[1]
    rows, width = [], 1
    step = max(1, 20_000_000 // (B * nj))
    for s in range(0, ni, step):
        dd = 0.0
        for a in range(3):
            d = xi[:, s:s + step, None, a] - xj[:, None, :, a]
            d = d - torch.round(d / L) * L
            dd = dd + d * d
        near = dd < r * r
        if same:
            at = torch.arange(s, min(ni, s + step), device=DEV)
            near[:, at - s, at] = False
        width = max(width, int(near.sum(-1).max()))
        rows.append(near)
    idx = torch.zeros((B, ni, width), dtype=torch.long, device=DEV)
    mask = torch.zeros((B, ni, width), dtype=torch.bool, device=DEV)
    s = 0
    for near in rows:
        b, i, j = near.nonzero(as_tuple=True)
        at = (near.cumsum(-1) - 1)[b, i, j]
        idx[b, s + i, at] = j
        mask[b, s + i, at] = True
        s += near.shape[1]
    return idx, mask


def pair_sums(mi, mj, xi, xj, si, sj, idx, mask, L, rc, taper):
    """Force and lab torque on every i, half the energy, virial and pair
    count of its rows (every pair is met from both sides)."""
    B = xi.shape[0]
    take = torch.arange(B, device=DEV)[:, None, None]
    d = xi[:, :, None] - xj[take, idx]
    d = d - torch.round(d / L) * L
    dd = (d * d).sum(-1)
    live = mask & (dd < rc * rc)
    # the places that pad a row: a molecule 5 A away, without weight
    d = torch.where(live[..., None], d, torch.tensor([5.0, 0.0, 0.0], dtype=F64, device=DEV))
    dd = torch.where(live, dd, torch.full_like(dd, 25.0))
    rin, r = rc - taper, dd.sqrt()
    u, l = r - rc, r - rin
    c1 = (1.0 / (rin - rc)) ** 5
    mid = r > rin
    S = torch.where(mid, c1 * u ** 3 * (10 * l * l - 5 * u * l + u * u), torch.ones_like(r)) * live
    dS = torch.where(mid, -30 * c1 * u * u * l * l / r, torch.zeros_like(r)) * live
    s12, ds12 = torch.ones_like(r), torch.zeros_like(r)
    if mi["st2"]:
        rl, ru = mi["st2"]
        w3 = (ru - rl) ** 3
        t = (r > rl) & (r < ru)
        s12 = torch.where(r <= rl, torch.zeros_like(r), s12)
        s12 = torch.where(t, (r - rl) ** 2 * (3 * ru - rl - 2 * r) / w3, s12)
        ds12 = torch.where(t, -6 * (r - rl) * (ru - r) / w3 / r, ds12)
    F, T = torch.zeros_like(xi), torch.zeros_like(xi)
    P = torch.zeros_like(d)
    ec, el = torch.zeros_like(r), torch.zeros_like(r)
    for a in range(len(mi["q"])):
        fa = torch.zeros_like(d)
        base = d + si[:, :, None, a]
        for b in range(len(mj["q"])):
            qq = mi["q"][a] * mj["q"][b] * COULOMB
            e = math.sqrt(mi["eps"][a] * mj["eps"][b])
            if qq == 0.0 and e == 0.0:
                continue
            v = base - sj[:, :, b][take, idx]
            i2 = 1.0 / (v * v).sum(-1)
            f = 0.0
            if qq != 0.0:
                c = qq * i2.sqrt()
                ec += c
                f = c * i2 * S * s12
            if e != 0.0:
                s6 = ((mi["sig"][a] + mj["sig"][b]) * 0.5) ** 6
                t6 = s6 * i2 ** 3
                el += 400.0 * e * (t6 * t6 - t6)
                f = f + 400.0 * e * i2 * (12 * t6 * t6 - 6 * t6) * S
            fa += v * f[..., None]
        P += fa
        fa = fa.sum(2)
        F += fa
        T += torch.linalg.cross(si[:, :, a], fa)
    cc = dS * (el + s12 * ec) + S * ds12 * ec
    P += cc[..., None] * d
    F += (cc[..., None] * d).sum(2)
    E = ((ec * s12 + el) * S).sum((1, 2)) * 0.5
    V = torch.stack([(d[..., a] * P[..., c]).sum((1, 2)) * 0.5 for a in range(3)
                     for c in range(3)], -1)
    return F, T, E, V, live.sum((1, 2)) * 0.5


class Rows:
    """Candidate rows between sets of molecules, kept while nothing moved far."""

    def __init__(self, mods, rc, taper, margin=1.5):
        self.mods, self.rc, self.taper, self.margin = mods, rc, taper, margin
        self.ref = None

    def forces(self, xs, qs, L):
        L = torch.as_tensor(L, dtype=F64, device=DEV)
        if L.dim() == 0:
            L = L.expand(3)
        if self.ref is not None:
            far = max(float((x - r).norm(dim=-1).max()) for x, r in zip(xs, self.ref))
            if 2 * far + float((L - self.L).norm()) > self.margin:
                self.ref = None
        if self.ref is None:
            self.ref, self.L, k = [x.clone() for x in xs], L.clone(), len(xs)
            self.rows = {(i, j): candidates(xs[i], xs[j], float(L[0]), self.rc + self.margin, i == j)
                         for i in range(k) for j in range(k)}
        out, parts = [], {}
        s = [offsets(m, q) for m, q in zip(self.mods, qs)]
        for i, mi in enumerate(self.mods):
            F = T = 0.0
            for j, mj in enumerate(self.mods):
                idx, mask = self.rows[(i, j)]
                f, t, e, v, p = pair_sums(mi, mj, xs[i], xs[j], s[i], s[j], idx, mask, L, self.rc,
                                          self.taper)
                F, T = F + f, T + t
                parts[(i, j)] = (e, v, p)
            out.append((F, T))
        E = sum(p[0] for p in parts.values())
        V = sum(p[1] for p in parts.values())
        n = sum(p[2] for p in parts.values())
        return out, E, V, n


def _randn(g, *shape):
    return torch.randn(shape, generator=g, dtype=F64).to(DEV)


def spin(w, q):
    """dq/dt of quaternions q turning with body-frame angular velocity w."""
    x, y, z = w.unbind(-1)
    a, b, c, d = q.unbind(-1)
    return 0.5 * torch.stack([-x * b + y * c - z * d, x * a - y * d - z * c,
                              -x * d - y * a + z * b, x * c + y * b + z * a], -1)


@functools.lru_cache(maxsize=64)
def liquid(names, counts, L, temp):
    """COMs and quaternions per component of a liquid: damped MD at 1 fs from
    a lattice with random orientations, the velocities drawn back to temp
    every step."""
    g = torch.Generator()
    g.manual_seed(1000 + sum(counts))
    n = sum(counts)
    side = math.ceil(n ** (1 / 3) - 1e-9)
    cell = torch.stack(torch.meshgrid(*[torch.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)
    cell = cell[torch.randperm(len(cell), generator=g)[:n].sort().values]
    x = ((cell + 0.5) * (L / side)).to(F64).to(DEV)
    which = torch.zeros(n, dtype=torch.long)
    if len(counts) > 1:
        which[torch.randperm(n, generator=g)[:counts[1]]] = 1
    which = which.to(DEV)
    q = _randn(g, n, 4)
    q = q / q.norm(dim=-1, keepdim=True)
    mods = [_model(m) for m in names]
    xs = [x[which == s][None].contiguous() for s in range(len(mods))]
    qs = [q[which == s][None].contiguous() for s in range(len(mods))]
    vs = [torch.zeros_like(x) for x in xs]
    ws = [torch.zeros_like(x) for x in xs]
    rows = Rows(mods, min(8.5, 0.5 * L - 0.1), 0.5, margin=min(1.5, 0.1 + 0.5 * max(0, L / 2 - 8.5)))
    dt = 0.001
    for _ in range(300):
        fs, _, _, _ = rows.forces(xs, qs, L)
        for s, m in enumerate(mods):
            tb = torch.matmul(fs[s][1][..., None, :], matrices(qs[s]))[..., 0, :]
            I = m["inertia"]
            w = ws[s]
            vs[s] = vs[s] + fs[s][0] * (dt / m["mass"])
            ws[s] = w + dt * (tb - torch.linalg.cross(w, w * I)) / I
            kt = RGAS / 10.0 * temp
            vs[s] = vs[s] * torch.sqrt(3 * kt / (m["mass"] * (vs[s] ** 2).sum(-1)).mean()).clamp(max=1.0)
            ws[s] = ws[s] * torch.sqrt(3 * kt / ((ws[s] ** 2 * I).sum(-1)).mean()).clamp(max=1.0)
            xs[s] = xs[s] + dt * vs[s].clamp(-40, 40)
            qs[s] = qs[s] + dt * spin(ws[s].clamp(-100, 100), qs[s])
            qs[s] = qs[s] / qs[s].norm(dim=-1, keepdim=True)
    return [(x[0], q[0]) for x, q in zip(xs, qs)]


def start(names, counts, L, k, temp, seed):
    """One start per component from the liquid: repeated k times per axis,
    every molecule moved and turned a little, Maxwell-Boltzmann velocities."""
    g = torch.Generator()
    g.manual_seed(seed)
    out = []
    for name, (x, q) in zip(names, liquid(tuple(names), tuple(counts), L / k, temp)):
        m = _model(name)
        cell = torch.stack(torch.meshgrid(*[torch.arange(k)] * 3, indexing="ij"), -1)
        x = (cell.reshape(-1, 1, 3).to(DEV) * (L / k) + x[None]).reshape(-1, 3)
        q = q.repeat(k ** 3, 1)
        # molecules in the order of a lattice's columns, as a start file lists them
        at = torch.remainder(x, L) / 3.1
        at = at.floor()
        order = torch.argsort(at[:, 0] * 1e4 + at[:, 1] * 1e2 + at[:, 2], stable=True)
        x, q = x[order], q[order]
        n = len(x)
        x = x + 0.01 * _randn(g, n, 3)
        q = q + 0.01 * _randn(g, n, 4)
        q = q / q.norm(dim=-1, keepdim=True)
        kt = RGAS / 10.0 * temp
        v = _randn(g, n, 3) * math.sqrt(kt / m["mass"])
        w = _randn(g, n, 3) * (kt / m["inertia"]).sqrt()
        out.append((x, q, v, w))
    return out


def nordsieck(s, dt):
    """(com, quat, dx, w) arrays as g6.System.upload takes them."""
    x, q, v, w = s
    n = len(x)
    dx, ww = np.zeros((5, 3, n)), np.zeros((5, 3, n))
    dx[0] = v.T.cpu().numpy() * dt
    ww[0] = w.T.cpu().numpy()
    return x.cpu().numpy(), q.cpu().numpy(), dx, ww


# ---- MD in plain torch: the Gear corrector, Nose thermostat and barostat ----

G5 = (3 / 16, 251 / 360, 1.0, 11 / 18, 1 / 6, 1 / 60)
G4 = (251 / 720, 1.0, 11 / 12, 1 / 3, 1 / 24)


def binomial(levels):
    """Taylor prediction of scaled derivatives."""
    n = len(levels)
    return [sum(math.comb(j, i) * levels[j] for j in range(i, n)) for i in range(n)]


def md_exact(mods, starts, L, rc, taper, dt, steps, nose=None, baro=None):
    """steps MD steps of B systems; starts per component (x, q, v, w) with a
    batch axis; nose = (T (B,), Q) or None; baro = (pressure, mass) or None."""
    B = starts[0][0].shape[0]
    X = [[x] + [v * dt] + [torch.zeros_like(x)] * 4 for x, q, v, w in starts]
    W = [[w] + [torch.zeros_like(w)] * 4 for x, q, v, w in starts]
    Q = [[q] + [torch.zeros_like(q)] * 4 for x, q, v, w in starts]
    n = sum(x[0].shape[1] for x in X)
    dof = 6.0 * n
    zeta = [torch.zeros(B, dtype=F64, device=DEV) for _ in range(5)]
    zsum = torch.zeros(B, dtype=F64, device=DEV)
    box = torch.full((3,), float(L), dtype=F64, device=DEV)
    if baro:
        vol = [box.prod()] + [torch.zeros((), dtype=F64, device=DEV)] * 5
    rows = Rows(mods, rc, taper)
    rescale = lambda b: b * (vol[0] / b.prod()) ** (1 / 3)  # noqa: E731
    for _ in range(steps):
        if nose:
            zeta = binomial(zeta)
        if baro:
            vol = binomial(vol)
            box = rescale(box)
        drag = zeta[0][:, None, None] * dt
        for s in range(len(mods)):
            X[s], W[s] = binomial(X[s]), binomial(W[s])
            p = binomial(Q[s])
            # the orientation is predicted in value and first derivative
            Q[s] = [p[0] / p[0].norm(dim=-1, keepdim=True), p[1]] + Q[s][2:]
        fs, E, V, count = rows.forces([x[0] for x in X], [q[0] for q in Q], box)
        K, ek, kin = 0.0, [], 0.0
        for s, m in enumerate(mods):
            I = m["inertia"]
            tb = torch.matmul(fs[s][1][..., None, :], matrices(Q[s][0]))[..., 0, :]
            w0 = W[s][0]
            ext = drag * 0.5 + (vol[1] / (6.0 * vol[0]) if baro else 0.0)
            new = fs[s][0] * (dt * dt * 0.5 / m["mass"]) - X[s][1] * ext
            d = new - X[s][2]
            X[s] = [x + c * d for x, c in zip(X[s], G5)]
            new = (tb - torch.linalg.cross(w0, w0 * I)) * dt / I - w0 * drag
            d = new - W[s][1]
            W[s] = [w + c * d for w, c in zip(W[s], G4)]
            q = Q[s]
            q0 = q[0] + G4[0] * (spin(w0, q[0]) * dt - q[1])
            lv = [q0]
            for j in range(1, 5):  # derivatives of q from the corrected w
                lv.append(sum(spin(W[s][i], lv[j - 1 - i]) for i in range(j)) * (dt / j))
            Q[s] = lv
            v = X[s][1]
            et = (v * v).sum((1, 2)) * m["mass"] * 0.5 / (dt * dt)
            er = ((W[s][0] ** 2) * I).sum((1, 2)) * 0.5
            K = K + et + er
            ek.append((et, er))
            kin = kin + torch.einsum("bna,bnc->bac", v, v).reshape(B, 9) * (m["mass"] / (dt * dt))
        T = 20.0 * K / (RGAS * dof)
        if nose:
            zf = (T - nose[0]) / nose[1]
            d = zf - zeta[1]
            zeta = [z + c * d for z, c in zip(zeta, G4)]
            zsum = zsum + zeta[0]
        if baro:
            vp = sum(kin[0, a] + V[0, a] for a in (0, 4, 8))
            press = vp / 3.0 * 10.0 / 101326.0 / (box.prod() * 6.0225e23 * 1e-30)
            d = (press - baro[0]) / baro[1] * 0.5 - vol[2]
            vol = [x + c * d for x, c in zip(vol, G5)]
            box = rescale(box)
    return X, Q, W, dict(energy=E, temperature=T, virial=V, kinetic=kin, pairs=count)


def answer(com, quat, dx, w, th):
    """What a program reads after a log interval."""
    return dict(com=com, quat=quat, dx=dx, w=w, energy=th[..., 0].copy(),
                temperature=th[..., 3].copy(), virial=th[..., 4:13].copy(),
                kinetic=th[..., 16:25].copy(), pairs=th[..., 14].copy())


def exact_answer(X, Q, W, th, s=0, b=0):
    lv = lambda t: np.stack([x[b].T.cpu().numpy() for x in t])  # noqa: E731
    one = lambda k: th[k][b].cpu().numpy()  # noqa: E731
    return dict(com=X[s][0][b].cpu().numpy(), quat=lv(Q[s]), dx=lv(X[s][1:]), w=lv(W[s]),
                **{k: one(k) for k in ("energy", "temperature", "virial", "kinetic", "pairs")})


DT, TAPER = 0.002, 0.5
MODEL = dict(tip4p=g6.TIP4P, tip5p=g6.TIP5P, st2=g6.ST2, spce=g6.SPCE, meoh=g6.OPLSMEOH)
BARO = (1.0, 1e-4)  # @PCN4: 1 atm and the reference's mass


def system(c, name, n, L, rc, s, nose_t=None):
    y = g6.System(MODEL[name], n, L, rc, TAPER, DT, prec=g6.FP64 if c.get("fp64") else g6.FP32,
                  skin=c["skin"])
    com, q, dx, w = nordsieck(s, DT)
    y.upload(com, q, dx, w)
    if nose_t:
        y.set_nose(nose_t, nose_t * 2500.0)
    return y


def temps(c):
    return [220.0 * (320.0 / 220.0) ** (k / max(1, c["rungs"] - 1)) for k in range(c["rungs"])]


def ladder_start(n, L, k, T, seed):
    return start(["tip4p"], [REPEAT[n][0]], L, REPEAT[n][1], 270.0, seed + 1000 * n + k)[0]


# ---- Monte Carlo and the surrogate in plain torch and numpy -----------------

def bf16(x):
    return torch.as_tensor(x, dtype=torch.float32).to(torch.bfloat16).to(F64).to(DEV)


def pair_matrix(x, q, L, rc=9.0):
    """The TIP4P pair energies e (n, n) (internal units), zero diagonal."""
    m = _model("tip4p")
    s = offsets(m, q)
    d = x[:, None] - x[None]
    o = torch.round(d / L) * L
    d = d - o
    dd = (d * d).sum(-1).fill_diagonal_(1e4)
    r, rin = dd.sqrt(), rc - TAPER
    u, l = r - rc, r - rin
    S = torch.where(r > rin, (1.0 / (rin - rc)) ** 5 * u ** 3 * (10 * l * l - 5 * u * l + u * u),
                    torch.ones_like(r)) * (dd < rc * rc)
    e = torch.zeros_like(r)
    for a in range(4):
        for b in range(4):
            qq, ee = m["q"][a] * m["q"][b] * COULOMB, m["eps"][a] * m["eps"][b]
            if qq == 0.0 and ee == 0.0:
                continue
            v = s[:, None, a] + x[:, None] - s[None, :, b] - x[None] - o
            i2 = 1.0 / (v * v).sum(-1)
            if qq != 0.0:
                e += qq * i2.sqrt()
            else:
                t6 = m["sig"][0] ** 6 * i2 ** 3
                e += 400.0 * m["eps"][0] * (t6 * t6 - t6)
    return torch.where(S > 0, e * S, torch.zeros_like(e))


def features(x, q, L):
    """The 32 symmetry functions of every molecule (n, 32), within 6 A."""
    s = offsets(_model("tip4p"), q) + x[:, None]
    O, H, n = s[:, 0], s[:, 2:4], len(x)
    idx, mask = candidates(O[None], O[None], L, 6.0, True)
    idx, mask = idx[0], mask[0].to(F64)
    d = O[idx] - O[:, None]
    d = d - torch.round(d / L) * L
    r = torch.where(mask > 0, (d * d).sum(-1), torch.ones_like(mask)).sqrt()
    fc = 0.5 * (torch.cos(math.pi * r / 6.0) + 1.0) * mask
    out = [(torch.exp(-4.0 * (r - mu) ** 2) * fc).sum(1) for mu in 2.4 + 0.5 * np.arange(8)]
    ra = (O[:, None, None] + d[:, :, None] - H[:, None]).norm(dim=-1)
    rb = (H[idx] - O[idx][:, :, None] + d[:, :, None]).norm(dim=-1)
    for rh in (ra, rb):
        out += [(torch.exp(-10.0 * (rh - mu) ** 2).sum(-1) * fc).sum(1) for mu in (1.6, 1.9, 2.2, 2.6)]
    cs = torch.matmul(d, d.transpose(1, 2).contiguous()) / (r[:, :, None] * r[:, None])
    tri = torch.triu(torch.ones(r.shape[1], r.shape[1], dtype=F64, device=DEV), 1)
    ff = fc[:, :, None] * fc[:, None] * tri
    e2 = r[:, :, None] ** 2 + r[:, None] ** 2
    for eta in (0.02, 0.08):
        ex = torch.exp(-eta * e2) * ff
        for lam in (1.0, -1.0):
            out += [2.0 ** (1 - z) * ((1.0 + lam * cs) ** z * ex).sum((1, 2)) for z in (1, 2, 4, 8)]
    return torch.stack(out, 1)


def split(params):
    p = torch.as_tensor(params, dtype=F64, device=DEV)
    a = np.cumsum([0, 2048, 64, 4096, 64, 64, 1])
    W1, b1, W2, b2, w3, b3 = (p[a[i]:a[i + 1]] for i in range(6))
    return W1.view(64, 32), b1, W2.view(64, 64), b2, w3, b3


def network(params, norm, x):
    """Energies of feature rows: BF16 weights, everything else in 64 bits."""
    W1, b1, W2, b2, w3, b3 = split(params)
    nm = torch.as_tensor(norm, dtype=F64, device=DEV)
    h = torch.nn.functional.silu((x - nm[:32]) * nm[32:64] @ bf16(W1).T + b1)
    h = torch.nn.functional.silu(h @ bf16(W2).T + b2)
    return nm[65] * (h @ w3 + b3) + nm[64]


@functools.lru_cache(maxsize=32)
def screen(n, L):
    """A network for delayed acceptance: fixed random layers, the output
    layer fitted to the pair energies of a few configurations of the liquid."""
    xs, es = [], []
    for k in range(6):
        x, q, _, _ = start(["tip4p"], [n], L, 1, 250.0, 77 + k)[0]
        f = 0.99 + 0.004 * k
        xs.append(features(x * f, q, L * f))
        es.append(0.5 * pair_matrix(x * f, q, L * f).sum(1))
    x, e = torch.cat(xs), torch.cat(es)
    norm = torch.cat([x.mean(0), 1.0 / x.std(0).clamp(min=1e-6), e.mean()[None], e.std()[None]])
    g = torch.Generator()
    g.manual_seed(3)
    W1 = (torch.rand(64, 32, generator=g, dtype=F64) - 0.5) * 0.5
    W2 = (torch.rand(64, 64, generator=g, dtype=F64) - 0.5) * 0.6
    z = torch.zeros(64, dtype=F64)
    par = torch.cat([W1.reshape(-1), z, W2.reshape(-1), z, z, z[:1]])
    h = torch.nn.functional.silu((x - norm[:32]) * norm[32:64] @ bf16(W1).T)
    h = torch.nn.functional.silu(h @ bf16(W2).T).cpu()
    t = ((e - norm[64]) / norm[65]).cpu()
    A = h.T @ h + 1e-3 * len(h) * torch.eye(64, dtype=F64)
    par[2048 + 64 + 4096 + 64:-1] = torch.linalg.solve(A, h.T @ (t - t.mean()))
    return par.numpy().astype(np.float32), norm.cpu().numpy().astype(np.float32)


def philox(idx, slot, key):
    """Philox4x32-10 of counter (idx, slot, tag): four numbers in (0, 1)."""
    M = 0xFFFFFFFF
    c, k = [idx & M, idx >> 32, slot, 0x4E505400], [key & M, key >> 32]
    for _ in range(10):
        p0, p1 = 0xD2511F53 * c[0], 0xCD9E8D57 * c[2]
        c = [(p1 >> 32) ^ c[1] ^ k[0], p1 & M, (p0 >> 32) ^ c[3] ^ k[1], p0 & M]
        k = [(k[0] + 0x9E3779B9) & M, (k[1] + 0xBB67AE85) & M]
    return [(v + 0.5) * 2.0 ** -32 for v in c]


NPT = dict(temp=250.0, bar=1.0, disp=0.15, rot=8.0, dlnv=0.005, pvol=1.0 / 28.0, voxa=9.0)


def quat_mul(p, q):
    a, b, c, d = p
    w, x, y, z = q
    return np.array([a * w - b * x - c * y - d * z, a * x + b * w + c * z - d * y,
                     a * y - b * z + c * w + d * x, a * z + b * y - c * x + d * w])


def proposal(x, q, L, idx, key):
    """(volume move?, ln V'/V, x, q, L, exact uniform, surrogate uniform); x
    is None for a void move."""
    u = philox(idx, 0, key)
    if u[0] < NPT["pvol"]:
        lnv = NPT["dlnv"] * (2.0 * u[1] - 1.0)
        s = math.exp(lnv / 3.0)
        return True, lnv, None if 18.0 >= L * s else x * s, q, L * s, u[2], u[3]
    nd = max(1, int(L / NPT["voxa"]))
    cell = min(int(u[1] * nd ** 3), nd ** 3 - 1)
    o = np.array(philox(idx, 0xFFFF, key)[:3]) * (L / nd)

    def cell_of(y):
        y = y - o
        # halves of a cell go away from zero
        away = lambda v: np.sign(v) * np.floor(np.abs(v) + 0.5)  # noqa: E731
        y = y - away(y / L) * L
        j = np.mod(away(y * (nd / L)).astype(int), nd)
        return (j[:, 2] * nd + j[:, 1]) * nd + j[:, 0]

    X, Qn = x.copy(), q.copy()
    members = np.nonzero(cell_of(x) == cell)[0]
    d = NPT["disp"] / math.sqrt(3.0)
    e = math.tan(0.5 * NPT["rot"] * math.pi / 180.0) / math.sqrt(3.0)
    for k, i in enumerate(members):
        a, b = philox(idx, 1 + 2 * k, key), philox(idx, 2 + 2 * k, key)
        X[i] += d * (2.0 * np.array(a[:3]) - 1.0)
        t = quat_mul(np.array([1.0] + [e * (2.0 * v - 1.0) for v in (a[3], b[0], b[1])]), q[i])
        Qn[i] = t / np.linalg.norm(t)
    if len(members) > 96 or (cell_of(X[members]) != cell).any():
        X = None
    return False, 0.0, X, Qn, L, u[2], u[3]


def npt_exact(c, x, q, L, seed, net):
    dev = lambda a: torch.as_tensor(a, dtype=F64, device=DEV)  # noqa: E731
    energy = lambda x, q, L: float(pair_matrix(dev(x), dev(q), L).sum()) * 0.5  # noqa: E731
    surrogate = lambda x, q, L: float(network(*net, features(dev(x), dev(q), L)).sum())  # noqa: E731
    beta, pk, n = 1.0 / NPT["temp"], NPT["bar"] * 1e5 * 1e-30 / 1.380066e-23, len(x)
    U = energy(x, q, L)
    Us = surrogate(x, q, L) if c["K"] else 0.0
    accepted = 0

    def weight(du, volume, lnv, L2):
        arg = -du * I2J * J2K * beta
        return arg - pk * (L2 ** 3 - L ** 3) * beta + (n + 1) * lnv if volume else arg

    for move in range(c["moves"]):
        got, off = None, 0.0
        for k in range(max(1, c["K"])):
            volume, lnv, x2, q2, L2, u, us = proposal(x, q, L, move * max(1, c["K"]) + k, seed)
            if x2 is None:
                continue
            if c["K"]:
                U2s = surrogate(x2, q2, L2)
                arg = weight(U2s - Us, volume, lnv, L2)
                if not (arg >= 0.0 or us < math.exp(arg)):
                    continue
                off = U2s - Us
            got = (volume, lnv, x2, q2, L2, u)
            break
        if got is None:
            continue
        volume, lnv, x2, q2, L2, u = got
        U2 = energy(x2, q2, L2)
        arg = -(U2 - U - off) * I2J * J2K * beta if c["K"] else weight(U2 - U, volume, lnv, L2)
        if arg >= 0.0 or u < math.exp(arg):
            x, q, L, U, Us = x2, q2, L2, U2, Us + off
            accepted += 1
    return dict(com=x, quat=q.T.copy(), edge=L, energy=U, accepted=accepted)


def stream(seed):
    """The 31-bit uniforms of MT19937 (init_genrand), 1 - x."""
    b = np.random.MT19937()
    b._legacy_seeding(int(seed))
    while True:
        for v in b.random_raw(4096):
            yield int(v)


def mc_exact(c, x, q, L, seed):
    """mc2's trials: Gaussian turn and displacement of one molecule."""
    n, rc, beta = c["n"], 9.0, 1.0 / 300.0
    raw = stream(seed)
    u = np.array([1.0 - (next(raw) >> 1) / 2147483648.0 for _ in range(14 * c["trials"] + 2)])
    z = np.sqrt(-2.0 * np.log(u[:-1])) * np.sin(2.0 * math.pi * u[1:])
    x, q = x.copy(), q.copy()
    P = pair_matrix(torch.as_tensor(x, device=DEV), torch.as_tensor(q, device=DEV), L).cpu().numpy()
    eps = float(np.triu(P, 1).sum())
    m = _model("tip4p")
    body, rin = m["sites"].cpu().numpy(), rc - TAPER
    sites = lambda x, q: x[:, None] + body @ matrices(torch.as_tensor(q)).numpy().transpose(0, 2, 1)  # noqa: E731
    s = sites(x, q)
    delta, ratio = np.full(n, 0.2), np.full(n, 0.5)
    inc, floor = float(np.float32(1.05)), float(np.float32(0.05))
    pos = accepted = 0
    for _ in range(c["trials"]):
        t = min(int(u[pos] * n + 1.0) - 1, n - 1)
        dt, dr = delta[t], delta[t] * ratio[t]
        rot, move = z[pos + 1:pos + 7:2] * dr, z[pos + 7:pos + 13:2] * dt
        pos += 13
        a, b, e, f = np.array([1.0, *rot]) / math.sqrt(1.0 + (rot ** 2).sum())
        w, i, j, k = q[t]
        qn = np.array([a * w - b * i - e * j - f * k, a * i + b * w + e * k - f * j,
                       a * j + e * w - b * k + f * i, a * k + f * w + b * j - e * i])
        qn = -qn if qn[0] < 0 else qn
        xn = x[t] + move
        sn = sites(xn[None], qn[None])[0]
        d = x - xn
        o = np.round(d / L) * L
        r = np.sqrt(((d - o) ** 2).sum(1))
        near = np.nonzero(r < rc)[0]
        near = near[near != t]
        v = s[near][:, :, None] - sn[None, None] - o[near][:, None, None]
        i2 = 1.0 / (v ** 2).sum(-1)
        t6 = m["sig"][0] ** 6 * i2[:, 0, 0] ** 3
        en = 400.0 * m["eps"][0] * (t6 * t6 - t6)
        en = en + (np.sqrt(i2[:, 1:, 1:]) * np.outer(m["q"][1:], m["q"][1:])).sum((1, 2)) * COULOMB
        rr = r[near]
        p, l = rr - rc, rr - rin
        S = np.where(rr > rin, (1.0 / (rin - rc)) ** 5 * p ** 3 * (10 * l * l - 5 * p * l + p * p), 1.0)
        new = np.zeros(n)
        new[near] = en * S
        de = float((new - P[t]).sum())
        ok = de < 0.0
        if not ok:
            ok = u[pos] < math.exp(-de * I2J * J2K * beta)
            pos += 1
        if ok:
            accepted += 1
            eps += de
            P[t], P[:, t] = new, new
            x[t], q[t], s[t] = xn, qn, sn
            delta[t] *= inc
            ratio[t] = ratio[t] * inc if np.abs(move).mean() * ratio[t] < np.abs(rot).mean() else ratio[t] / inc
        else:
            delta[t] = max(delta[t] / inc, floor)
    return dict(com=x, quat=q, delta=delta, ratio=ratio, energy=eps, accepted=accepted)


def training_rows(c, seed):
    """Feature-like rows and targets: an analytic function of them."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    x = torch.randn(c["rows"], 32, generator=g, device=DEV) * 0.6 + 1.5
    mix = torch.linspace(-1, 1, 32, device=DEV)
    t = torch.tanh(x[:, ::2].mean(1) - 1.5) * 300.0 + torch.sin(x @ mix) * 100.0 - 2000.0
    norm = np.concatenate([np.full(32, 1.5), np.full(32, 1 / 0.6), [-2000.0, 110.0]])
    return x.cpu().numpy(), t.cpu().numpy(), norm.astype(np.float32)


def train_exact(c, seed):
    x, t, norm = training_rows(c, seed)
    par = torch.as_tensor(g6_params(seed), dtype=F64, device=DEV)
    xd, td = torch.as_tensor(x, device=DEV).to(F64), torch.as_tensor(t, device=DEV).to(F64)
    td = (td - float(norm[64])) / float(norm[65])
    raw, m = stream(11), c["rows"]
    perm = list(range(m))
    mo, ve, step, losses = torch.zeros_like(par), torch.zeros_like(par), 0, []
    unit = np.concatenate([norm[:64], [0.0, 1.0]])
    for _ in range(c["epochs"]):
        for k in range(m - 1, 0, -1):
            r = next(raw) % (k + 1)
            perm[k], perm[r] = perm[r], perm[k]
        order = torch.tensor(perm, device=DEV)
        loss = []
        for b in range(m // c["batch"]):
            at = order[b * c["batch"]:(b + 1) * c["batch"]]
            # the gradient at the BF16 weights goes to the master weights
            w = par.clone()
            w[:2048], w[2112:6208] = bf16(par[:2048]), bf16(par[2112:6208])
            w.requires_grad_(True)
            W1, b1, W2, b2, w3, b3 = split(w)
            nm = torch.as_tensor(unit, dtype=F64, device=DEV)
            h = torch.nn.functional.silu((xd[at] - nm[:32]) * nm[32:64] @ W1.T + b1)
            h = torch.nn.functional.silu(h @ W2.T + b2)
            ls = ((h @ w3 + b3 - td[at]) ** 2).mean()
            g, = torch.autograd.grad(ls, w)
            step += 1
            mo, ve = 0.9 * mo + 0.1 * g, 0.999 * ve + 0.001 * g * g
            par = par - 2e-3 * (mo / (1 - 0.9 ** step)) / ((ve / (1 - 0.999 ** step)).sqrt() + 1e-8)
            loss.append(float(ls.detach()))
        losses.append(sum(loss) / len(loss))
    return dict(params=par.cpu().numpy(), loss=np.array(losses))


def g6_params(seed):
    r = np.random.default_rng(seed)
    a1, a2, a3 = math.sqrt(6 / 96), math.sqrt(6 / 128), math.sqrt(6 / 65)
    return np.concatenate([r.uniform(-a1, a1, 2048), np.zeros(64), r.uniform(-a2, a2, 4096),
                           np.zeros(64), r.uniform(-a3, a3, 64), [0.0]]).astype(np.float32)


# ---- what a program has in hand, and one pass --------------------------------

def mc_edge(n):
    return round((n / DENSITY) ** (1 / 3), 3)


def mixture_edge(c):
    return round(3.625 * c["k"] * (c["water"] + c["meoh"]) ** (1 / 3), 3)


def prepare(c, seed):
    if c["kind"] == "md":
        s, = start([c["model"]], [c["m"]], c["L"], c["k"], 300.0, seed)
        y = system(c, c["model"], molecules(c), c["L"], c["rc"], s, 300.0 if c["nose"] else None)
        if c["baro"]:
            y.set_andersen(*BARO)
        return c, y
    if c["kind"] == "ladder":
        ys = []
        for n, L in chosen(c):
            for k, T in enumerate(temps(c)):
                ys.append(system(c, "tip4p", n, L, 9.0, ladder_start(n, L, k, T, seed), T))
        return c, g6.Ladder(ys)
    if c["kind"] == "mixture":
        sw, sm = start(["tip4p", "meoh"], [c["water"], c["meoh"]], mixture_edge(c), c["k"], 300.0, seed)
        L = mixture_edge(c)
        rc = mixture_rc(c)
        w = system(c, "tip4p", len(sw[0]), L, rc, sw, 300.0)
        m = system(c, "meoh", len(sm[0]), L, rc, sm)
        return c, g6.Mixture(w, m)
    if c["kind"] in ("mc", "npt"):
        L = mc_edge(c["n"])
        temp = 300.0 if c["kind"] == "mc" else NPT["temp"]
        s, = start(["tip4p"], [c["n"]], L, 1, temp, seed)
        y = g6.System(g6.TIP4P, c["n"], L, 9.0, TAPER, DT, prec=g6.FP64, skin=0.0)
        com, q, dx, w = nordsieck(s, DT)
        y.upload(com, q, dx, w)
        if c["kind"] == "mc":
            y.mc_begin(temp, seed % 2 ** 32, 0.2, 0.5)
            return c, y
        y.npt_begin(NPT["temp"], NPT["bar"], seed, NPT["disp"], NPT["rot"], NPT["dlnv"],
                    NPT["pvol"], NPT["voxa"])
        return c, (y, g6.Mlp(*screen(c["n"], L)) if c["K"] else None)
    x, t, norm = training_rows(c, seed)
    return c, (g6.Mlp(g6_params(seed), norm), x, t)


def mixture_rc(c):
    return min(8.5, math.floor(10 * (mixture_edge(c) / 2 - c["skin"] - 0.05)) / 10)


def run(state):
    c, y = state
    if c["kind"] == "md":
        y.step(c["steps"])
        return answer(*y.download(), y.thermo())
    if c["kind"] == "ladder":
        y.step(c["steps"])
        th = y.thermo()
        got = [s.download() for s in y.systems]
        out, at = [], 0
        for _ in chosen(c):
            part = got[at:at + c["rungs"]]
            out.append(answer(*[np.stack(a) for a in zip(*part)], th[at:at + c["rungs"]]))
            at += c["rungs"]
        return out
    if c["kind"] == "mixture":
        y.step(c["steps"])
        th, parts = y.thermo()
        out = [answer(*s.download(), th) for s in (y.first, y.second)]
        return out + [parts[:3]]
    if c["kind"] == "mc":
        accepted = y.mc_trials(c["trials"])
        com, q, d, r, e = y.mc_state()
        return dict(com=com, quat=q, delta=d, ratio=r, energy=e, accepted=int(accepted))
    if c["kind"] == "npt":
        s, net = y
        n = s.npt_run(c["moves"], mlp=net, K=c["K"]) if c["K"] else s.npt_run(c["moves"])
        com, q, L, U = s.npt_state()
        return dict(com=com, quat=q, edge=L, energy=U, accepted=n["accepted"])
    net, x, t = y
    loss = net.train(x, t, c["epochs"], c["batch"], 2e-3, 11)
    return dict(params=net.get()[0], loss=loss)


def exact(c, seed):
    batch = lambda s: tuple(a[None] for a in s)  # noqa: E731
    if c["kind"] == "md":
        s, = start([c["model"]], [c["m"]], c["L"], c["k"], 300.0, seed)
        n = molecules(c)
        nose = (torch.tensor([300.0], dtype=F64, device=DEV), 300.0 * 2500.0 * DT) if c["nose"] else None
        baro = (BARO[0], BARO[1] * 6.0 * n / DT ** 2) if c["baro"] else None
        return exact_answer(*md_exact([_model(c["model"])], [batch(s)], c["L"], c["rc"], TAPER, DT,
                                      c["steps"], nose, baro))
    if c["kind"] == "ladder":
        out = []
        for n, L in chosen(c):
            T = temps(c)
            s = [ladder_start(n, L, k, t, seed) for k, t in enumerate(T)]
            T = torch.tensor(T, dtype=F64, device=DEV)
            got = md_exact([_model("tip4p")], [tuple(torch.stack(a) for a in zip(*s))], L, 9.0, TAPER,
                           DT, c["steps"], (T, T * 2500.0 * DT))
            one = [exact_answer(*got, b=b) for b in range(c["rungs"])]
            out.append({k: np.stack([o[k] for o in one]) for k in one[0]})
        return out
    if c["kind"] == "mixture":
        s = start(["tip4p", "meoh"], [c["water"], c["meoh"]], mixture_edge(c), c["k"], 300.0, seed)
        nose = (torch.tensor([300.0], dtype=F64, device=DEV), 300.0 * 2500.0 * DT)
        got = md_exact([_model("tip4p"), _model("meoh")], [batch(a) for a in s], mixture_edge(c),
                       mixture_rc(c), TAPER, DT, c["steps"], nose)
        return [exact_answer(*got, s=k) for k in (0, 1)] + [None]
    if c["kind"] in ("mc", "npt"):
        L = mc_edge(c["n"])
        x, q, _, _ = start(["tip4p"], [c["n"]], L, 1, 300.0 if c["kind"] == "mc" else NPT["temp"], seed)[0]
        x, q = x.cpu().numpy(), q.cpu().numpy()
        if c["kind"] == "mc":
            return mc_exact(c, x, q, L, seed % 2 ** 32)
        return npt_exact(c, x, q, L, seed, screen(c["n"], L) if c["K"] else None)
    return train_exact(c, seed)
