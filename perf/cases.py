"""Performance cases of the mdpd355 engine: what its users run, from one
small droplet on a handle of its own to a pool of 256.

Every case advances simulations by a number of steps through the public
Python host module and takes back the particles' unwrapped positions (the
columns xu yu zu of a dump) and velocities.  The engine keeps both in FP32
and its gather widens them, so they are returned as float32.

listed()   the named cases;  draw(rng)  one more of the same ranges
prepare()  what a program holds before the call: handles set up at their
           first step, or an open pool and the configured systems of its jobs
run()      one pass: `run N` on a handle, or a whole batch of pool jobs
work()     bytes and operations a pass cannot do without
exact()    the same trajectory in 64 bits, in plain torch
"""
import math
import os
import statistics
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "usermeso-2.0-mdpd_amd"))

RHO, RC, RD, SKIN, DT = 6.05, 1.0, 0.75, 0.3, 0.01


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest liquid anyone runs: launches and latency count
        {"name": "droplet-1k", "kind": "droplet", "n": 1000, "steps": 80},
        # the median droplet of a size study, alone on a handle
        {"name": "droplet-9k", "kind": "droplet", "n": 8667, "steps": 80},
        # a large droplet, the top of the study's sizes
        {"name": "droplet-40k", "kind": "droplet", "n": 40001, "steps": 60},
        # the classic DPD fluid (the other pair style): L = 22, density 3, dt = 0.04
        {"name": "dpd-32k", "kind": "dpd", "n": 32000, "steps": 60},
        # the liquid slab of the contact-angle example, with the Lucy weight
        {"name": "slab-97k", "kind": "slab", "n": 96800, "steps": 50},
        # the largest slab one handle is asked for
        {"name": "slab-194k", "kind": "slab", "n": 193600, "steps": 50},
        # the slab watched while it runs: g(r) every 10 steps and a density profile
        {"name": "observed-97k", "kind": "observed", "n": 96800, "steps": 50},
        # slit channel: frozen lattice walls, wall fractions and bounce-back, two types
        {"name": "channel-122k", "kind": "channel", "n": 122400, "steps": 50},
        # pore flow past frozen grains under a body force, two types: the largest single system
        {"name": "pore-480k", "kind": "pore", "n": 480000, "steps": 20},
        # a small batch of droplets in one pool
        {"name": "batch-24", "kind": "batch", "n": 24, "steps": 80},
        # the batch a size study submits at once: 256 droplets, 2.4 million particles
        {"name": "batch-256", "kind": "batch", "n": 256, "steps": 80},
        # jobs arriving at a pool that runs others: droplets and slabs, 1,000 to 200,000 particles
        {"name": "served-24", "kind": "served", "n": 24, "steps": 60},
    ]


def draw(rng):
    kind = rng.choice(["droplet", "droplet", "dpd", "slab", "observed", "channel", "pore", "batch", "served"])
    lo, hi = {"droplet": (1000, 60000), "dpd": (3000, 200000), "slab": (15000, 200000), "observed": (15000, 120000),
              "channel": (15000, 160000), "pore": (40000, 480000), "batch": (8, 192), "served": (8, 32)}[kind]
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if kind == "pore":
        return {"kind": kind, "n": n, "steps": rng.randint(10, 20)}
    return {"kind": kind, "n": n, "steps": rng.randint(30, 80)}


# ---------------------------------------------------------------------------
# inputs: particles spread evenly at random, as a liquid's are (a Kronecker
# sequence from a random start, jittered), in no spatial order, as a data
# file lists them; Maxwell velocities at kT = 1
# ---------------------------------------------------------------------------
def _spread(rng, n):
    g = 1.2207440846057596                    # root of g^4 = g + 1: the sequence of best spread in 3-D
    a = np.array([1 / g, 1 / g ** 2, 1 / g ** 3])
    return (rng.random(3) + np.arange(1, n + 1)[:, None] * a) % 1.0


def _f32(a):
    return a.astype(np.float32).astype(np.float64)


def _inside(x, box):
    """Wrapped into the box, in FP32 (the float just below L stays below it)."""
    x = _f32(x % np.asarray(box))
    top = np.nextafter(np.float32(1.0) * np.asarray(box, np.float32), np.float32(0)).astype(np.float64)
    return np.minimum(x, top)


def _velocities(rng, n):
    v = rng.normal(0.0, 1.0, (n, 3))
    return _f32(v - v.mean(axis=0))


def _droplet(rng, n):
    R = (3.0 * n / (4.0 * np.pi * RHO)) ** (1.0 / 3.0)
    L = 2.5 * R
    p = (_spread(rng, int(2.0 * n) + 200) * 2.0 - 1.0) * R
    p = p[(p ** 2).sum(axis=1) < R * R][:n]
    x = p + L / 2 + rng.normal(0.0, 0.05, (n, 3))
    return {"box": (L, L, L), "x": _inside(x, (L, L, L)), "v": _velocities(rng, n), "deck": "liquid"}


def _slab(rng, n, box=None, thick=10.0):
    if box is None:                           # the repository's two slabs are 40 wide
        ly = max(n / (RHO * thick * 40.0), 8.0)
        box = (n / (RHO * thick * ly), ly, 2.0 * thick)
    x = _spread(rng, n) * np.array([box[0], box[1], thick]) + np.array([0.0, 0.0, thick / 2])
    x += rng.normal(0.0, 0.05, (n, 3))
    return {"box": tuple(box), "x": _inside(x, box), "v": _velocities(rng, n), "deck": "liquid", "lucy": True}


def _slab_job(rng, n):
    side = math.sqrt(n / (RHO * 10.0))
    return _slab(rng, n, box=(side, side, 20.0))


def _dpd(rng, n):
    L = (n / 3.0) ** (1.0 / 3.0) if n != 32000 else 22.0
    x = _spread(rng, n) * L + rng.normal(0.0, 0.05, (n, 3))
    return {"box": (L, L, L), "x": _inside(x, (L, L, L)), "v": _velocities(rng, n), "deck": "dpd"}


def _channel(rng, n):
    lz = 0.5 * round(2.0 * n / (40.0 * (RHO * 10.0 + 16.0)))
    box = (40.0, 12.0, max(lz, 4.5))
    g = lambda lo, hi: np.arange(lo, hi, 0.5) + 0.25                                # noqa: E731
    walls = np.stack(np.meshgrid(g(0.0, box[0]), np.r_[g(0.0, 1.0), g(11.0, 12.0)], g(0.0, box[2]), indexing="ij"),
                     -1).reshape(-1, 3)
    nf = n - len(walls)
    fluid = _spread(rng, nf) * np.array([box[0], 9.8, box[2]]) + np.array([0.0, 1.1, 0.0])
    fluid += np.clip(rng.normal(0.0, 0.03, (nf, 3)), -0.09, 0.09)
    types = np.r_[np.ones(nf, np.int32), np.full(len(walls), 2, np.int32)]
    v = np.zeros((n, 3))
    v[:nf] = _velocities(rng, nf)
    return {"box": box, "x": _inside(np.r_[fluid, walls], box), "v": v, "types": types, "deck": "channel"}


def _pore(rng, n):
    lz = 4.0
    ly = max(100.0 * math.sqrt(n / 480000.0), 24.0)
    lx = n / (6.0 * lz * ly)
    box = np.array([lx, ly])
    discs, area = [], 0.0
    while area < 0.40 * lx * ly:
        r, c = rng.uniform(4.0, 10.0) * min(1.0, ly / 60.0), rng.uniform((0, 0), (lx, ly))
        if all(np.hypot(*((c - q) - box * np.round((c - q) / box))) >= r + rq for q, rq in discs):
            discs.append((c, r))
            area += np.pi * r * r
    x = _spread(rng, n) * np.array([lx, ly, lz]) + rng.normal(0.0, 0.05, (n, 3))
    x = _inside(x, (lx, ly, lz))
    wall = np.zeros(n, bool)
    for q, r in discs:
        d = x[:, :2] - q
        d -= box * np.round(d / box)
        wall |= (d * d).sum(axis=1) < r * r
    v = _velocities(rng, n)
    v[wall] = 0.0
    return {"box": (lx, ly, lz), "x": x, "v": v, "types": np.where(wall, 1, 2).astype(np.int32), "deck": "pore"}


def _sizes(case):
    """Particles of each simulation of a case (a batch's sizes lie on the
    quantiles of LogNormal(ln 8000, 0.5) in [2000, 40000], served ones on those
    of the log-uniform law from 1,000 to 200,000)."""
    k, n = case["kind"], case["n"]
    if k == "batch":
        z = statistics.NormalDist(math.log(8000.0), 0.5)
        return [int(min(max(math.exp(z.inv_cdf((i + 0.5) / n)), 2000), 40000)) for i in range(n)]
    if k == "served":
        return [int(1000.0 * 200.0 ** ((i + 0.5) / n)) for i in range(n)]
    return [n]


def _systems(case, seed):
    """The simulations of a case: box, particles, deck and TEA seed of each."""
    rng = np.random.default_rng([seed, case["n"], case["steps"]])
    kind = case["kind"]
    make = {"droplet": _droplet, "slab": _slab, "observed": _slab, "dpd": _dpd, "channel": _channel, "pore": _pore,
            "batch": _droplet}
    sizes = _sizes(case)
    if kind in ("batch", "served"):           # jobs come in no order of size
        sizes = [sizes[i] for i in rng.permutation(len(sizes))]
    out = []
    for i, n in enumerate(sizes):
        f = make[kind] if kind != "served" else (_droplet, _slab_job)[i % 2]
        out.append(dict(f(rng, n), seed=int(rng.integers(1, 1 << 30))))
    return out


# ---------------------------------------------------------------------------
# decks: the repository's own workloads
# ---------------------------------------------------------------------------
DECKS = {
    "liquid": """
        mass 1 1.0
        pair_style mdpd/meso 1.0 1.0 {seed}
        pair_coeff * * -40 25 4.5 1.0 0.75
        fix rho all aboundary/rho/meso cut_rho 0.75 {weight}
        fix int all nve/meso
        timestep 0.01
    """,
    "dpd": """
        mass 1 1.0
        pair_style dpd/meso 1.0 {seed}
        pair_coeff * * 25.0 4.5 3.0 1.0 1.0
        fix int all nve/meso
        timestep 0.04
    """,
    "channel": """
        mass * 1.0
        group fluid type 1
        group wall type 2
        pair_style mdpd/meso 1.0 1.0 {seed} fluid wall
        pair_coeff 1 1 -40 25 18.0 1.0 0.75
        pair_coeff 1 2 -20 25 18.0 1.0 0.75
        pair_coeff 2 2 -40 25 18.0 1.0 0.75
        fix BC all aboundary/rho/meso cut_rho 0.75 phi_c 0.5 cut_phi 1.0 rho_wall 8.0 wall wall mobile fluid
        fix int fluid nve/meso
        timestep 0.01
    """,
    "pore": """
        mass * 1.0
        group fluid type 2
        pair_style mdpd/meso 1.0 1.0 {seed}
        pair_coeff 1 1 -40 25 4.5 1.0 0.75
        pair_coeff 1 2 -40 0 4.5 1.0 0.75
        pair_coeff 2 2 -40 25 4.5 1.0 0.75
        fix rho all aboundary/rho/meso cut_rho 0.75
        fix push fluid addforce/meso 0.02 0 0
        fix int fluid nve/meso
        timestep 0.01
    """,
}
DENSITY = {"liquid": "mdpd/atomic/meso 6.05", "dpd": "dpd/atomic/meso", "channel": "mdpd/atomic/meso 8.0",
           "pore": "mdpd/atomic/meso 6.0"}


def _handle(m):
    import mdpd355
    s = mdpd355.System(0)
    s.command("atom_style " + DENSITY[m["deck"]])
    types = m.get("types")
    s.create_box(1 if types is None else 2, (0, 0, 0), m["box"])
    s.create_atoms(np.ones(len(m["x"]), np.int32) if types is None else types, m["x"], m["v"])
    s.commands("neighbor 0.3 bin\nneigh_modify every 1 delay 0 check yes\n"
               + DECKS[m["deck"]].format(seed=m["seed"], weight="weight lucy" if m.get("lucy") else "")
               + "\nrun_style mvv/meso")
    return s


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------
class _Keep:
    """What one state owns; closed with it."""

    def __init__(self, handles, boxes, steps):
        self.handles, self.boxes, self.steps = handles, boxes, steps
        self.pool = self.tmp = None

    def __del__(self):
        for h in self.handles + ([self.pool] if self.pool is not None else []):
            h.close()
        if self.tmp is not None:
            self.tmp.cleanup()


def prepare(case, seed):
    import mdpd355
    made = _systems(case, seed)
    k = _Keep([_handle(m) for m in made], [np.array(m["box"]) for m in made], case["steps"])
    k.kind = case["kind"]
    if k.kind in ("batch", "served"):
        # the batch is resident at once; the served jobs share half of the
        # memory they would take together, so some wait for others to finish
        slots = sum((len(m["x"]) + 255) // 256 * 256 for m in made)
        want = 1500.0 * slots + float(1 << 22)
        if k.kind == "served":
            want = max(0.5 * want, 1500.0 * 1.3 * max(len(m["x"]) for m in made) + float(1 << 24))
        k.pool = mdpd355.Pool(want, max(len(made), 16))
        k.pool.tune("split", 1)               # a fixed launch shape: results reproducible bit for bit
    else:
        if k.kind == "observed":
            k.tmp = tempfile.TemporaryDirectory()
            k.handles[0].commands(
                f"fix g all rdf/fast/meso output {k.tmp.name}/rdf.out nbin 100 every 10\n"
                f"fix p all density/meso output {k.tmp.name}/prof along z nbin 40 every 50 window 10")
        k.handles[0].setup()
    return k


def _unwrapped(x, image, box):
    return (x + image * box).astype(np.float32)


def run(state):
    if state.pool is None:
        s = state.handles[0]
        s.run(state.steps)
        out = {"x": _unwrapped(s.gather("x"), s.gather("image"), state.boxes[0]),
               "v": s.gather("v").astype(np.float32)}
        if state.kind == "observed":
            out["g"] = s.fix_result("g")[1]
            out["profile"] = s.fix_result("p")[1]
        return out
    p = state.pool
    if state.kind == "batch":
        ids = [p.submit(s, state.steps) for s in state.handles]
    else:                                     # two more jobs arrive with every eight passes
        ids = []
        for i in range(0, len(state.handles), 2):
            ids += [p.submit(s, state.steps) for s in state.handles[i:i + 2]]
            p.advance(max_passes=8)
    p.run()
    x = [_unwrapped(p.gather(j, "x"), p.gather(j, "image"), b) for j, b in zip(ids, state.boxes)]
    v = [p.gather(j, "v").astype(np.float32) for j in ids]
    for j in ids:
        p.release(j)
    p.done()
    return {"x": np.concatenate(x), "v": np.concatenate(v)}


def work(case):
    """Per particle and step: position, velocity and random signature read and
    written once, the density written and read; every pair inside the cutoff
    evaluated once (four TEA rounds, the Gaussian and the force: ~150
    operations), plus each density weight (~12)."""
    n = sum(_sizes(case))
    rho = 3.0 if case["kind"] == "dpd" else RHO
    pairs = 0.5 * rho * 4.0 / 3.0 * math.pi
    weights = 0.0 if case["kind"] == "dpd" else pairs * RD ** 3
    per = n * case["steps"]
    return {"bytes": per * (28.0 + 28.0 + 8.0) + n * 24.0, "flops": per * (150.0 * pairs + 12.0 * weights)}


# ---------------------------------------------------------------------------
# the trajectory in 64 bits (mDPD; a DPD particle's random signature is made
# from the FP32 bits of its velocity, so those trajectories have no 64-bit
# value, nor has the histogram of a float's bins)
# ---------------------------------------------------------------------------
M32 = 0xFFFFFFFF


def _tea(v0, v1, rounds):
    s = 0
    for _ in range(rounds):
        s = (s + 0x9E3779B9) & M32
        v0 = (v0 + (((v1 << 4) + 0xA341316C) ^ (v1 + s) ^ ((v1 >> 5) + 0xC8013EA4))) & M32
        v1 = (v1 + (((v0 << 4) + 0xAD90777D) ^ (v0 + s) ^ ((v0 >> 5) + 0x7E95761E))) & M32
    return v0, v1


def _premix(v0, v1, rounds):
    v0, v1 = _tea(v0, v1, rounds)
    return v0 ^ v1


def _brev(x):
    r = torch.zeros_like(x)
    for b in range(32):
        r |= ((x >> b) & 1) << (31 - b)
    return r


def _gauss(si, sj):
    v0, v1 = _tea(torch.maximum(si, sj), torch.minimum(si, sj), 4)
    t = ((v0 & 0x7FFFFFFF) - (1 << 30)).double() / 2.0 ** 31
    f = torch.sin(math.pi * t)
    f = torch.where((v0 & 0x80000000) != 0, -f, f)
    r = torch.sqrt(-2.0 * torch.log(torch.clamp(v1, min=1).double() / 2.0 ** 32))
    return torch.clamp(r * f, -4.0, 4.0)


class _Exact:
    def __init__(self, m):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        t = lambda a: torch.as_tensor(a, dtype=torch.float64, device=dev)           # noqa: E731
        self.x, self.v, self.L, self.dev = t(m["x"]), t(m["v"]), t(m["box"]), dev
        n, self.deck, self.seed, self.lucy = len(m["x"]), m["deck"], m["seed"], bool(m.get("lucy"))
        self.n = n
        types = m.get("types")
        self.ty = torch.zeros(n, dtype=torch.int64, device=dev) if types is None else \
            torch.as_tensor(types, dtype=torch.int64, device=dev) - 1
        A, B, g, fluid = {"liquid": ([[-40]], [[25]], 4.5, None),
                          "channel": ([[-40, -20], [-20, -40]], [[25, 25], [25, 25]], 18.0, 0),
                          "pore": ([[-40, -40], [-40, -40]], [[25, 0], [0, 25]], 4.5, 1)}[self.deck]
        self.A, self.B, self.gamma = t(A).reshape(-1), t(B).reshape(-1), g
        self.nt = len(A)
        self.moves = torch.ones(n, 1, dtype=torch.float64, device=dev) if fluid is None else \
            (self.ty == fluid).double()[:, None]
        self.push = t([0.02, 0.0, 0.0]) * self.moves if self.deck == "pore" else 0.0
        self.phi = torch.zeros(n, dtype=torch.float64, device=dev)
        self.tag = _brev(torch.arange(1, n + 1, device=dev))
        self.hold = None

    def pairs(self):
        """Pairs i < j with r < rc + skin at the last listing; listed anew when a particle has moved skin / 2."""
        if self.hold is not None and float(((self.x - self.hold) ** 2).sum(1).max()) < (0.49 * SKIN) ** 2:
            return self.pi, self.pj
        self.hold = self.x.clone()
        L, dev = self.L, self.dev
        w = self.x - L * torch.floor(self.x / L)
        nc = torch.clamp((L / (RC + SKIN)).floor().long(), min=3)
        c = torch.minimum((w / L * nc).long(), nc - 1)
        cell = (c[:, 2] * nc[1] + c[:, 1]) * nc[0] + c[:, 0]
        ncell = int(nc.prod())
        order = torch.argsort(cell)
        count = torch.bincount(cell, minlength=ncell)
        start = torch.cumsum(count, 0) - count
        cap = int(count.max())
        table = torch.full((ncell, cap), -1, dtype=torch.int64, device=dev)
        table[cell[order], torch.arange(self.n, device=dev) - start[cell[order]]] = order
        full = torch.nonzero(count > 0)[:, 0]
        cz, cy, cx = full // (nc[0] * nc[1]), full // nc[0] % nc[1], full % nc[0]
        got = []
        step = max(1, (1 << 25) // (cap * cap))
        for k in range(14):                   # half of the stencil, the cell itself among it
            ox, oy, oz = (k + 13) % 3 - 1, (k + 13) // 3 % 3 - 1, (k + 13) // 9 - 1
            other = ((cz + oz) % nc[2] * nc[1] + (cy + oy) % nc[1]) * nc[0] + (cx + ox) % nc[0]
            for b in range(0, len(full), step):
                i, j = table[full[b:b + step]][:, :, None], table[other[b:b + step]][:, None, :]
                d = w[i.clamp(min=0)] - w[j.clamp(min=0)]
                d = d - L * torch.round(d / L)
                ok = ((d * d).sum(-1) < (RC + SKIN) ** 2) & (i >= 0) & (j >= 0)
                if k == 0:
                    ok &= i < j
                a, p, q = torch.nonzero(ok, as_tuple=True)
                got.append((i[a, p, 0], j[a, 0, q]))
        self.pi, self.pj = torch.cat([g[0] for g in got]), torch.cat([g[1] for g in got])
        return self.pi, self.pj

    def near(self, cut):
        i, j = self.pairs()
        d = self.x[i] - self.x[j]
        d = d - self.L * torch.round(d / self.L)
        r2 = (d * d).sum(1)
        k = torch.nonzero((r2 < cut * cut) & (r2 >= 1e-20))[:, 0]
        return i[k], j[k], d[k], torch.sqrt(r2[k])

    def forces(self, step):
        i, j, d, r = self.near(RC)
        h = RD
        wr = torch.clamp(h - r, min=0.0)
        if self.lucy:
            wt, f = (h + 3.0 * r) * wr ** 3, 105.0 / (16.0 * math.pi * h ** 7)
        else:
            wt, f = wr ** 2, 15.0 / (2.0 * math.pi * h ** 5)
        rho = torch.zeros(self.n, dtype=torch.float64, device=self.dev)
        rho.index_add_(0, i, wt).index_add_(0, j, wt)
        rho *= f
        sig = _premix(self.tag, torch.full_like(self.tag, _premix(self.seed, step, 64)), 32)
        ti, tj = self.ty[i], self.ty[j]
        A, B = self.A[ti * self.nt + tj], self.B[ti * self.nt + tj]
        wc, wcr = 1.0 - r / RC, torch.clamp(1.0 - r / RD, min=0.0)
        dot = (d * (self.v[i] - self.v[j])).sum(1)
        xi = _gauss(sig[i], sig[j])
        base = A * wc + B * (rho[i] + rho[j]) * wcr
        drag, kick = -self.gamma * wc * wc * dot / r, math.sqrt(2.0 * self.gamma) * wc * xi / math.sqrt(DT)
        fi = fj = (base + drag + kick) / r
        if self.deck == "channel":            # pairs of a mobile particle with a wall particle, on the mobile side
            def scaled(mob, wall, phi):
                ph = torch.clamp(phi, max=0.5)
                hh = torch.clamp(1.0 - (2.088 * ph ** 3 + 1.478 * ph) ** 0.25, min=0.025) * RC
                q = 1.0 + 0.187 * (RC / hh - 1.0) - 0.093 * (1.0 - hh / RC) ** 3
                return torch.where((mob == 0) & (wall == 1), (base + q * drag + torch.sqrt(q) * kick) / r, fi)
            fi, fj = scaled(ti, tj, self.phi[i]), scaled(tj, ti, self.phi[j])
        F = torch.zeros_like(self.x)
        F.index_add_(0, i, d * fi[:, None]).index_add_(0, j, -d * fj[:, None])
        return F + self.push

    def walls(self):
        """Wall fraction of the mobile particles; those deeper than one half bounce back."""
        if self.deck != "channel":
            return
        i, j, d, r = self.near(1.0)
        i, j, d, r = torch.cat([i, j]), torch.cat([j, i]), torch.cat([d, -d]), torch.cat([r, r])
        k = torch.nonzero((self.ty[i] == 0) & (self.ty[j] == 1))[:, 0]
        i, d, r = i[k], d[k], r[k]
        phi = torch.zeros_like(self.phi).index_add_(0, i, (1.0 + 3.0 * r) * (1.0 - r) ** 3)
        self.phi = phi * 105.0 / (16.0 * math.pi * 8.0)
        nrm = torch.zeros_like(self.x).index_add_(0, i, d * (1.0 - r)[:, None] ** 2)
        b = torch.nonzero(self.phi > 0.5)[:, 0]
        nn = nrm[b] / nrm[b].norm(dim=1, keepdim=True)
        old = self.x[b] - self.v[b] * 0.5 * DT
        into = torch.clamp((self.v[b] * nn).sum(1, keepdim=True), min=0.0)
        self.v[b] = -self.v[b] + 2.0 * into * nn
        self.x[b] = old + DT * self.v[b]

    def run(self, steps):
        f = self.forces(0)
        for t in range(1, steps + 1):
            self.v += 0.5 * DT * f * self.moves
            self.x += DT * self.v * self.moves
            self.walls()
            f = self.forces(t)
            self.v += 0.5 * DT * f * self.moves
        return self.x.cpu().numpy(), self.v.cpu().numpy()


def exact(case, seed):
    # a trajectory of more than ~50 million particle-steps takes over 20 seconds
    if case["kind"] == "dpd" or sum(_sizes(case)) * case["steps"] > 5e7:
        return None
    got = [_Exact(m).run(case["steps"]) for m in _systems(case, seed)]
    out = {"x": np.concatenate([g[0] for g in got]), "v": np.concatenate([g[1] for g in got])}
    if case["kind"] == "observed":
        out["g"] = out["profile"] = None
    return out
