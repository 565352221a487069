"""Systems past the wide kernels' limit, against the oracle.

A split-2 or 4 launch of at most WIDE_TILES tiles takes the wide first and
force passes, so the parity tests' small systems check those; here a system of
a few tiles more takes the kernels that large runs take, at every split and in
every mode:

  setup        densities, forces, energies and virials of the start
  run 1        the same of the last step's pass, on the engine's own state
               (positions, half-step velocities, densities, wall fractions and
               signatures), which the end-of-run kick has not changed
  run 1 twice  equals run 2 bit for bit: the fused pass applies the forces that
               the first run's last pass, checked above, wrote
  dump         the fused pass with output writes those forces

Tolerances: densities as in the parity tests.  Forces, energies and virials
1e-5 over the system, as there; per particle twice that: the largest of 33,000
errors of one distribution is expected at 4.6 of its widths, of the parity
tests' 2,400 at 3.9.
"""
import os
import re

import numpy as np
import pytest
from scipy.spatial import cKDTree

from conftest import PKG, uniform_box
from test_gpu_arb import DECK
from test_gpu_parity import DR_FP32, SEED, dpd_system, mdpd_system, oracle_params

pytestmark = pytest.mark.gpu

N = 33000
WALLS = (30.0, 10.0, 28.0)


def wide_tiles():
    text = open(os.path.join(PKG, "csrc", "kernels_step.hip")).read()
    return int(re.search(r"constexpr int WIDE_TILES = (\d+);", text).group(1))


def walls_box():
    # as the wall tests' channel, 33,600 particles
    rng = np.random.default_rng(5)
    lx, ly, lz = WALLS
    nw, nf = int(8.0 * lx * 2.0 * lz), int(3.0 * lx * 8.0 * lz)
    wy = rng.uniform(0, 2.0, nw)
    walls = np.c_[rng.uniform(0, lx, nw), np.where(wy < 1.0, wy, wy + 8.0), rng.uniform(0, lz, nw)]
    fluid = np.c_[rng.uniform(0, lx, nf), rng.uniform(0.8, 9.2, nf), rng.uniform(0, lz, nf)]
    v = np.zeros((nf + nw, 3))
    v[:nf] = rng.normal(0, 1, (nf, 3))
    x = np.r_[fluid, walls]
    return x.astype(np.float32).astype(np.float64), v.astype(np.float32).astype(np.float64), \
        np.r_[np.ones(nf, np.int32), np.full(nw, 2, np.int32)]


class Case:
    """One kind of system: how to make it and its forces in 64 bits."""

    def __init__(self, engine, orc, kind):
        self.engine, self.orc, self.kind = engine, orc, kind
        self.dt = {"dpd": 0.04}.get(kind, 0.01)
        self.L = (N / (3.0 if kind == "dpd" else 6.05)) ** (1.0 / 3.0)
        if kind == "walls":
            self.x, self.v, self.types = walls_box()
            self.L = WALLS
            self.p = orc.params((0, 0, 0), WALLS, 0.01, mass=(1.0, 1.0), ntypes=2, cut=1.0, cut_r=0.75,
                                A=np.array([[-40.0, -20.0], [-20.0, -40.0]]), B=25.0, gamma=18.0, sigma=6.0)
        else:
            self.x, self.v = uniform_box(N, self.L, 77)
            self.types = np.ones(N, np.int32)
            if kind == "two types":
                self.types[::3] = 2
                g = np.array([[4.5, 4.5], [4.5, 2.0]])
                self.p = orc.params((0, 0, 0), (self.L,) * 3, 0.01, ntypes=2, mass=(1.0, 1.0), cut=[[1, 1], [1, 0.9]],
                                    cut_r=[[0.75, 0.75], [0.75, 0.7]], A=[[-40, -30], [-30, -20]],
                                    B=[[25, 25], [25, 20]], gamma=g, sigma=np.sqrt(2 * g), expw=1.0)
            elif kind == "dpd":
                self.p = orc.params((0, 0, 0), (self.L,) * 3, 0.04, cut=1.0, A=25.0, gamma=4.5, sigma=3.0, expw=1.0)
            else:
                self.p = oracle_params(orc, self.L)
        self.n = len(self.x)
        self.t0 = self.types - 1
        self.mask = np.where(self.types == 2, 1 | 4, 1 | 2) if kind == "walls" else np.ones(self.n, int)
        self.moves = self.types == 1 if kind == "walls" else np.ones(self.n, bool)

    def make(self, split):
        e, kind = self.engine, self.kind
        if kind == "walls":
            s = e.System()
            s.command("atom_style mdpd/atomic/meso 8.0")
            s.create_box(2, (0, 0, 0), WALLS)
            s.create_atoms(self.types, self.x, self.v)
            s.commands(DECK)
        elif kind == "two types":
            s = mdpd_system(e, self.x, self.v, self.L, types=self.types, ntypes=2, coeff="1 1 -40 25 4.5 1.0 0.75",
                            extra="pair_coeff 1 2 -30 25 4.5 1.0 0.75\npair_coeff 2 2 -20 20 2.0 0.9 0.7")
        elif kind == "dpd":
            s = dpd_system(e, self.x, self.v, self.L)
        else:
            s = mdpd_system(e, self.x, self.v, self.L, lucy=kind == "lucy")
        s.tune("split", split)
        return s

    def check(self, s, step, kick):
        """The last pass of s (it read the velocities before a half-kick)."""
        orc = self.orc
        x, v, f = s.gather("x"), s.gather("v"), s.gather("f")
        if kick:
            v[self.moves] -= 0.5 * self.dt * f[self.moves]
        sig = s.debug_signatures()
        if self.kind == "dpd":
            want = orc.force_dpd(x, v, sig, self.t0, self.p)
        else:
            seed = 2654868 if self.kind == "walls" else SEED
            assert np.array_equal(sig, orc.sig_mdpd(np.arange(1, self.n + 1), orc.seed_now(seed, step)))
            lucy = self.kind == "lucy"
            ref = orc.density(x, self.t0, np.ones(self.n, int), self.p, 0.75, lucy=lucy)
            rho = s.gather("rho")
            # the parity tests' floor: the steepest weight times a distance's
            # FP32 error, for each neighbor within r_d
            box = np.broadcast_to(self.L, (3,))
            tree = cKDTree(x % box, boxsize=box)
            near = tree.query_ball_point(x % box, 0.75 * 1.001, return_length=True) - 1
            slope = 16.0 / 9.0 * 105.0 / (16.0 * np.pi * 0.75**7) * 0.75**3 if lucy else 15.0 / (np.pi * 0.75**4)
            assert np.all(np.abs(rho - ref) <= 1e-5 * ref + near * slope * DR_FP32), step
            if self.kind == "walls":
                a = orc.arb(2, 4, cut_phi=1.0, phi_c=0.5, rho_wall=8.0)
                want = orc.force_mdpd_arb(x, v, rho, sig, self.t0, self.mask, s.gather("phi"), self.p, a)
            else:
                want = orc.force_mdpd(x, v, rho, sig, self.t0, self.p)
        for got, ref, what in zip((f, s.gather("e_pair"), s.gather("virial")), want, ("force", "energy", "virial")):
            got, ref = got.reshape(self.n, -1), ref.reshape(self.n, -1)
            err, mag = np.linalg.norm(got - ref, axis=1), np.linalg.norm(ref, axis=1)
            worst = np.max(err / np.maximum(mag, np.sqrt(np.mean(mag**2))))
            glob = np.linalg.norm(err) / np.linalg.norm(mag)
            print(f"step {step}, {what}: global {glob:.2e}, worst {worst:.2e}")
            assert glob <= 1e-5 and worst <= 2e-5, (step, what)


@pytest.mark.parametrize("split", [1, 2, 4])
@pytest.mark.parametrize("kind", ["liquid", "lucy", "two types", "dpd", "walls"])
def test_large_system_matches_oracle(engine, orc, tmp_path, kind, split):
    case = Case(engine, orc, kind)
    assert (case.n + 255) // 256 * 4 > wide_tiles()
    a, b = case.make(split), case.make(split)
    a.setup()
    case.check(a, 0, False)
    a.run(1)
    case.check(a, 1, True)
    f1 = a.gather("f")
    a.run(1)
    b.command(f"dump d all custom 1 {tmp_path}/d id fx fy fz")
    b.run(2)
    for k in ("x", "v", "f", "rho", "phi"):
        np.testing.assert_array_equal(a.gather(k), b.gather(k), err_msg=k)
    frames = open(tmp_path / "d").read().split("ITEM: ATOMS id fx fy fz\n")[1:]
    rows = np.array([r.split() for r in frames[1].split("ITEM")[0].splitlines()], dtype=np.float64)
    out = np.empty((case.n, 3))
    out[rows[:, 0].astype(int) - 1] = rows[:, 1:]
    np.testing.assert_array_equal(out.astype(np.float32), f1.astype(np.float32))
    a.close()
    b.close()
