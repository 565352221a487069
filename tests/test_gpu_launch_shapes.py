"""The per-step kernels' launch shapes agree bit for bit.

A small system on a handle of its own takes the wide first and force passes;
the same system in a pool, whose launches cover at least 65,536 slots, takes
the two- or four-wave ones at the same split.  Both add the same terms in the
same order, so positions, velocities, forces and densities are equal.
"""
import numpy as np
import pytest

from conftest import uniform_box
from test_gpu_arb import DECK, LX, LY, LZ, channel
from test_gpu_parity import IDX, _neighbor_sets, dpd_system, mdpd_system

pytestmark = pytest.mark.gpu


def _box(engine, n, L, **kw):
    x, v = uniform_box(n, L, 100 + n)
    return mdpd_system(engine, x, v, L, **kw)


def _two_types(engine):
    n, L = 1500, 6.5
    x, v = uniform_box(n, L, 17)
    types = np.where(np.arange(n) % 3 == 0, 2, 1).astype(np.int32)
    return mdpd_system(engine, x, v, L, types=types, ntypes=2, coeff="1 1 -40 25 4.5 1.0 0.75",
                       extra="pair_coeff 1 2 -30 25 4.5 1.0 0.75\npair_coeff 2 2 -20 20 2.0 0.9 0.7")


def _walls(engine):
    x, v, types, _ = channel()
    s = engine.System()
    s.command("atom_style mdpd/atomic/meso 8.0")
    s.create_box(2, (0, 0, 0), (LX, LY, LZ))
    s.create_atoms(types, x, v)
    s.commands(DECK)
    return s


def _dpd(engine):
    x, v = uniform_box(648, 6.0, 5)
    return dpd_system(engine, x, v, 6.0)


def _uneven(engine):
    # a liquid next to its vapor: rows of none to ~50 pairs in one tile, the
    # longest dealt over several rounds of raising the common part
    x, v = uniform_box(700, 5.0, 23)
    gas, _ = uniform_box(500, 12.0, 24)
    x = np.concatenate([x, gas[np.any(gas > 5.5, axis=1)]])
    return mdpd_system(engine, x, np.random.default_rng(2).normal(size=x.shape), 12.0)


CASES = {
    "one": lambda e: _box(e, 1, 4.0),
    "tile - 1": lambda e: _box(e, 63, 4.0),
    "tile": lambda e: _box(e, 64, 4.0),
    "tile + 1": lambda e: _box(e, 65, 4.0),
    "liquid": lambda e: _box(e, 1296, 6.0),
    "lucy": lambda e: _box(e, 1296, 6.0, lucy=True),
    # ~170 entries and ~80 pairs a row: several rounds of chunks and of pairs
    "dense": lambda e: _box(e, 1200, 4.0, rho_est=18.75, extra="timestep 0.001"),
    "two types": _two_types,
    "uneven": _uneven,
    "walls": _walls,
    "dpd": _dpd,
}


@pytest.mark.parametrize("split", [2, 4])
@pytest.mark.parametrize("case", list(CASES))
def test_small_system_equals_its_pool_job(engine, case, split):
    s = CASES[case](engine)
    p = engine.Pool(float(1 << 29), 16)
    p.tune("split", split)
    j = p.submit(s, 12)
    p.run()
    s.tune("split", split)
    s.run(12)
    for k in ("x", "v", "f", "rho"):
        a = s.gather(k)
        assert np.isfinite(a).all()
        np.testing.assert_array_equal(p.gather(j, k), a, err_msg=f"{case}, split {split}: {k}")
    p.close()
    s.close()


# (particles, box edge): the one-launch sort at its smallest, at one particle
# per thread and past it, at its largest and past it; a box of too many cells
# for it (several chunks of the one-launch scan); one past that scan's largest
@pytest.mark.parametrize("n, L", [(300, 5.3), (1024, 5.6), (1025, 5.6), (2000, 13.1), (2000, 14.4), (10240, 12.0),
                                  (10241, 12.0), (3000, 27.5), (4000, 46.0)])
def test_sorted_order_over_scan_sizes(engine, orc, n, L):
    x, v = uniform_box(n, L, int(10 * L))
    s = mdpd_system(engine, x, v, L)
    s.setup()
    xc = orc.wrap(x.astype(np.float32), (0, 0, 0), (L, L, L))
    keys = orc.sort_keys(xc, (0, 0, 0), (L, L, L), 1.3)
    origin, got, _ = s.debug_sorted()
    assert np.array_equal(origin, orc.stable_sort(keys))
    assert np.array_equal(got, keys[origin])
    # after re-sorts on the step path every table still belongs to its positions
    s.run(30)
    assert s.nbuild >= 2
    origin, got, xw = s.debug_sorted()
    assert np.array_equal(np.sort(origin), np.arange(n))
    assert np.array_equal(got, orc.sort_keys(xw, (0, 0, 0), (L, L, L), 1.3))
    assert np.all(np.diff(got.astype(np.int64)) >= 0)
    # and so do the rows (a cell's centres shared by four waves up to 2,560 cells)
    counts, rows = s.debug_neighbors()
    mine = _neighbor_sets(origin, counts, rows)
    xc = np.empty_like(xw)
    xc[origin] = xw
    _, want = orc.neighbors(xc, (0, 0, 0), (L, L, L), 1.3)
    for i in range(n):
        assert mine[i] == {(int(e) & IDX, int(e) >> 27) for e in want[i]}, i
    s.close()


# the one-launch sort is taken by the steps between re-sorts (a slow fluid's
# many: up to its largest; a re-sort every step: up to a third of that)
@pytest.mark.parametrize("n, extra", [(10240, "timestep 0.001"), (10241, "timestep 0.001"),
                                      (3072, "neigh_modify every 1 delay 0 check no"),
                                      (3400, "neigh_modify every 1 delay 0 check no")])
def test_sorted_order_over_resort_rates(engine, orc, n, extra):
    L = (n / 6.05) ** (1.0 / 3.0)
    x, v = uniform_box(n, L, n)
    s = mdpd_system(engine, x, v, L, extra=extra)
    s.setup()
    keys = orc.sort_keys(orc.wrap(x.astype(np.float32), (0, 0, 0), (L, L, L)), (0, 0, 0), (L, L, L), 1.3)
    origin, got, _ = s.debug_sorted()
    assert np.array_equal(origin, orc.stable_sort(keys))
    assert np.array_equal(got, keys[origin])
    s.run(40)
    origin, got, xw = s.debug_sorted()
    assert np.array_equal(np.sort(origin), np.arange(n))
    assert np.array_equal(got, orc.sort_keys(xw, (0, 0, 0), (L, L, L), 1.3))
    assert np.all(np.diff(got.astype(np.int64)) >= 0)
    s.close()


# within a graph of several steps the rebuild phase makes the commit of the
# step before, launched by itself the commit is its own launch: the one-launch
# sort, the one-launch scan, the chunked scan, wall passes, a pool's jobs
@pytest.mark.parametrize("case", ["one", "liquid", "dpd", "walls", (10241, 12.0), (4000, 46.0)], ids=str)
@pytest.mark.parametrize("neigh", ["every 1 delay 0 check yes", "every 3 delay 5 check yes", "every 2 delay 4 check no"])
def test_graph_steps_equal_single_launches(engine, case, neigh):
    def make():
        s = CASES[case](engine) if isinstance(case, str) else _box(engine, *case)
        s.command("neigh_modify " + neigh)
        return s
    steps = 27
    got = []
    for graph in (0, 1):
        s = make()
        s.tune("split", 2)
        s.tune("graph", graph)
        s.run(steps)
        got.append([s.gather(k) for k in ("x", "v", "f", "image")] + [s.nbuild])
        s.close()
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)
    for graph in (0, 1):
        p = engine.Pool(float(1 << 29), 16)
        p.tune("split", 2)
        p.tune("graph", graph)
        made = [make(), make()]
        jobs = [p.submit(made[0], steps), p.submit(made[1], 5)]
        p.run()
        for k, want in zip(("x", "v", "f", "image"), got[0]):
            np.testing.assert_array_equal(p.gather(jobs[0], k), want, err_msg=f"pool, graph {graph}: {k}")
        p.close()
        for s in made:
            s.close()


def test_jobs_harvested_together_equal_their_own_runs(engine):
    # two mDPD jobs and a DPD job end in the same pass, with a longer two-type
    # job between them (evaluated by the same launches only once it has ended)
    # and a box of far more cells than particles; the second batch is packed
    # into pinned memory at submission
    def systems():
        x, v = uniform_box(700, 5.0, 8)
        sparse = uniform_box(10, 20.0, 9)
        return [(mdpd_system(engine, x, v, 5.0), 15), (_two_types(engine), 22), (_dpd(engine), 15),
                (mdpd_system(engine, *sparse, 20.0), 15)]
    ref = []
    for s, k in systems():
        s.tune("split", 1)
        s.run(k)
        ref.append({q: s.gather(q) for q in ("x", "v", "f", "image", "e_pair", "virial", "tag", "type", "mask")})
        s.close()
    p = engine.Pool(float(1 << 29), 16)
    p.tune("split", 1)
    for batch in range(2):
        ids = [p.submit(s, k) for s, k in systems()]
        p.run()
        for j, want in zip(ids, ref):
            for q, w in want.items():
                np.testing.assert_array_equal(p.gather(j, q), w, err_msg=f"batch {batch}, job {j}: {q}")
            p.release(j)
    p.close()


# four waves share a tile's rows, a chunk of eight entries each in turn: fewer
# rows than a tile, a partial and a full one, rows shorter than a chunk and
# (1,200 particles in a box of 4) of some twenty chunks
@pytest.mark.parametrize("n, L", [(2, 4.0), (63, 4.0), (65, 4.0), (257, 4.0), (1200, 4.0)])
def test_rdf_counts_every_pair_once_from_each_side(engine, tmp_path, n, L):
    x, v = uniform_box(n, L, 31 + n)
    s = mdpd_system(engine, x, v, L, rho_est=max(6.0, n / L**3), extra=f"""
        timestep 0.001
        fix g all rdf/fast/meso output {tmp_path}/rdf.out nbin 20 every 3""")
    s.run(3)
    xr = s.gather("x")
    g = s.fix_result("g")[1]
    d = xr[:, None, :] - xr[None, :, :]
    d -= L * np.round(d / L)
    r = np.sqrt((d * d).sum(-1))[~np.eye(n, dtype=bool)]
    unit = 1.0 / n / (4.0 / 3.0 * 3.1415 * ((np.arange(1, 21) * 0.05) ** 3 - (np.arange(20) * 0.05) ** 3)) / (n / L**3)
    # a distance within 1e-5 of a bin's edge may fall on either side of it
    lo = np.array([((r >= b * 0.05 + 1e-5) & (r < (b + 1) * 0.05 - 1e-5)).sum() for b in range(20)])
    hi = np.array([((r >= b * 0.05 - 1e-5) & (r < (b + 1) * 0.05 + 1e-5)).sum() for b in range(20)])
    assert np.all(g >= (lo - 1e-6) * unit) and np.all(g <= (hi + 1e-6) * unit)
    s.close()


# systems admitted together are unpacked sixteen to a launch, as wide as the
# largest of them
@pytest.mark.parametrize("count", [1, 16, 17])
def test_jobs_admitted_together_equal_their_own_runs(engine, count):
    sizes = [(40 + 61 * k % 700, 4.0 + k % 3) for k in range(count)]
    p = engine.Pool(float(1 << 29), 32)
    p.tune("split", 2)
    made = [_box(engine, n, L) for n, L in sizes]
    jobs = [p.submit(s, 4) for s in made]
    p.run()
    for s, j in zip(made, jobs):
        s.tune("split", 2)
        s.run(4)
        for k in ("x", "v", "tag", "image"):
            np.testing.assert_array_equal(p.gather(j, k), s.gather(k), err_msg=f"job {j}: {k}")
        s.close()
    p.close()


# one wave per tile (rows past their end, a full staging area, tails of every
# length) against two: the same terms in another order.  A density is a sum of
# at most ~170 positive weights (relative error of either order below
# 170 2^-24 = 1e-5); forces within the bound that both keep to the oracle
@pytest.mark.parametrize("case", [c for c in CASES if c != "walls"])
def test_one_wave_per_tile_sums_the_same_terms(engine, case):
    got = []
    for split in (1, 2):
        s = CASES[case](engine)
        s.tune("split", split)
        s.setup()
        got.append((s.gather("rho"), s.gather("f")))
        s.close()
    (ra, fa), (rb, fb) = got
    np.testing.assert_allclose(ra, rb, rtol=2e-5)
    rms = np.sqrt((fb**2).sum(-1).mean())
    size = np.maximum(np.sqrt((fb**2).sum(-1)), rms)
    assert np.all(np.sqrt(((fa - fb) ** 2).sum(-1)) <= 2e-5 * size + 1e-30)


# a wall fraction below zero (rho_wall < 0) scales a mobile particle's pairs
# with wall particles as any other does: a pool's launches (more tiles than the
# wide kernels take) deal the ends of long rows to other lanes
@pytest.mark.parametrize("split", [2, 4])
def test_negative_wall_fractions_scale_every_pair(engine, split):
    x, v, types, nf = channel()
    s = engine.System()
    s.command("atom_style mdpd/atomic/meso 8.0")
    s.create_box(2, (0, 0, 0), (LX, LY, LZ))
    s.create_atoms(types, x, v)
    s.commands(DECK.replace("rho_wall 8.0", "rho_wall -8.0"))
    p = engine.Pool(float(1 << 29), 16)
    p.tune("split", split)
    j = p.submit(s, 6)
    p.run()
    assert p.stat("capacity") > 512 * 64
    s.tune("split", split)
    s.run(6)
    assert s.gather("phi")[:nf].min() < 0
    for k in ("x", "v", "f", "rho"):
        np.testing.assert_array_equal(p.gather(j, k), s.gather(k), err_msg=f"split {split}: {k}")
    p.close()
    s.close()


# energies and virials of the last pass are evaluated by one launch over all
# jobs that end together: sixty of them are more tiles than the wide kernels
# take, a job's own handle is not
@pytest.mark.parametrize("split", [2, 4])
@pytest.mark.parametrize("case", ["liquid", "two types", "uneven", "walls", "dpd"])
def test_results_of_many_jobs_ending_together_equal_their_own_runs(engine, case, split):
    s = CASES[case](engine)
    count = -(-513 * 64 // ((s.natoms + 255) // 256 * 256))
    p = engine.Pool(float(1 << 29), count)
    p.tune("split", split)
    jobs = [p.submit(s, 5) for _ in range(count)]
    p.run()
    s.tune("split", split)
    s.run(5)
    for k in ("f", "e_pair", "virial"):
        want = s.gather(k)
        for j in jobs:
            np.testing.assert_array_equal(p.gather(j, k), want, err_msg=f"{case}, split {split}, job {j}: {k}")
    p.close()
    s.close()
