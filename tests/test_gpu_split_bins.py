"""The particle kernels' output of a bin: 64-slot blocks filled from a stash,
the run of what is left, and the joining of split tiles (k_close_chunks).

Particle counts lie on the edges of a wavefront (64), a workgroup (256, 512)
and a chunk; speeds make none, some or most particles leave their tile.  The
charge grid is integer, so fields and particles are the same bit for bit
however a tile is split and whether identities are kept.
"""
import numpy as np
import pytest

from helpers import by_pid, rel_l2, sim_for

pytestmark = pytest.mark.gpu

N = (24, 16, 8)
COUNTS = (1, 63, 64, 65, 257, 513, 4099, 20011)
TOL = 1e-12


@pytest.fixture(scope="module")
def ohp():
    import ohhelppic3d_amd
    return ohhelppic3d_amd


def plasma(count, speed, seed):
    rng = np.random.default_rng(seed)
    sp = []
    for qm, q, m in ((-1e-3, -1e-4, count), (1e-3, 1e-4, max(1, count // 3))):
        # most of them in the tile at the origin, so that its bin is the one split
        x = np.concatenate([rng.uniform(0, 8, m - m // 4), rng.uniform(0, N[0], m // 4)])
        y = np.concatenate([rng.uniform(0, 8, m - m // 4), rng.uniform(0, N[1], m // 4)])
        sp.append(dict(qm=qm, q=q, x=x, y=y, z=rng.uniform(0, N[2], m),
                       vx=rng.normal(0, speed, m), vy=rng.normal(0, speed, m),
                       vz=rng.normal(0, speed, m)))
    return sp


def run(sim, ohp, ids):
    sim.step(3)
    fields = [sim.grid(w) for w in (ohp.FIELD_RHO, ohp.FIELD_PHI, ohp.FIELD_EX)]
    parts = [by_pid(sim.store_particles(s, True)) if ids else
             {k: np.sort(v) for k, v in sim.store_particles(s).items()} for s in range(2)]
    return fields, parts, sim.cell_counts(), sim.diagnostics()


def same(a, b):
    assert all(np.array_equal(x, y) for x, y in zip(a[0], b[0]))
    for s in range(2):
        for k in b[1][s]:
            assert np.array_equal(a[1][s][k], b[1][s][k]), (s, k)
    assert np.array_equal(a[2], b[2])


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("speed", [0.0, 2.0, 6.0])
@pytest.mark.parametrize("count", COUNTS)
def test_split_tiles_equal_whole_tiles(ohp, orc, precision, speed, count):
    prec = ohp.FP64 if precision == "fp64" else ohp.MIXED
    sp = plasma(count, speed, count)
    got = {}
    for chunks in (1, 2, 3, 7):
        for tile in ((8, 8, 8), (4, 4, 4)):
            with sim_for(sp, N, precision=prec, tile=tile, chunks=chunks, slack=8.0,
                         weight_order=1) as sim:
                got[chunks, tile] = run(sim, ohp, True)
                assert got[chunks, tile][3]["repacks"] == 0
    first = got[1, (8, 8, 8)]
    for g in got.values():
        same(g, first)
    # without identities: the same particles as a multiset
    cfg = ohp.SimConfig(n=N, qm=[d["qm"] for d in sp], q_macro=[d["q"] for d in sp],
                        capacity=[len(d["x"]) for d in sp], dt=0.1, b0=(0.0, 0.0, 0.5),
                        precision=prec, weight_order=1, tile=(8, 8, 8), slack=8.0, chunks=3)
    with ohp.Simulation(cfg) as sim:
        for s, d in enumerate(sp):
            sim.load_particles(s, d["x"], d["y"], d["z"], d["vx"], d["vy"], d["vz"])
        plain = run(sim, ohp, False)
    for s in range(2):
        for k in plain[1][s]:
            assert np.array_equal(plain[1][s][k], np.sort(first[1][s][k]))
    assert np.array_equal(plain[0][0], first[0][0]) and np.array_equal(plain[2], first[2])
    if precision == "fp64":
        osim = orc.OracleSim(N, sp, 0.1, (0.0, 0.0, 0.5), 1)
        osim.step(3)
        for s in range(2):
            for k in ("x", "y", "z", "vx", "vy", "vz"):
                # a position that wraps carries the box length's rounding
                assert np.max(np.abs(first[1][s][k] - osim.sp[s][k])) <= TOL * max(N), (s, k)
        assert rel_l2(first[0][0], osim.rho) <= 1e-11


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_split_boundary_operator_equals_step(ohp, precision):
    prec = ohp.FP64 if precision == "fp64" else ohp.MIXED
    sp = plasma(5000, 4.0, 3)
    with sim_for(sp, N, precision=prec, tile=(8, 8, 8), chunks=5, slack=8.0) as a, \
            sim_for(sp, N, precision=prec, tile=(8, 8, 8), chunks=1, slack=8.0) as b:
        for _ in range(3):
            a.deposit()
            a.field_solve()
            a.gather_push()
            a.boundary()
        b.step(3)
        for s in range(2):
            pa, pb = (by_pid(m.store_particles(s, True)) for m in (a, b))
            for k in pb:
                assert np.array_equal(pa[k], pb[k]), (s, k)
        assert np.array_equal(a.cell_counts(), b.cell_counts())


def test_automatic_split_of_a_density_peak(ohp):
    # one tile holds most of the particles: the plan splits it, and the result
    # is that of whole tiles
    rng = np.random.default_rng(11)
    n = (32, 32, 32)
    m = 400000
    x = np.concatenate([rng.uniform(8, 16, (3, 3 * m // 4)), rng.uniform(0, 32, (3, m // 4))], 1)
    v = rng.normal(0, 1.0, (3, m))
    sp = [dict(qm=-1e-3, q=-1e-4, x=x[0], y=x[1], z=x[2], vx=v[0], vy=v[1], vz=v[2])]
    out = []
    for chunks in (0, 1):
        with sim_for(sp, n, precision=ohp.MIXED, tile=(8, 8, 8), chunks=chunks, slack=0.5,
                     weight_order=1) as sim:
            sim.step(2)
            out.append((sim.grid(ohp.FIELD_RHO), by_pid(sim.store_particles(0, True)),
                        sim.cell_counts()))
            with ohp.Group() as grp:
                grp.attach(sim)
                grp.step(9)
                assert grp.stats()["items"] > (64 if chunks == 0 else 63)
            out[-1] += (sim.grid(ohp.FIELD_RHO), by_pid(sim.store_particles(0, True)))
    for a, b in zip(*out):
        if isinstance(a, dict):
            assert all(np.array_equal(a[k], b[k]) for k in a)
        else:
            assert np.array_equal(a, b)
