"""When a re-binning step overflows a bin: stayers and arrivals together have to
exceed its slots, whatever leaves it in the same step.

Plasmas of free particles (charge-to-mass 1e-12) at the default slack, so fast
that a tile's old count and its arrivals together do not fit, while what stays
and arrives does: tiles whole, split by the plan or by the given chunks, alone
and in a group."""
import numpy as np
import pytest

from helpers import by_pid

pytestmark = pytest.mark.gpu

PREC = ["fp64", "mixed"]


@pytest.fixture(scope="module")
def ohp():
    import ohhelppic3d_amd
    return ohhelppic3d_amd


def plasma(ohp, n, ppc, speed, precision, hump=False, **kw):
    m = ppc * n[0] * n[1] * n[2]
    cfg = ohp.SimConfig(n=n, qm=[-1e-12, 1e-12], q_macro=[-1.0 / ppc, 1.0 / ppc], capacity=[m, m],
                        dt=0.1, precision=ohp.FP64 if precision == "fp64" else ohp.MIXED,
                        weight_order=1, track_ids=True, **kw)
    sim = ohp.Simulation(cfg)
    if hump:
        sim.seed_hump_maxwell([m, m], (speed, speed), 9.0, min(n) / 16.0, budget=2052)
    else:
        sim.seed_uniform_maxwell([m, m], (speed, speed))
    return sim


def same(ohp, a, b):
    assert np.array_equal(a.grid(ohp.FIELD_RHO), b.grid(ohp.FIELD_RHO))
    assert np.array_equal(a.cell_counts(), b.cell_counts())
    for s in range(2):
        p, q = (by_pid(m.store_particles(s, True)) for m in (a, b))
        assert all(np.array_equal(p[k], q[k]) for k in q), s


# (grid, ppc, cells per step, density peak)
LOADS = [((32, 32, 32), 16, 0.3, False), ((32, 32, 32), 64, 0.5, False),
         ((64, 64, 64), 32, 0.3, True)]


@pytest.mark.parametrize("precision", PREC)
@pytest.mark.parametrize("chunks", [0, 3])
@pytest.mark.parametrize("n,ppc,vdt,hump", LOADS)
def test_fast_plasma_overflows_no_bin(ohp, precision, chunks, n, ppc, vdt, hump):
    with plasma(ohp, n, ppc, vdt / 0.1, precision, hump, chunks=chunks) as a, \
            plasma(ohp, n, ppc, vdt / 0.1, precision, hump, chunks=1, slack=4.0) as b:
        a.step(12)
        assert a.diagnostics()["repacks"] == 0
        b.step(12)
        same(ohp, a, b)


@pytest.mark.parametrize("precision", PREC)
@pytest.mark.parametrize("chunks", [0, 3])
def test_fast_plasma_in_a_group(ohp, precision, chunks):
    n = (32, 32, 32)
    with plasma(ohp, n, 16, 3.0, precision, chunks=chunks) as a, \
            plasma(ohp, n, 16, 3.0, precision, chunks=1, slack=4.0) as b, \
            plasma(ohp, (16, 24, 32), 16, 4.0, precision, chunks=chunks) as c, \
            ohp.Group() as grp:
        grp.attach(a)
        grp.attach(c)
        grp.step(11)
        assert a.diagnostics()["repacks"] == 0 and c.diagnostics()["repacks"] == 0
        b.step(11)
        same(ohp, a, b)


@pytest.mark.parametrize("precision", PREC)
@pytest.mark.parametrize("chunks", [1, 4])
def test_boundary_operator(ohp, precision, chunks):
    n = (32, 32, 32)
    with plasma(ohp, n, 32, 4.0, precision, chunks=chunks) as a, \
            plasma(ohp, n, 32, 4.0, precision, chunks=1, slack=4.0) as b:
        for _ in range(4):
            a.deposit()
            a.field_solve()
            a.gather_push()
            a.boundary()
        assert a.diagnostics()["repacks"] == 0
        b.step(4)
        b.deposit()
        a.deposit()
        for s in range(2):
            p, q = (by_pid(m.store_particles(s, True)) for m in (a, b))
            assert all(np.array_equal(p[k], q[k]) for k in q), s
