"""Split tiles at their limits: bins that overflow, more items than a tile has
blocks, and wavefronts most of whose particles leave.  The charge grid is
integer, so fields and particles equal those of whole tiles bit for bit."""
import numpy as np
import pytest

from helpers import by_pid, sim_for

pytestmark = pytest.mark.gpu

N = (24, 16, 16)
PREC = ["fp64", "mixed"]


@pytest.fixture(scope="module")
def ohp():
    import ohhelppic3d_amd
    return ohhelppic3d_amd


def free(count, seed, speed=0.0, wave=0.0):
    """Two species of free particles; `wave`: flow towards the middle of x."""
    rng = np.random.default_rng(seed)
    sp = []
    for qm, q, m in ((-1e-12, -1e-4, count), (1e-12, 1e-4, count // 3)):
        x, y, z = (rng.uniform(0, k, m) for k in N)
        sp.append(dict(qm=qm, q=q, x=x, y=y, z=z,
                       vx=rng.normal(0, speed, m) + wave * np.sin(2 * np.pi * x / N[0]),
                       vy=rng.normal(0, speed, m), vz=rng.normal(0, speed, m)))
    return sp


def make(ohp, sp, precision, **kw):
    return sim_for(sp, N, precision=ohp.FP64 if precision == "fp64" else ohp.MIXED,
                   weight_order=1, **kw)


def same(ohp, a, b):
    for w in (ohp.FIELD_RHO, ohp.FIELD_PHI, ohp.FIELD_EX):
        assert np.array_equal(a.grid(w), b.grid(w))
    for s in range(2):
        p, q = (by_pid(m.store_particles(s, True)) for m in (a, b))
        assert all(np.array_equal(p[k], q[k]) for k in q), s
    assert np.array_equal(a.cell_counts(), b.cell_counts())


@pytest.mark.parametrize("precision", PREC)
@pytest.mark.parametrize("chunks", [1, 3, 40])
@pytest.mark.parametrize("grouped", [False, True])
def test_overflow(ohp, precision, chunks, grouped):
    # the flow doubles the middle tiles' counts within a few steps
    sp = free(60000, 5, speed=0.5, wave=12.0)
    steps = 11  # in a group: a sequence of eight, then single steps
    with make(ohp, sp, precision, tile=(4, 4, 4), chunks=chunks, slack=0.01) as a, \
            make(ohp, sp, precision, tile=(4, 4, 4), chunks=1, slack=12.0) as b:
        b.step(steps)
        assert b.diagnostics()["repacks"] == 0
        if grouped:
            with ohp.Group() as grp:
                grp.attach(a)
                grp.step(steps)
        else:
            a.step(steps)
        assert a.diagnostics()["repacks"] > 0
        same(ohp, a, b)


@pytest.mark.parametrize("precision", PREC)
@pytest.mark.parametrize("chunks", [65, 300])
def test_more_items_than_blocks(ohp, precision, chunks):
    sp = free(100003, 6, speed=2.0)
    with make(ohp, sp, precision, tile=(8, 8, 8), chunks=chunks, slack=1.0) as a, \
            make(ohp, sp, precision, tile=(8, 8, 8), chunks=1, slack=1.0) as b:
        a.step(3)
        b.step(3)
        assert a.diagnostics()["repacks"] == 0
        same(ohp, a, b)


@pytest.mark.parametrize("precision", PREC)
@pytest.mark.parametrize("tile", [(4, 4, 4), (8, 8, 8), (16, 8, 4)])
@pytest.mark.parametrize("chunks", [1, 3])
def test_most_particles_leave(ohp, precision, tile, chunks):
    # 3 cells per step and axis: more than half of a wavefront at once
    sp = free(40009, 7, speed=30.0)
    with make(ohp, sp, precision, tile=tile, chunks=chunks, slack=2.0) as a, \
            make(ohp, sp, precision, tile=(8, 8, 4), chunks=1, slack=8.0) as b:
        a.step(3)
        b.step(3)
        assert a.diagnostics()["repacks"] == 0
        same(ohp, a, b)


@pytest.mark.parametrize("precision", PREC)
@pytest.mark.parametrize("chunks", [1, 3])
def test_boundary_operator_overflow(ohp, precision, chunks):
    sp = free(60000, 8, speed=0.5, wave=12.0)
    with make(ohp, sp, precision, tile=(4, 4, 4), chunks=chunks, slack=0.01) as a, \
            make(ohp, sp, precision, tile=(4, 4, 4), chunks=1, slack=12.0) as b:
        for _ in range(6):
            a.deposit()
            a.field_solve()
            a.gather_push()
            a.boundary()
        assert a.diagnostics()["repacks"] > 0
        b.step(6)
        for s in range(2):
            p, q = (by_pid(m.store_particles(s, True)) for m in (a, b))
            assert all(np.array_equal(p[k], q[k]) for k in q), s
        assert np.array_equal(a.cell_counts(), b.cell_counts())
