"""Axis lengths n = A B with A, B <= 16 (transformed as two steps in registers):
every A and B, both sides of the largest such length, next to lengths that the
LDS stages keep, on each axis, with full and partial groups of lines."""
import numpy as np
import pytest

from helpers import rel_l2

pytestmark = pytest.mark.gpu

TWO_STEP = (4, 6, 9, 12, 25, 26, 28, 32, 44, 45, 49, 63, 75, 96, 121, 126, 143, 165, 169, 182,
            195, 208, 224, 225, 240, 256)
STAGES = (2, 13, 200, 243, 250, 260)
# a chain of rounding errors over at most 8 additions in each of 2 steps, and
# the reference's own: below 40 eps of the largest value
TOL = 1e-14


@pytest.fixture(scope="module")
def ohp():
    import ohhelppic3d_amd
    return ohhelppic3d_amd


def halfcomplex(a, axis):
    """R2HC along `axis` from numpy's transform."""
    n = a.shape[axis]
    f = np.moveaxis(np.fft.fft(a, axis=axis), axis, 0)
    out = [f[k].real if 2 * k <= n else f[n - k].imag for k in range(n)]
    return np.moveaxis(np.array(out), 0, axis)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("length", TWO_STEP + STAGES)
def test_r2hc_and_back(ohp, axis, length):
    # lines: an odd number of them, and an even one with 16-byte pairs
    for others in ((3, 11), (36, 2)):
        n = list(others)
        n.insert(axis, length)
        a = np.random.default_rng(length).standard_normal(n[::-1])  # [z][y][x]
        ref = a
        for ax in (2, 1, 0):
            ref = halfcomplex(ref, ax)
        got = ohp.fft3d_r2r(a.ravel(), tuple(n))
        assert np.max(np.abs(got - ref.ravel())) <= TOL * np.max(np.abs(ref))
        back = ohp.fft3d_r2r(got, tuple(n), backward=True)
        assert np.max(np.abs(back - a.ravel())) <= TOL * np.max(np.abs(ref)) / np.sqrt(a.size)


def poisson(ohp, n, rho):
    cfg = ohp.SimConfig(n=n, qm=[-1.0], q_macro=[-1.0], capacity=[0])
    sim = ohp.Simulation(cfg)
    sim.put_grid(ohp.FIELD_RHO, rho)
    return sim


@pytest.mark.parametrize("length", TWO_STEP + STAGES)
def test_poisson_z(ohp, orc, length):
    for nx, ny in ((5, 3), (6, 4)):
        n = (nx, ny, length)
        rho = np.random.default_rng(length).standard_normal(nx * ny * length)
        with poisson(ohp, n, rho) as sim:
            sim.field_solve()
            assert rel_l2(sim.grid(ohp.FIELD_PHI), orc.poisson(n, rho)) <= 1e-12


def test_members_of_every_form_equal_alone(ohp):
    # one launch per form over all members: 16 x 16, other A x B, LDS stages
    shapes = ((4, 32, 256), (13, 6, 45), (256, 5, 7), (12, 256, 4), (2, 63, 200), (8, 8, 8))

    def make(n, seed):
        rng = np.random.default_rng(seed)
        m = 500
        cfg = ohp.SimConfig(n=n, qm=[-1.0], q_macro=[-0.01], capacity=[m], dt=0.1)
        sim = ohp.Simulation(cfg)
        pos = [rng.uniform(0, k, m) for k in n]
        sim.load_particles(0, *pos, *rng.normal(0, 0.1, (3, m)))
        return sim

    alone = []
    for i, n in enumerate(shapes):
        with make(n, i) as sim:
            sim.step(3)
            alone.append([sim.grid(w) for w in (ohp.FIELD_RHO, ohp.FIELD_PHI, ohp.FIELD_EX)])
    sims = [make(n, i) for i, n in enumerate(shapes)]
    try:
        with ohp.Group() as grp:
            for s in sims:
                grp.attach(s)
            grp.step(3)
            for s, ref in zip(sims, alone):
                for w, r in zip((ohp.FIELD_RHO, ohp.FIELD_PHI, ohp.FIELD_EX), ref):
                    assert np.array_equal(s.grid(w), r)
    finally:
        for s in sims:
            s.close()


# x and y lengths whose passes go by planes (up to 512 of them, up to four
# wavefronts of lines, up to 64 KiB of LDS) and their nearest neighbours
PLANES = ((4, 4, 1), (4, 4, 512), (4, 4, 520), (6, 45, 5), (45, 6, 5), (39, 26, 3), (55, 50, 3),
          (64, 48, 4), (64, 64, 2), (32, 32, 32))


@pytest.mark.parametrize("n", PLANES)
def test_planes_equal_axis_passes(ohp, orc, n):
    rho = np.random.default_rng(n[2]).standard_normal(n[0] * n[1] * n[2])
    with poisson(ohp, n, rho) as sim:
        sim.field_solve()
        assert rel_l2(sim.grid(ohp.FIELD_PHI), orc.poisson(n, rho)) <= 1e-12

    def make():
        rng = np.random.default_rng(n[0])
        cfg = ohp.SimConfig(n=n, qm=[-1.0, 1.0], q_macro=[-0.01, 0.01], capacity=[700, 300], dt=0.1)
        sim = ohp.Simulation(cfg)
        for s, m in enumerate((700, 300)):
            sim.load_particles(s, *[rng.uniform(0, k, m) for k in n], *rng.normal(0, 0.3, (3, m)))
        return sim

    # alone, and beside a member with a 2-point axis, for which no launch of the
    # group goes by planes: the same bit for bit
    with make() as a, make() as b, poisson(ohp, (2, 2, 2), np.zeros(8)) as other:
        a.step(3)
        with ohp.Group() as grp:
            grp.attach(b)
            grp.attach(other)
            grp.step(3)
            for w in (ohp.FIELD_RHO, ohp.FIELD_PHI, ohp.FIELD_EX, ohp.FIELD_EY, ohp.FIELD_EZ):
                assert np.array_equal(a.grid(w), b.grid(w))
