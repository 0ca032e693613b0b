"""The energy sums of a step and of a separate solve: work-item and row counts
below, at and beyond one and eight entries per thread of the reducing block."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# tiles of 4^3: 1, 63, 1024, 1025 + a few, and more than 8192 items
SIZES = ((4, 4, 4), (12, 12, 28), (32, 64, 32), (36, 60, 32), (84, 80, 84))


@pytest.fixture(scope="module")
def ohp():
    import ohhelppic3d_amd
    return ohhelppic3d_amd


@pytest.mark.parametrize("n", SIZES)
def test_sums_match_the_state(ohp, n):
    rng = np.random.default_rng(n[0])
    m = 2 * n[0] * n[1] * n[2]
    cfg = ohp.SimConfig(n=n, qm=[-1.0, 0.5], q_macro=[-0.01, 0.02], capacity=[m, m], dt=0.05,
                        tile=(4, 4, 4))
    with ohp.Simulation(cfg) as sim:
        for s in range(2):
            sim.load_particles(s, *[rng.uniform(0, k, m) for k in n], *rng.normal(0, 0.2, (3, m)))
        sim.step(1)
        d = sim.diagnostics()
        rho, phi = sim.grid(ohp.FIELD_RHO), sim.grid(ohp.FIELD_PHI)
        for s in range(2):
            p = sim.store_particles(s)
            mass = cfg.q_macro[s] / cfg.qm[s]
            ke = 0.5 * mass * float((p["vx"] ** 2 + p["vy"] ** 2 + p["vz"] ** 2).sum())
            assert abs(d["ke_new"][s] - ke) <= 1e-12 * abs(ke)
        # both sides round sums of these terms: 1e-12 of their absolute sum
        terms = 0.5 * rho * phi
        assert abs(d["field_energy"] - terms.sum()) <= 1e-12 * np.abs(terms).sum()
        assert abs(d["net_charge"] - rho.sum()) <= 1e-12 * np.abs(rho).sum()
        sim.field_solve()
        d = sim.diagnostics()
        phi = sim.grid(ohp.FIELD_PHI)
        terms = 0.5 * sim.grid(ohp.FIELD_RHO) * phi
        assert abs(d["field_energy"] - terms.sum()) <= 1e-12 * np.abs(terms).sum()
