"""Particles that leave their tile's one-cell halo in a step: their number, and
the cost of counting them when nearly every lane does."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TILE = 8
DT = 0.1


@pytest.fixture(scope="module")
def ohp():
    import ohhelppic3d_amd
    return ohhelppic3d_amd


def plasma(ohp, n, m, speed, precision):
    """Two species that move in straight lines (charge-to-mass 1e-12)."""
    cfg = ohp.SimConfig(n=n, qm=[-1e-12, 1e-12], q_macro=[-1e-3, 1e-3], capacity=[m, m], dt=DT,
                        track_ids=True, precision=precision, weight_order=1,
                        tile=(TILE, TILE, TILE), chunks=1)
    sim = ohp.Simulation(cfg)
    sim.seed_uniform_maxwell([m, m], (speed, speed))
    return sim


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("speed", [0.5, 6.0, 30.0])
def test_count(ohp, precision, speed):
    n, m = (24, 16, 32), 20001
    with plasma(ohp, n, m, speed, ohp.FP64 if precision == "fp64" else ohp.MIXED) as sim:
        want = 0
        for s in range(2):
            p = sim.store_particles(s, with_ids=True)
            fast = np.zeros(m, bool)
            for x, v, k in zip("xyz", ("vx", "vy", "vz"), n):
                origin = np.floor(p[x] / TILE) * TILE
                rel = np.floor(p[x] + p[v] * DT) - origin + 1
                # the mixed form looks at the move itself, the FP64 form at
                # the wrapped position
                fast |= (rel % k if precision == "fp64" else rel) > TILE + 1
                fast |= rel < (0 if precision == "mixed" else -np.inf)
            want += int(fast.sum())
        sim.step(1)
        got = sim.diagnostics()["fast_particles"]
        # a mixed position lies within 2^-24 of the exact one, so 120006
        # coordinates change cell with probability 2^-23 each
        assert abs(got - want) <= (0 if precision == "fp64" else 2)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_counting_does_not_dominate(ohp, precision):
    # a fast particle takes eight global atomics where a slow one takes LDS
    # ones: 25 to 55 times a slow step; one atomic of its own on the counter
    # per particle: several hundred times
    n, m = (64, 64, 64), 16 * 64 ** 3
    best = {}
    for speed in (1.0, 30.0):
        with plasma(ohp, n, m, speed, ohp.FP64 if precision == "fp64" else ohp.MIXED) as sim:
            times = []
            for _ in range(4):
                t = time.perf_counter()
                sim.step(1)
                times.append(time.perf_counter() - t)
            best[speed] = min(times)
    assert best[30.0] < 150 * best[1.0], best
