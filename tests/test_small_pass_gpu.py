"""The small batch's particle pass (one slot per lane, movers moved in the
pass) against the oracle: counts around its sub-chunks (64 slots), groups and
tiles, pools on both sides of its size limits, every model, outlets and none,
rows of at most 6 neighbours and wider ones, inactive particles that move, and
crowded divisions (more than 16 requests in a sub-chunk)."""
import numpy as np
import pytest

from mcst import cases
from parity import assert_parity, make_pair


@pytest.mark.gpu
@pytest.mark.parametrize("model", ["monod_mass", "dual_monod", "monod", "fixed_length", "simple_acetate", "quad_monod"])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 257, 1024, 1025, 5003])
def test_counts_and_models(model, n):
    c = cases.small_case(model, n_c=[12, 1, 700][n % 3], n_particles=n, feeds=n % 2 == 1)
    eng, g, o = make_pair(c, probes=0)
    for steps in (1, 4):
        eng.step(steps)
        o.step(steps)
        assert_parity(g, o, probes=False)
    eng.close()


@pytest.mark.gpu
@pytest.mark.parametrize("model,cap", [("dual_monod", 1024 * 1024), ("dual_monod", 1024 * 1024 + 1), ("quad_monod", 1024 * 1024),
                                       ("monod", 3072 * 1024), ("monod", 3072 * 1024 + 1)])
def test_pools_around_the_limit(model, cap):
    c = cases.small_case(model, n_c=40, n_particles=30_000)
    eng, g, o = make_pair(c, probes=0, capacity=cap)
    eng.step(5)
    o.step(5)
    assert_parity(g, o, probes=False)
    eng.close()


@pytest.mark.gpu
@pytest.mark.parametrize("cap_extra,division_cap", [(0, None), (150, None), (5000, 37), (5000, None)])
@pytest.mark.parametrize("degree", [3, 9])
def test_crowded_divisions_and_inactive_movers(cap_extra, division_cap, degree):
    import mcst
    from oracle.oracle import OracleRun

    n, n_c = 4000, 30
    rng = np.random.default_rng(degree)
    e = np.array([(i, (i + d) % n_c) for i in range(n_c) for d in range(1, degree + 1)])
    q = rng.uniform(1e-3, 1e-2, len(e))
    eng = mcst.Engine("monod_mass")
    g = eng.add_run(n_c, 0.01, 5)
    o = OracleRun("monod_mass", n_c, 1, 0.01, 5)
    status = np.where(rng.random(n) < 0.2, rng.integers(2, 4, n), 0)
    pos = np.sort(rng.integers(0, n_c, n))
    m = rng.uniform(1e-15, 3e-15, n)  # most have twice their birth mass: they divide at once
    for x in (g, o):
        x.add_flowmap(np.full(n_c, 1e-3), e[:, 0], e[:, 1], q)
        x.add_feed("constant", 2e-3, 0.0, 0, n_c // 2, [0], [10.0])
        x.set_concentrations(np.full((1, n_c), 5.0))
        x.set_compaction(0.5, 0)  # the inactive stay for some steps
        if division_cap:
            x.set_division_cap(division_cap)
        x.set_particles(n + cap_extra, pos, status, np.stack([m, np.full(n, 1e-15)]), np.zeros(n), np.zeros(n), 1e9)
    eng.commit()
    for _ in range(4):
        eng.step(1)
        o.step(1)
        assert_parity(g, o, probes=False)
    assert g.counters()["births"] > 0 or cap_extra == 0
    eng.close()
