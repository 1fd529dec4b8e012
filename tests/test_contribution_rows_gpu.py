"""Contribution rows (MCST_CONTRIB_ROWS=1, one run): the blocks' accumulators
are summed in a fixed order, so where each lane of a block adds to compartments
of its own the contributions are the same bits in every engine; and every pass
shape agrees with the oracle with them."""
import numpy as np
import pytest

from mcst import cases
from parity import assert_parity, make_pair

N, N_C = 300_000, 256


@pytest.mark.gpu
@pytest.mark.parametrize("slots_per_lane,capacity", [(1, N), (4, 1100 * 1024)])  # the small pool's pass, and the general one
def test_sums_do_not_depend_on_the_order_of_blocks(slots_per_lane, capacity, monkeypatch):
    import mcst

    monkeypatch.setenv("MCST_CONTRIB_ROWS", "1")
    monkeypatch.setenv("MCST_PARTICLE_BLOCK", "256")
    slot = np.arange(N)
    pos = slot // (64 * slots_per_lane) % 4 * 64 + slot % 64  # wave and lane of the slot
    m = np.random.default_rng(1).uniform(1e-15, 2e-15, N)
    seen = []
    for _ in range(4):
        eng = mcst.Engine("monod_mass")
        g = eng.add_run(N_C, 0.01, 5)
        g.add_flowmap(np.full(N_C, 1e-3), [], [], [])
        g.set_concentrations(np.full((1, N_C), 5.0))
        g.set_particles(capacity, pos, np.zeros(N, np.uint8), np.stack([m, np.full(N, 1e-15)]), np.zeros(N),
                        np.zeros(N), 1e9)
        eng.commit()
        eng.step(1)
        first = g.contributions()
        eng.step(6)
        seen.append((first, g.contributions(), g.concentrations()))
        eng.close()
    assert (seen[0][0] < 0).all()
    for other in seen[1:]:
        for a, b in zip(seen[0], other):
            np.testing.assert_array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("model,n_c,n,capacity", [("monod_mass", 1, 700, None), ("dual_monod", 64, 5000, None),
                                                  ("dual_monod", 65, 5000, 1100 * 1024), ("quad_monod", 700, 30_000, None),
                                                  ("quad_monod", 3000, 30_000, 1100 * 1024),
                                                  ("simple_acetate", 129, 9000, 3100 * 1024)])
@pytest.mark.parametrize("probes", [0, 1 << 16])
def test_rows_match_oracle(model, n_c, n, capacity, probes, monkeypatch):
    monkeypatch.setenv("MCST_CONTRIB_ROWS", "1")
    c = cases.small_case(model, n_c=n_c, n_particles=n)
    eng, g, o = make_pair(c, probes=probes, capacity=capacity)
    for steps in (1, 2):
        eng.step(steps)
        o.step(steps)
        assert_parity(g, o, probes=probes > 0)
    eng.capture(2)
    eng.replay(1)
    eng.synchronize()
    o.step(2)
    assert_parity(g, o, probes=probes > 0)
    eng.close()
