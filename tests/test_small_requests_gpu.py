"""Division requests of small pools past 4096 sub-chunks of 64 slots (the
ranks are summed over many blocks of them): everyone asks, some or none are
accepted, in slot order, in single runs and batches, against the oracle."""
import numpy as np
import pytest

from mcst import cases
from parity import assert_parity


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [[262_145], [300_001], [700_000], [150_000, 64, 120_000, 90_001]])
@pytest.mark.parametrize("room,division_cap", [(0, None), (70_000, None), (200_000, 100_003)])
def test_crowded_requests_are_accepted_in_slot_order(sizes, room, division_cap):
    import mcst
    from oracle.oracle import OracleRun

    eng = mcst.Engine("monod_mass")
    pairs = []
    for k, n in enumerate(sizes):
        c = cases.small_case("monod_mass", n_c=30, n_particles=n, seed=3 + k)
        c.params = np.array([0.5, 0.01, 0.5, 0.0, 1e-15, 0.1])  # every cell divides in every step
        c.capacity = n + room // len(sizes)
        g = eng.add_run(c.n_c, c.dt, c.seed)
        o = OracleRun(c.model, c.n_c, c.n_s, c.dt, c.seed)
        for x in (g, o):
            c.apply(x)
            x.set_compaction(0.01, 0)
            if division_cap:
                x.set_division_cap(division_cap)
        pairs.append((g, o))
    eng.commit()
    for steps in (1, 2):
        eng.step(steps)
        for g, o in pairs:
            o.step(steps, threads=8)
            assert_parity(g, o, probes=False)
    eng.close()
