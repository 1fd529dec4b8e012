"""The tiles of the next step are laid out by the block that keeps a step's
books, in another table than the one the step's own blocks read (a resolve
block without work may start after the books): populations that fill new tiles
with nearly every step, in calls of odd and even lengths and replayed graphs
of both, with a second engine's steps on the card at the same time, against the
oracle."""
import numpy as np
import pytest

from mcst import cases
from parity import assert_parity


def growing(eng, n, seed, cap):
    """A run whose cells all divide, `cap` of them a step."""
    from oracle.oracle import OracleRun

    c = cases.small_case("monod_mass", n_c=12, n_particles=n, seed=seed)
    c.params = np.array([0.5, 0.01, 0.5, 0.0, 1e-15, 0.1])
    c.capacity = n + 40 * cap
    g = eng.add_run(c.n_c, c.dt, c.seed)
    o = OracleRun(c.model, c.n_c, c.n_s, c.dt, c.seed)
    for x in (g, o):
        c.apply(x)
        x.set_division_cap(cap)
        x.set_compaction(0.01, 0)
    return g, o


@pytest.mark.gpu
@pytest.mark.parametrize("runs", [1, 3])
@pytest.mark.parametrize("graph", [1, 2, 3])
def test_growing_tile_counts_match_oracle(runs, graph):
    import mcst

    busy = mcst.Engine("dual_monod")
    c = cases.small_case("dual_monod", n_c=700, n_particles=400_000, seed=5)
    c.apply(busy.add_run(c.n_c, c.dt, c.seed))
    busy.commit()
    eng = mcst.Engine("monod_mass")
    pairs = [growing(eng, 900 + 500 * k, 3 + k, 1024 - 300 * k) for k in range(runs)]
    eng.commit()
    taken = 0
    for steps in (7, 1, 4, 3):
        busy.step(40)
        eng.step(steps)
        taken += steps
        for g, o in pairs:
            o.step(steps)
            assert_parity(g, o, probes=False)
    eng.capture(graph)
    for times in (1, 2, 1):
        busy.step(20)
        eng.replay(times)
        eng.synchronize()
        for g, o in pairs:
            o.step(graph * times)
            assert_parity(g, o, probes=False)
    for g, _ in pairs:
        assert g.n > 14 * 1024 // 3
    eng.close()
    busy.close()
