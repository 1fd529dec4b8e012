"""Time-dependent feeds across the blocks of steps (256) whose flows the host
prepares at once: calls that end before, on and after a block's end, one step
at a time and many, a run that joins at another step count, and single stages,
against the oracle."""
import pytest

from mcst import cases
from parity import assert_parity


def with_feeds(n, seed):
    c = cases.small_case("dual_monod", n_c=12, n_particles=n, seed=seed)
    c.feeds = [("linear", 1e-3, 0.02, 3, 9, [0, 1], [8.0, 0.5]), ("constant", 2e-3, 0.0, 0, 6, [0], [10.0]),
               ("exponential", 0.0, -3.0, 10, None, [1], [1e-4])]
    c.params = None  # slow growth: hundreds of steps
    return c


@pytest.mark.gpu
@pytest.mark.parametrize("calls", [[1] * 3 + [252, 1, 1, 3], [254, 2, 255], [255, 1, 257], [600], [256, 256, 1]])
def test_calls_across_the_blocks(calls):
    import mcst
    from oracle.oracle import OracleRun

    eng = mcst.Engine("dual_monod")
    eng.reserve(40_000, 2)
    eng.commit()
    pairs = []

    def join(seed):
        c = with_feeds(1500, seed)
        g = eng.add_run(c.n_c, c.dt, c.seed)
        o = OracleRun(c.model, c.n_c, c.n_s, c.dt, c.seed)
        for x in (g, o):
            c.apply(x)
            x.set_compaction(0.01, 0)
        assert eng.admit() == 1
        pairs.append((g, o))

    join(1)
    for k, n in enumerate(calls):
        if k == 1:
            join(2)
        eng.step(n)
        for _, o in pairs:
            o.step(n)
    eng.step_stages(63)
    eng.profile(2)
    for g, o in pairs:
        o.step(3)
        assert_parity(g, o, probes=False)
    eng.close()
