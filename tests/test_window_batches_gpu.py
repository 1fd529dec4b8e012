"""Batches with a compartment window: blocks that take turns of one group, of
several, or one range of groups, over runs of one and of several windows (and
one that fits whole), in and out of compartment order, against the oracle."""
import numpy as np
import pytest

from mcst import cases
from parity import assert_parity


@pytest.mark.gpu
@pytest.mark.parametrize("group", [None, "0", "1", "3", "4"])
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("sizes", [[(5089, 30_000), (40, 700), (12_000, 60_000)],
                                   [(5300, 9000), (5200, 3000), (6000, 5), (5500, 20_000), (5089, 2049)]])
def test_windowed_batches_match_oracle(group, mixed, sizes, monkeypatch):
    import mcst
    from oracle.oracle import OracleRun

    if group:
        monkeypatch.setenv("MCST_TILE_GROUP", group)
    eng = mcst.Engine("quad_monod")
    pairs = []
    for k, (n_c, n) in enumerate(sizes):
        c = cases.small_case("quad_monod", n_c=n_c, n_particles=n, n_maps=1, seed=11 + k)
        g = eng.add_run(c.n_c, c.dt, c.seed)
        o = OracleRun(c.model, c.n_c, c.n_s, c.dt, c.seed)
        for x in (g, o):
            c.apply(x)
            x.set_compaction(0.01, 0)
        if mixed:  # the oracle's initial particles at random places, for both
            p = o.particles()
            pos = np.random.default_rng(k).integers(0, n_c, n)
            for x in (g, o):
                x.set_particles(2 * n, pos, p["status"], p["state"], p["age_hyd"], p["age_div"], o.weight)
        pairs.append((g, o))
    eng.commit()
    eng.step(3)
    for g, o in pairs:
        o.step(3)
        assert_parity(g, o, probes=False)
    eng.close()


@pytest.mark.gpu
def test_a_range_per_block_where_runs_are_as_many_as_turns(monkeypatch, capfd):
    import re

    import mcst

    monkeypatch.setenv("MCST_VERBOSE", "1")
    for runs, capacity, group in ((1, 3_000_000, "1"), (2, 3_000_000, "1"), (9, 300_000, "0")):
        eng = mcst.Engine("quad_monod")
        for k in range(runs):
            c = cases.small_case("quad_monod", n_c=5100, n_particles=500, n_maps=1, seed=k)
            c.capacity = capacity
            c.apply(eng.add_run(c.n_c, c.dt, c.seed))
        eng.commit()
        err = capfd.readouterr().err
        assert re.findall(r"block=(\d+).* group=(\d+)", err)[-1] == ("1024", group)
        eng.close()
