"""The small pool's pass with its groups dealt to the blocks one at a time or in
one range each, by default, forced (any other length of turn means a range) and
tuned, in single runs and batches, against the oracle."""
import re

import pytest

from mcst import cases
from parity import assert_parity

SIZES = [(12, 1), (40, 30_000), (7, 1025), (30, 9000), (300, 64)]


def make(runs, capacity=None):
    import mcst
    from oracle.oracle import OracleRun

    eng = mcst.Engine("dual_monod")
    pairs = []
    for k, (n_c, n) in enumerate(runs):
        c = cases.small_case("dual_monod", n_c=n_c, n_particles=n, seed=3 + k)
        c.capacity = capacity or 4 * n
        g = eng.add_run(c.n_c, c.dt, c.seed)
        o = OracleRun(c.model, c.n_c, c.n_s, c.dt, c.seed)
        for x in (g, o):
            c.apply(x)
            x.set_compaction(0.01, 0)
        pairs.append((g, o))
    eng.commit()
    return eng, pairs


@pytest.mark.gpu
@pytest.mark.parametrize("group", [None, "0", "1", "3", "1000000"])
@pytest.mark.parametrize("block", [None, "256", "512", "1024"])
@pytest.mark.parametrize("runs", [[(40, 30_000)], [(700, 600_000)], SIZES])
def test_turns_match_oracle(group, block, runs, monkeypatch, capfd):
    monkeypatch.setenv("MCST_VERBOSE", "1")
    if group:
        monkeypatch.setenv("MCST_TILE_GROUP", group)
    if block:
        monkeypatch.setenv("MCST_PARTICLE_BLOCK", block)
    eng, pairs = make(runs, 1_000_000 if len(runs) == 1 else None)
    want = ("1" if group == "1" else "0") if group else "1" if len(runs) == 1 else "0"
    assert re.findall(r"group=(\d+)", capfd.readouterr().err)[-1] == want
    eng.step(3)
    for g, o in pairs:
        o.step(3, threads=8)
        assert_parity(g, o, probes=False)
    eng.close()


@pytest.mark.gpu
def test_a_small_batch_is_tuned():
    eng, pairs = make(SIZES)
    choice = eng.autotune(2)
    assert choice["block"] in (256, 512, 1024) and choice["group"] in (0, 1)
    done = pairs[0][0].counters()["steps"]
    eng.step(2)
    for g, o in pairs:
        o.step(done + 2)
        cg, co = g.counters(), o.counters()
        assert cg == co
    eng.close()
