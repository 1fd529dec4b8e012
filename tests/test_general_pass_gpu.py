"""The particle pass of large pools (k_particle), without probes, in every launch
shape that can be tuned or forced, on populations small enough for the oracle:
the pools are past the size up to which the small pool's pass takes over, and
the shape that was chosen is looked at."""
import re

import pytest

from mcst import cases
from parity import assert_parity

PAST = 1025 * 1024       # slots: past the small pool's limit for models of few values per lane
PAST_WIDE = 3073 * 1024  # ... and of many


def engine(specs, capacity, **kw):
    """specs: (model, n_c, n); the first run takes the pool's slots."""
    import mcst
    from oracle.oracle import OracleRun

    eng = mcst.Engine(specs[0][0])
    pairs = []
    for k, (model, n_c, n) in enumerate(specs):
        c = cases.small_case(model, n_c=n_c, n_particles=n, seed=5 + k, **kw)
        c.capacity = capacity if k == 0 else 4 * n
        g = eng.add_run(c.n_c, c.dt, c.seed)
        o = OracleRun(c.model, c.n_c, c.n_s, c.dt, c.seed)
        for x in (g, o):
            c.apply(x)
            x.set_compaction(0.01, 0)
        pairs.append((g, o))
    eng.commit()
    return eng, pairs


def shape(capfd):
    m = re.findall(r"block=(\d+) grid=\d+ lds=\d+ priv=(\d) group=(\d+) window=(\d+)", capfd.readouterr().err)
    return tuple(int(v) for v in m[-1])


def check(eng, pairs, calls=(1, 3)):
    for steps in calls:
        eng.step(steps)
        for g, o in pairs:
            o.step(steps, threads=8)
            assert_parity(g, o, probes=False)


@pytest.mark.gpu
@pytest.mark.parametrize("model,n_c,n,capacity", [("monod_mass", 12, 6000, PAST), ("dual_monod", 700, 50_001, PAST),
                                                  ("quad_monod", 900, 30_000, PAST), ("fixed_length", 1, 255, PAST),
                                                  ("simple_acetate", 40, 9000, PAST_WIDE),
                                                  ("monod", 300, 20_000, PAST_WIDE)])
@pytest.mark.parametrize("block", ["256", "512", "1024"])
@pytest.mark.parametrize("feeds", [False, True])
def test_whole_run_accumulators_of_every_block_size(model, n_c, n, capacity, block, feeds, monkeypatch, capfd):
    monkeypatch.setenv("MCST_VERBOSE", "1")
    monkeypatch.setenv("MCST_PARTICLE_BLOCK", block)
    eng, pairs = engine([(model, n_c, n)], capacity, feeds=feeds)
    assert shape(capfd)[:3] == (int(block), 1, 1)
    check(eng, pairs)
    eng.close()


@pytest.mark.gpu
@pytest.mark.parametrize("env", [{"MCST_CONTRIB_LDS": "0"}, {"MCST_TILE_GROUP": "0"}, {"MCST_TILE_GROUP": "4"}])
def test_forced_variants(env, monkeypatch):
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    eng, pairs = engine([("dual_monod", 64, 60_000)], PAST)
    check(eng, pairs)
    eng.close()


@pytest.mark.gpu
@pytest.mark.parametrize("block", [None, "256", "512", "1024"])
def test_batch_in_turns(block, monkeypatch, capfd):
    monkeypatch.setenv("MCST_VERBOSE", "1")
    if block:
        monkeypatch.setenv("MCST_PARTICLE_BLOCK", block)
    eng, pairs = engine([("monod_mass", 12, 200_000), ("monod_mass", 300, 1), ("monod_mass", 30, 90_000),
                         ("monod_mass", 7, 1025), ("monod_mass", 500, 150_000)], 2 * PAST)
    got = shape(capfd)
    assert got[2] == 4 and (not block or got[0] == int(block))
    check(eng, pairs)
    eng.retire(pairs.pop(0)[0])  # its arrays are gone; the others' phantom sub-chunks stay on memory they own
    check(eng, pairs, (2,))
    eng.close()


@pytest.mark.gpu
@pytest.mark.parametrize("block", [None, "256", "512", "1024"])
def test_retired_first_run(block, monkeypatch):
    """Run 0 has the largest tables and goes first: the prefetch past the last
    group stands at the last live tile, never at run 0."""
    if block:
        monkeypatch.setenv("MCST_PARTICLE_BLOCK", block)
    eng, pairs = engine([("monod_mass", 20_000, 30_000), ("monod_mass", 40, 3000), ("monod_mass", 300, 9000)], PAST)
    check(eng, pairs, (2,))
    eng.retire(pairs.pop(0)[0])
    check(eng, pairs, (1, 4))
    eng.close()


@pytest.mark.gpu
def test_tuned_batch_without_probes(capfd, monkeypatch):
    monkeypatch.setenv("MCST_VERBOSE", "1")
    eng, pairs = engine([("monod_mass", 12, 30_000), ("monod_mass", 30, 9000), ("monod_mass", 7, 500)], PAST)
    choice = eng.autotune(1)
    assert shape(capfd)[:3] == (choice["block"], 1, choice["group"])
    done = pairs[0][0].counters()["steps"]
    eng.step(2)
    for g, o in pairs:
        o.step(done + 2)
        assert g.counters() == o.counters()
    eng.close()
