"""Event counters of batches on both sides of each size at which the number of
counter shards per run changes (16 and 256 runs), against the oracle: runs of
uneven size, so that groups of the resolve kernel hold one run and several."""
import numpy as np
import pytest

from mcst import cases


@pytest.mark.gpu
@pytest.mark.parametrize("n_runs", [1, 3, 16, 17, 256, 257])
def test_counters_of_a_batch(n_runs):
    import mcst
    from oracle.oracle import OracleRun

    eng = mcst.Engine("monod_mass")
    g, o = [], []
    for i in range(n_runs):
        n = [40, 1, 1025, 300, 5000][i % 5] if n_runs > 1 else 20000
        c = cases.small_case("monod_mass", n_c=[12, 5, 1][i % 3], n_particles=n, seed=100 + i)
        r = eng.add_run(c.n_c, c.dt, c.seed)
        q = OracleRun(c.model, c.n_c, c.n_s, c.dt, c.seed)
        for x in (r, q):
            c.apply(x)
        q.set_compaction(0.01, 0)
        g.append(r)
        o.append(q)
    eng.commit()
    eng.step(4)
    for q in o:
        q.step(4)
    for r, q in zip(g, o):
        assert r.counters() == q.counters()
    total = {k: sum(r.counters()[k] for r in g) for k in ("births", "moves", "exits", "processed")}
    assert all(total[k] > 0 for k in total if n_runs > 1 or k != "exits"), total
    np.testing.assert_array_equal(g[0].particles()["pos"], o[0].particles()["pos"])
    eng.close()
