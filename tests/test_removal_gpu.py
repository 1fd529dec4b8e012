"""Removal of inactive slots in both of its forms (one block per run; counts
per tile and a fill by the whole grid, for runs of more than 512 tiles of
capacity) against the oracle: runs that start with a share of Exit and Dead
slots, at sizes around the forms' chunks (4096 slots, 1024-slot tiles)."""
import numpy as np
import pytest

from mcst import cases
from parity import close


def define(run, c, n, cap, share, seed):
    rng = np.random.default_rng(seed)
    c.apply(run, particles=False)
    status = np.where(rng.random(n) < share, rng.integers(2, 4, n), 0)
    run.set_particles(cap, rng.integers(0, c.n_c, n), status, rng.uniform(1e-15, 1.2e-15, (2, n)),
                      rng.uniform(0, 5, n), rng.uniform(0, 5, n), 1e9)


@pytest.mark.gpu
@pytest.mark.parametrize("cap", [0, 520 * 1024])  # 0: twice the particles
@pytest.mark.parametrize("share", [0.03, 0.5, 0.995, 1.0])
@pytest.mark.parametrize("n", [1, 7, 1025, 4096, 4099, 8200, 50001])
def test_removal_matches_oracle(n, share, cap):
    import mcst
    from oracle.oracle import OracleRun

    eng = mcst.Engine("monod_mass")
    pairs = []
    for k, m in enumerate((n, 3000)):  # a second run shares the launch
        c = cases.small_case("monod_mass", n_c=8, seed=5 + k)
        g = eng.add_run(c.n_c, c.dt, c.seed)
        o = OracleRun(c.model, c.n_c, c.n_s, c.dt, c.seed)
        for x in (g, o):
            define(x, c, m, max(cap, 2 * m), share, 17 + k)
            x.set_compaction(0.01, 0)
        pairs.append((g, o))
    eng.commit()
    for steps in (1, 1, 5):
        eng.step(steps)
        for g, o in pairs:
            o.step(steps)
            assert g.counters() == o.counters()
            p, q = g.particles(), o.particles()
            np.testing.assert_array_equal(p["pos"], q["pos"])
            np.testing.assert_array_equal(p["status"], q["status"])
            for k in ("state", "age_hyd", "age_div"):
                close(p[k], q[k], what=k)
    eng.close()
