"""The particle pass loads the variables a model reads and stores those it
writes: every variable of Idle, inactive and dividing slots against the oracle,
from states whose written-only and division-only variables hold other values,
for the small batch's pass and the general one (pools past its limit), counts
that end inside a lane's pair or a sub-chunk, and requests past the 16 staged
per sub-chunk."""
import numpy as np
import pytest

from mcst import cases
from parity import assert_parity

MODELS = ["monod_mass", "dual_monod", "monod", "fixed_length", "simple_acetate", "quad_monod"]
OTHER = {"monod": [3, 5], "simple_acetate": [5, 6, 7, 8], "quad_monod": [4, 5, 6, 7]}  # not read by the update


@pytest.mark.gpu
@pytest.mark.parametrize("model", MODELS)
@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("n,inactive,dividing", [(1, 0.0, 1.0), (127, 0.3, 0.0), (2049, 0.2, 0.05), (3001, 0.4, 0.9)])
def test_all_variables_against_the_oracle(model, general, n, inactive, dividing):
    import mcst
    from oracle.oracle import OracleRun

    c = cases.small_case(model, n_c=20, n_particles=n)
    o = OracleRun(c.model, c.n_c, c.n_s, c.dt, c.seed)
    c.apply(o)
    p = o.particles()
    rng = np.random.default_rng(n)
    x = p["state"].copy()
    for v in OTHER.get(model, []):
        x[v] = rng.uniform(0.5, 2.0, n) * 1e-7
    x[0] = np.where(rng.random(n) < dividing, 4.0 * x[0], x[0])
    status = np.where(rng.random(n) < inactive, rng.integers(2, 4, n), 0)
    cap = 3072 * 1024 + 1 if general else 2 * n + 100
    eng = mcst.Engine(c.model)
    g = eng.add_run(c.n_c, c.dt, c.seed)
    o = OracleRun(c.model, c.n_c, c.n_s, c.dt, c.seed)
    for r in (g, o):
        c.apply(r)
        r.set_compaction(0.9, 0)  # the inactive stay
        r.set_particles(cap, p["pos"], status, x, np.zeros(n), np.zeros(n), 1e9)
    eng.commit()
    for steps in (1, 1, 3):
        eng.step(steps)
        o.step(steps)
        assert_parity(g, o, probes=False)
    eng.close()
