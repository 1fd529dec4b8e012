"""The particle pass's compartment windows and turns: networks whose values
just fit LDS whole, just do not, and need several windows; populations from
less than a block's turn to many turns, in and out of compartment order."""
import numpy as np
import pytest

from mcst import cases
from parity import assert_parity


@pytest.mark.gpu
@pytest.mark.parametrize("model,n_c,n", [("quad_monod", 3072, 40000), ("quad_monod", 3073, 40000), ("quad_monod", 5088, 300),
                                         ("quad_monod", 5089, 40000), ("quad_monod", 20000, 60000),
                                         ("dual_monod", 6145, 30000), ("dual_monod", 20353, 50000),
                                         ("monod", 30000, 20000), ("simple_acetate", 9000, 10000)])
@pytest.mark.parametrize("mixed", [False, True])
def test_windowed_passes_match_oracle(model, n_c, n, mixed):
    import mcst
    from oracle.oracle import OracleRun

    c = cases.small_case(model, n_c=n_c, n_particles=n, n_maps=1)
    eng = mcst.Engine(model)
    g = eng.add_run(c.n_c, c.dt, c.seed)
    o = OracleRun(c.model, c.n_c, c.n_s, c.dt, c.seed)
    for x in (g, o):
        c.apply(x)
        x.set_compaction(0.01, 0)
    if mixed:  # the oracle's initial particles at random places, for both
        p = o.particles()
        pos = np.random.default_rng(3).integers(0, n_c, n)
        for x in (g, o):
            x.set_particles(2 * n, pos, p["status"], p["state"], p["age_hyd"], p["age_div"], o.weight)
    eng.commit()
    eng.step(3)
    o.step(3)
    assert_parity(g, o, probes=False)
    eng.close()
