"""Device export (mcst_run_get_properties, mcst_run_get_repartition) at the
sizes where its shares of LDS change: all variables or some of them, one
window of compartments or several, one block of slots or several, particles in
compartment order or not; against sums over the particles themselves."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("model", ["monod_mass", "quad_monod"])
@pytest.mark.parametrize("n_c,n", [(1, 1), (3, 4096), (910, 4097), (911, 9001), (2730, 64), (2731, 30001),
                                   (8192, 20000), (8193, 20000), (16385, 50001), (40000, 3)])
@pytest.mark.parametrize("in_order", [True, False])
def test_export_equals_sums_over_the_particles(model, n_c, n, in_order):
    import mcst

    rng = np.random.default_rng(n_c + n)
    eng = mcst.Engine(model)
    r = eng.add_run(n_c, 0.01, 7)
    e = np.array([0, n_c - 1]) if n_c > 1 else np.zeros(0, int)
    r.add_flowmap(np.full(n_c, 1e-3), e, e[::-1], np.full(len(e), 1e-6))
    r.set_concentrations(np.ones((eng.n_s, n_c)))
    pos = rng.integers(0, n_c, n)
    if in_order:
        pos = np.sort(pos)
    state = rng.uniform(0.5, 1.5, (eng.n_var, n))
    status = np.where(rng.random(n) < 0.1, rng.integers(2, 4, n), 0)
    r.set_particles(n + 100, pos, status, state, np.zeros(n), np.zeros(n), 1e-9)
    eng.commit()
    values, spatial = r.properties()
    idle = status == 0
    want = np.concatenate([state, state[:1]]) * idle  # both models' mass is the first variable
    np.testing.assert_array_equal(values, want)
    sums = np.stack([np.bincount(pos, weights=w, minlength=n_c) for w in want])
    # at most n terms of one sign: each order of summation errs by less than n * 2^-53
    np.testing.assert_allclose(spatial, sums, rtol=2 * n * 2.0**-53, atol=0)
    np.testing.assert_allclose(r.properties(values=False)[1], sums, rtol=2 * n * 2.0**-53, atol=0)
    np.testing.assert_array_equal(r.repartition(), np.bincount(pos[idle], minlength=n_c))
    eng.close()
