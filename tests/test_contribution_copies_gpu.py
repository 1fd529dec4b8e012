"""The copies of the contribution accumulator: batches on both sides of the
number of values (16 384) above which one copy is used, for models with 1, 2
and 4 species, and a batch that crosses it when a run joins and leaves."""
import pytest

from mcst import cases
from parity import assert_parity, assert_snapshot, make_pair, snapshot


@pytest.mark.gpu
@pytest.mark.parametrize("model,n_c", [("monod_mass", 16384), ("monod_mass", 16385), ("dual_monod", 8192),
                                       ("dual_monod", 8193), ("quad_monod", 4096), ("quad_monod", 4097),
                                       ("monod", 255), ("simple_acetate", 257)])
def test_batches_around_the_line(model, n_c):
    c = cases.small_case(model, n_c=n_c, n_particles=20000, n_maps=1)
    eng, g, o = make_pair(c)
    for steps in (1, 3):
        eng.step(steps)
        o.step(steps)
        assert_parity(g, o)
    eng.close()


@pytest.mark.gpu
def test_a_run_that_crosses_the_line_joins_and_leaves():
    import mcst
    from oracle.oracle import OracleRun

    eng = mcst.Engine("monod_mass")
    eng.reserve(200_000, 2)
    eng.commit()
    pairs = []
    for k, n_c in enumerate((40, 17000)):
        c = cases.small_case("monod_mass", n_c=n_c, n_particles=8000, seed=20 + k, n_maps=1)
        o = OracleRun(c.model, c.n_c, c.n_s, c.dt, c.seed)
        c.apply(o)
        o.set_compaction(0.01, 0)
        pairs.append((c, o))

    def join(c):
        r = eng.add_run(c.n_c, c.dt, c.seed)
        c.apply(r)
        assert eng.admit() == 1
        return r

    a = join(pairs[0][0])
    eng.step(2)
    b = join(pairs[1][0])  # one copy from here on
    eng.step(3)
    pairs[1][1].step(3)
    assert_snapshot(snapshot(b), pairs[1][1])
    eng.retire(b)          # several again
    eng.step(2)
    pairs[0][1].step(7)
    assert_snapshot(snapshot(a), pairs[0][1])
    eng.close()
