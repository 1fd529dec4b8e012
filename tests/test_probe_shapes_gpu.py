"""The launch shape of probing runs, whose pass has 256 threads a block: the
grid is that kernel's own (two blocks a compute unit, where the other pass may
have one of 512), and a block size tuned or forced for other runs leaves them
their LDS accumulator."""
import re

import pytest

from mcst import cases
from parity import assert_parity, make_pair


def shape(err):
    m = re.findall(r"particle pass: block=(\d+) grid=(\d+) lds=(\d+) priv=(\d)", err)
    return tuple(int(v) for v in m[-1])


@pytest.mark.gpu
@pytest.mark.parametrize("block", [None, "512", "1024"])
@pytest.mark.parametrize("network", ["whole", "window"])
def test_probing_pass_has_its_own_shape(block, network, monkeypatch, capfd):
    import mcst

    monkeypatch.setenv("MCST_VERBOSE", "1")
    # the windowed pass without probes has one block of 1024 threads a compute unit
    ref = mcst.Engine("quad_monod")
    c = cases.lattice50k(n_particles=1000)
    c.capacity = 600_000
    c.apply(ref.add_run(c.n_c, c.dt, c.seed))
    ref.commit()
    one, cus, _, _ = shape(capfd.readouterr().err)
    assert one == 1024
    ref.close()
    if block:
        monkeypatch.setenv("MCST_PARTICLE_BLOCK", block)
    if network == "whole":
        c = cases.small_case("dual_monod", n_c=700, n_particles=100_000)
    else:
        c = cases.lattice50k(n_particles=100_000)
    eng, g, o = make_pair(c, capacity=600_000)
    blk, grid, lds, priv = shape(capfd.readouterr().err)
    assert (blk, grid, priv) == (256, 2 * cus, 1)
    eng.step(3)
    o.step(3, threads=8)
    assert_parity(g, o)
    assert eng.autotune(1)["block"] == 256
    assert shape(capfd.readouterr().err)[0] == 256
    eng.close()
