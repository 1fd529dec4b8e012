"""How many steps of time-dependent feeds are prepared at once (feed_rows in
csrc/mcst_common.hpp, compiled for the host): a short call or a run's last
steps prepare no more than they take, single steps ever longer blocks, and the
work stays within twice the steps taken.  On the GPU: blocks that wrap around
the rows' ring and runs that end inside one, against the oracle."""
import ctypes
import os
import random
import shutil
import subprocess

import pytest

from mcst import cases
from parity import assert_parity

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "biocma-mcst_amd", "csrc")

PROGRAM = r"""
#include "mcst_common.hpp"
extern "C" uint32_t rows(uint32_t step, uint32_t target, uint64_t left, uint32_t last) {
  return mcst::feed_rows(step, target, left, last);
}
"""


@pytest.fixture(scope="module")
def feed_rows(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include"):
        pytest.skip("g++ or the HIP headers are not installed")
    d = tmp_path_factory.mktemp("feed_rows")
    src, lib = d / "rows.cpp", d / "librows.so"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{CSRC}", str(src), "-o", str(lib)], check=True, capture_output=True, timeout=120)
    rows = ctypes.CDLL(str(lib)).rows
    rows.argtypes = [ctypes.c_uint32, ctypes.c_uint32, ctypes.c_uint64, ctypes.c_uint32]
    rows.restype = ctypes.c_uint32
    return rows


def test_a_call_prepares_its_own_steps(feed_rows):
    for n in (1, 2, 5, 255, 256):
        assert feed_rows(0, 2**32 - 1, n, 0) == n
    assert feed_rows(0, 2**32 - 1, 10_000, 0) == 256
    assert feed_rows(7, 9, 10_000, 0) == 2 and feed_rows(2**32 - 2, 2**32 - 1, 4, 256) == 1


@pytest.mark.parametrize("seed", range(6))
def test_every_step_has_its_rows_at_twice_their_work(feed_rows, seed):
    """The host's loop: before a step its row and, within a call, the next
    step's must be there (none past the run's last)."""
    rng = random.Random(seed)
    target = rng.choice([40, 700, 2**32 - 1])
    step = begin = end = work = fills = 0
    while step < min(target, 900):
        left = 1 if seed == 0 else rng.choice([1, 1, 2, 7, 60, 300])
        while left and step < target:
            need = min(target, step + (2 if left > 1 else 1))
            if not (begin <= step and need <= end):
                rows = feed_rows(step, target, left, end - begin)
                assert 1 <= rows <= 256
                begin, end = step, step + rows
                work += rows
                fills += 1
            assert begin <= step and need <= end and need <= target
            step, left = step + 1, left - 1
    assert work <= 2 * step + fills  # a row prepared again where a block ends within a call
    assert seed or fills <= 12


@pytest.mark.gpu
@pytest.mark.parametrize("calls", [[3, 100, 200, 256, 1, 300], [1] * 20 + [250, 250], [300, 7, 300]])
@pytest.mark.parametrize("target", [None, 41, 257])
def test_blocks_and_early_ends_match_oracle(calls, target):
    import mcst
    from oracle.oracle import OracleRun

    c = cases.small_case("dual_monod", n_c=12, n_particles=700, seed=3)
    c.feeds = [("linear", 1e-3, 0.02, 3, 9, [0, 1], [8.0, 0.5]), ("exponential", 0.0, -3.0, 10, 4, [1], [1e-4])]
    c.params = None  # slow growth: hundreds of steps
    eng = mcst.Engine("dual_monod")
    pairs = []
    for t in (target, None):
        g = eng.add_run(c.n_c, c.dt, c.seed)
        o = OracleRun(c.model, c.n_c, c.n_s, c.dt, c.seed)
        for x in (g, o):
            c.apply(x)
            x.set_compaction(0.01, 0)
        if t:
            g.set_step_target(t)
        pairs.append((g, o, t or 2**32 - 1))
    eng.commit()
    done = 0
    for n in calls:
        eng.step(n)
        for _, o, t in pairs:
            if min(t, done + n) > min(t, done):
                o.step(min(t, done + n) - min(t, done))
        done += n
    for g, o, _ in pairs:
        assert_parity(g, o, probes=False)
    eng.close()
