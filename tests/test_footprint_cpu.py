"""Device bytes of a served run (serve.footprint) against the library's own
rules (run_copies, S_COPY_ENTRIES, VF_ROWS of csrc/mcst_common.hpp, compiled for
the host): the copies of its contributions and the rows of its time-dependent
feeds."""
import copy
import ctypes
import os
import shutil
import subprocess

import pytest

from mcst import cases
from mcst.serve import footprint

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "biocma-mcst_amd", "csrc")
PROGRAM = r"""
#include "mcst_common.hpp"
extern "C" uint32_t copies(int ns, uint32_t entries) {
  return entries <= mcst::S_COPY_ENTRIES ? mcst::run_copies(ns) : 1u;
}
extern "C" uint32_t vf_rows() { return mcst::VF_ROWS; }
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include"):
        pytest.skip("g++ or the HIP headers are not installed")
    d = tmp_path_factory.mktemp("footprint")
    src, lib = d / "rules.cpp", d / "librules.so"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{CSRC}", str(src), "-o", str(lib)], check=True, capture_output=True, timeout=120)
    return ctypes.CDLL(str(lib))


def bare(n_s, n_c):
    return cases.Case("x", "m", n_c, n_s, 0.01, 1, [])


@pytest.mark.parametrize("n_s", [1, 2, 3, 4])
@pytest.mark.parametrize("n_c", [1, 4096, 4097, 5461, 5462, 8192, 8193, 16384, 16385])
def test_liquid_counts_the_copies_the_library_keeps(rules, n_s, n_c):
    assert footprint(bare(n_s, n_c), 2) == 8 * (6 + rules.copies(n_s, n_s * n_c)) * n_s * n_c


def test_rows_of_time_dependent_feeds(rules):
    c = bare(2, 30)
    base = footprint(c, 3)
    row = 8 * rules.vf_rows()

    def more(feeds, gas=None):
        d = copy.copy(c)
        d.feeds, d.two_phase = feeds, {"gas_feeds": gas} if gas else None
        return footprint(d, 3) - base

    const, lin, exp = "constant", "linear", "exponential"
    assert more([(const, 1e-3, 0.0, 0, 5, [0], [1.0])]) == 0
    assert more([(lin, 1e-3, 0.1, 0, None, [0], [1.0])]) == row
    assert more([(lin, 1e-3, 0.1, 0, 5, [0], [1.0])]) == 2 * row  # and its outlet's threshold
    # an outlet's threshold follows its first feed
    assert more([(const, 1e-3, 0.0, 0, 5, [0], [1.0]), (lin, 1e-3, 0.1, 0, 5, [0], [1.0])]) == row
    assert more([(lin, 1e-3, 0.1, 0, 5, [0], [1.0]), (exp, 1e-3, 0.1, 2, 5, [0], [1.0])]) == 3 * row
    assert more([], [(exp, 1e-3, 0.1, 0, 5, [1], [1.0])]) == row  # a gas outlet has no threshold
