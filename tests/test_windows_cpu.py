"""Where the particle pass's compartment window stands (window_at, window_next
in csrc/mcst_common.hpp), compiled for the host: it lies in the network and
holds the compartment it was moved for, stays while that is in its middle half,
and does not move twice for one compartment (a move flushes the block's
accumulator), at the network's ends neither."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "biocma-mcst_amd", "csrc")

PROGRAM = r"""
#include "mcst_common.hpp"
#include <cstdio>
#include <cstdlib>
using namespace mcst;
int main(int, char** argv) {
  const uint32_t win = std::atoi(argv[1]), n_c = std::atoi(argv[2]);
  const uint32_t step = n_c > 3000 ? 37u : 1u;
  long bad = 0;
  for (uint32_t w0 = 0; w0 + win <= n_c; w0 += (n_c - win) / 64 + 1)
    for (uint32_t c0 = 0; c0 < n_c; c0 += step) {
      const uint32_t w1 = window_next(c0, w0, win, n_c);
      bad += w1 + win > n_c || window_at(c0, win, n_c) > c0 || c0 - window_at(c0, win, n_c) >= win;
      bad += c0 < w1 || c0 - w1 >= win;
      bad += c0 >= w0 + win / 4 && c0 < w0 + win / 4 + win / 2 && w1 != w0;
      bad += window_next(c0, w1, win, n_c) != w1;
    }
  std::printf("%ld\n", bad);
  return bad != 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include"):
        pytest.skip("g++ or the HIP headers are not installed")
    d = tmp_path_factory.mktemp("windows")
    src, exe = d / "windows.cpp", d / "windows"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{CSRC}",
                    str(src), "-o", str(exe)], check=True, capture_output=True, timeout=120)
    return exe


@pytest.mark.parametrize("win,n_c", [(1, 2), (2, 3), (3, 5), (4, 4), (64, 65), (64, 1000), (1017, 1018), (5088, 5089),
                                     (5088, 5500), (5088, 10175), (5088, 50000), (20352, 30000)])
def test_window_moves_once_and_holds_its_compartment(program, win, n_c):
    r = subprocess.run([str(program), str(win), str(n_c)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
