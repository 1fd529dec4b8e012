"""The state variables a model's update() is declared to read and write (READS,
WRITES), on the host: the built-in models' update() with NaN in every variable
outside READS gives the same results, writes all of WRITES and nothing else;
a plugin whose masks would store variables that were never loaded is refused
when it is built."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "biocma-mcst_amd")
CSRC = os.path.join(PKG, "csrc")

PROGRAM = r"""
#include "mcst_common.hpp"
#include "models.hpp"
#include <cmath>
#include <cstdio>
#include <cstring>
using namespace mcst;
static bool same(double a, double b) { return std::memcmp(&a, &b, sizeof a) == 0; }
template <class M>
int check() {
  double p[16] = {};
  M::defaults(p);
  int bad = 0;
  for (uint32_t k = 0; k < 4000; ++k) {
    double x[M::NV], y[M::NV], z[M::NV], c[M::NS], r[14] = {}, cx[M::NS] = {}, cy[M::NS] = {};
    M::init(p, x, 7, k);
    for (int v = 0; v < M::NV; ++v) x[v] *= u01(draw4(3, k, v, 1, 0).x) * 2.0;  // divisions and none
    for (int s = 0; s < M::NS; ++s) c[s] = k % 5 == s ? 0.0 : u01(draw4(4, k, s, 1, 0).x) * (k % 3 ? 1e-3 : 5.0);
    M::record(p, c, r);
    for (int v = 0; v < M::NV; ++v) {
      z[v] = x[v];
      y[v] = reads_var<M>(v) ? x[v] : NAN;
    }
    const int a = M::update(p, 0.01, x, r, cx), b = M::update(p, 0.01, y, r, cy);
    bad += a != b;
    for (int s = 0; s < M::NS; ++s) bad += !same(cx[s], cy[s]);
    for (int v = 0; v < M::NV; ++v) bad += writes_var<M>(v) ? !same(x[v], y[v]) : !same(x[v], z[v]);
  }
  bad += !vars_declared_soundly<M>();
  std::printf("%s %d\n", M::NAME, bad);
  return bad;
}
int main() {
  return check<MonodMass>() + check<DualMonod>() + check<Monod>() + check<FixedLength>() + check<SimpleAcetate>() +
                 check<QuadMonod>()
             ? 1
             : 0;
}
"""


def test_builtin_models_read_and_write_what_they_declare(tmp_path):
    if shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include"):
        pytest.skip("g++ or the HIP headers are not installed")
    src, exe = tmp_path / "vars.cpp", tmp_path / "vars"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{CSRC}", str(src), "-o", str(exe)], check=True, capture_output=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


@pytest.mark.parametrize("masks", ["READS = 0x1", "READS = 0x1, WRITES = 0x4", "WRITES = 0x5"])
def test_unsound_masks_do_not_build(masks, tmp_path):
    from build import build_udf

    src = open(os.path.join(PKG, "examples", "udf_minimal.hpp")).read()
    at = src.index("static constexpr const char* NAME")
    hdr = tmp_path / "masks.hpp"
    hdr.write_text(src[:at] + f"static constexpr uint32_t {masks};\n  " + src[at:])
    with pytest.raises(RuntimeError, match="READS"):
        build_udf(str(hdr), "UdfMinimal", str(tmp_path / "libmasks.so"), verbose=False)
