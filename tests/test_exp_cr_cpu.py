"""exp_cr (csrc/exp_acc.hpp), the device exponential of the granule, Golgi and
olive models, returns exp_acc's value bit for bit: built for the host with
hipcc, over random arguments of the models' and the whole range, tiny ones,
the ends of the range, infinities and NaN; exp_libm, the synaptic decay of
the resident RKC kernel, is the C library's wherever it claims to be.  (exp_acc itself is pinned to
60-digit values in test_exp_acc_cpu.py.)"""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "cerebellum-neuron-model-simulation-using-rkc_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"

PROGRAM = r"""
#include "exp_acc.hpp"
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
static long bad = 0;
static void one(double x) {
  const double a = cbrkc::exp_cr(x), b = cbrkc::exp_acc(x);
  if (std::memcmp(&a, &b, 8) != 0 && !(a != a && b != b)) {
    if (bad++ < 5) std::printf("%a: %a, not %a\n", x, a, b);
  }
}
int main() {
  srand48(3);
  for (long i = 0; i < 1000000; i++) {
    const double u = drand48() - 0.5;
    one(8.0 * u);
    one(1400.0 * u);
    one(1e-3 * u);
    one(1e-13 * u);
  }
  for (double x : {0.0, -0.0, 5e-324, 708.999, -707.999, 709.0, 709.79, 710.0, -708.0, -745.2, -746.0, 1e300, -1e300,
                   1.0 / 0.0, -1.0 / 0.0, 0.0 / 0.0, 0.34657359027997264, -0.34657359027997264})
    one(x);
  // exp_libm: the host libm's value wherever it says so, and that nearly always
  long unsure = 0, n = 2000000;
  for (long i = 0; i < n; i++) {
    const double u = drand48(), x = i % 2 ? -0.21 * u : -5.0 * u;
    bool sure;
    const double a = cbrkc::exp_libm(x, sure), b = std::exp(x);
    if (!sure) unsure++;
    else if (a != b && bad++ < 5) std::printf("exp_libm %a: %a, not %a\n", x, a, b);
  }
  if (unsure > n / 35) std::printf("unsure %ld of %ld\n", unsure, n);
  std::printf("bad %ld\n", bad);
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_exp_cr_equals_exp_acc(tmp_path):
    src = tmp_path / "t.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "t"
    subprocess.run([HIPCC, "-O2", "-ffp-contract=off", "-x", "hip", "--offload-arch=gfx950", "-I", CSRC, str(src),
                    "-o", str(exe)], check=True, capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    assert out.strip() == "bad 0", out
