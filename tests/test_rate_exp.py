"""The rate constants' exponential (astr_amd/csrc/rate_exp.hpp), its text
compiled for the host, against the C library's 80-bit one.

Bound: the double-precision exp of the GPU's library, which it takes the place
of, is off by at most 0.868 ulp and by 0.3015 RMS on the same distribution
(16 million arguments); neither may be larger here."""
import os
import subprocess

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "astr_amd", "csrc", "rate_exp.hpp")

PROGRAM = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>
#define __device__
#define __forceinline__ inline
using std::fma;
using std::ldexp;
static int __double2loint(double t) { int64_t b; std::memcpy(&b, &t, 8); return (int)b; }
#include "rate_exp.hpp"
int main() {
  const astr::RateExpConstants K;
  std::mt19937_64 g(1);
  double worst = 0.0;
  long double sum = 0.0L;
  const int n = 4000000;
  for (int i = 0; i < n; i++) {
    const double range[4] = {699.0, 60.0, 5.0, 0.4};
    const double x = range[i % 4] * (2.0 * (double)(g() >> 11) * 0x1p-53 - 1.0);
    const long double want = std::exp((long double)x);
    const double ulp = std::ldexp(1.0, std::ilogb((double)want) - 52);
    const double e = (double)(std::fabs((long double)astr::rate_exp_in(x, K) - want) / ulp);
    if (e > worst) worst = e;
    sum += (long double)e * e;
  }
  std::printf("%.4f %.4f %d\n", worst, (double)std::sqrt(sum / n),
              astr::rate_exp_in(0.0, K) == 1.0 && std::isnan(astr::rate_exp_in(NAN, K)));
}
"""


def test_exponential_is_as_exact_as_the_library_s(tmp_path):
    src, exe = tmp_path / "rate_exp.cpp", tmp_path / "rate_exp"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", os.path.dirname(HEADER), "-o", str(exe),
                    str(src)], check=True)
    worst, rms, special = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()
    assert special == "1"
    assert float(worst) <= 0.868 and float(rms) <= 0.3015, (worst, rms)
