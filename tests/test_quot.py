"""The sweeps' quotients by a shared or tabulated reciprocal (csrc/c3d_quot.h)
against `/`, on the CPU with stand-ins for the three hardware operations: the
estimates at the ends of their error (FP32 up to two ulps off, FP64 a relative
1e-7, twice what the device shows), and the fixup's documented cases.  Random
operands, zeros, infinities and NaN, and the operands that a wrong rounding would
show at first: the numerators whose quotient by a divisor lies nearest to a
midpoint of two floats, found by solving a 2^k = v (2 q + 1) + d for small d.
About every 16th FP32 divisor, FP64 ones at random."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#define __device__
#define __forceinline__ inline
static int off32;       // ulps
static double off64;    // relative
static float __builtin_amdgcn_rcpf(float v) {
  float r = 1.0f / v;
  for (int k = 0; k < std::abs(off32) && std::isfinite(r) && r != 0; ++k)
    r = std::nextafter(r, off32 > 0 ? INFINITY : -INFINITY);
  return r;
}
static double __builtin_amdgcn_rcp(double v) { return 1.0 / v * (1.0 + off64); }
template <typename T>
static T fixup(T q, T v, T a) {
  if (std::isnan(v) || std::isnan(a)) return NAN;
  const T s = std::signbit(v) != std::signbit(a) ? T(-1) : T(1);
  if ((v == 0 && a == 0) || (std::isinf(v) && std::isinf(a))) return NAN;
  if (v == 0 || std::isinf(a)) return s * INFINITY;
  if (a == 0 || std::isinf(v)) return s * T(0);
  return s * std::fabs(q);
}
static float __builtin_amdgcn_div_fixupf(float q, float v, float a) { return fixup(q, v, a); }
static double __builtin_amdgcn_div_fixup(double q, double v, double a) { return fixup(q, v, a); }
#include "c3d_quot.h"
using namespace c3d;

static uint64_t seed = 88172645463325252ull;
static uint64_t rnd() {
  seed ^= seed << 13; seed ^= seed >> 7; seed ^= seed << 17;
  return seed;
}
static long n, bad;
template <typename T>
static void same(T got, T want, T a, T v) {
  ++n;
  if (std::memcmp(&got, &want, sizeof(T)) && !(std::isnan(got) && std::isnan(want)))
    if (bad++ < 5) std::printf("%.17g / %.17g: %.17g, not %.17g\n", (double)a, (double)v,
                               (double)got, (double)want);
}
static void check(float a, float v) {
  for (off32 = -2; off32 <= 2; ++off32) same(quot(a, v, quot_recip(v)), a / v, a, v);
}
static void check(double a, double v) {
  static const double ends[] = {-1e-7, 0.0, 1e-7};
  for (double o : ends) {
    off64 = o;
    same(quot(a, v, quot_recip(v)), a / v, a, v);
  }
  if (v != 0 && std::isfinite(v)) same(quot(a, v, tab_recip(v, 1.0 / v)), a / v, a, v);
}
// all numerators of B bits with a 2^k = v (2 q + 1) + d, |d| <= dmax (times the
// power of two in v); V: v as an integer of B bits
template <typename T, int B>
static void midpoints(uint64_t V, int dmax) {
  typedef unsigned __int128 u128;
  const int s = __builtin_ctzll(V);
  if (s > 2) return;
  const uint64_t O = V >> s;
  for (int k = B - 1; k <= B; ++k) {
    u128 inv = 1;
    for (int i = 0; i < k - s; ++i) inv = inv & 1 ? (inv + O) / 2 : inv / 2;
    for (int d = -(dmax >> s); d <= dmax >> s; ++d) {
      if (!d) continue;
      uint64_t A = (uint64_t)(inv * (u128)(d < 0 ? -d : d) % O);
      if (d < 0) A = O - A;
      for (; A < 1ull << B; A += O)
        if (A >= 1ull << (B - 1)) check((T)A, (T)V);
    }
  }
}
int main() {
  for (uint64_t V = (1u << 23) + rnd() % 16; V < 1u << 24; V += 16 + (rnd() % 3 - 1))
    midpoints<float, 24>(V, 5);
  midpoints<float, 24>((1u << 24) - 1, 5);
  for (int i = 0; i < 100000; ++i) midpoints<double, 53>((1ull << 52) + rnd() % (1ull << 52), 5);
  midpoints<double, 53>((1ull << 53) - 1, 5);
  for (int i = 0; i < 1000000; ++i) {
    const double a = std::ldexp(1.0 + (rnd() >> 12) * 0x1p-52, (int)(rnd() % 61) - 30);
    const double v = std::ldexp(1.0 + (rnd() >> 12) * 0x1p-52, (int)(rnd() % 61) - 30);
    const double sa = rnd() & 1 ? a : -a, sv = rnd() & 1 ? v : -v;
    check(sa, sv);
    check((float)sa, (float)sv);
    // a tabulated FP64 reciprocal of the pivot that was rounded to FP32
    const float f = (float)sv;
    same(quot((float)sa, f, tab_recip(f, 1.0 / sv)), (float)sa / f, (float)sa, f);
  }
  const double sp[] = {0.0, -0.0, 1.0, -3.0, INFINITY, -INFINITY, NAN};
  for (double a : sp)
    for (double v : sp) {
      check(a, v);
      check((float)a, (float)v);
    }
  std::printf("%ld quotients, %ld differ\n", n, bad);
  return bad != 0;
}
"""


def test_quot_rounds_like_division(tmp_path):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("no g++")
    (tmp_path / "quot.cpp").write_text(SRC)
    fma = ["-mfma"] if " fma " in open("/proc/cpuinfo").read() else []
    subprocess.run([gxx, "-O2", "-std=c++17", "-ffp-contract=off", *fma, "-I",
                    os.path.join(ROOT, "channel3d_amd", "csrc"), "quot.cpp", "-o", "quot"],
                   cwd=tmp_path, check=True)
    r = subprocess.run([str(tmp_path / "quot")], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
