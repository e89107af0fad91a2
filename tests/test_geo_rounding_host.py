"""quotient() and root() of csrc/vsm_geo.h on the CPU, with estimates of the
reciprocal and the inverse root that are off by as much as the hardware's may
be, next to the middle between two numbers, where rounding is decided by the
last bits of the iteration.

Bounds: the quotient before its last rounding is off by |a/b - q| |b y - 1|,
with q within 1.5 units in the last place of a/b and the reciprocal y within
2^-53 (1 + 2^-40) of 1/b, so by less than 2^-52 units; twice that if the units
change between them, and half a unit for the rounding: 1/2 + 2^-50.  The root
before its last rounding is off by the last correction (at most 1.5 units) times
the error of half the inverse root (one Goldschmidt step from 2^-24: below
2^-47): 1/2 + 2^-46."""
import os
import shutil
import subprocess

import pytest

from vissatsatellitestereo_amd import build

MAIN = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <random>
#define __device__
#define __forceinline__ inline
static double off = 0;                           // relative error of the estimates
inline double __builtin_amdgcn_rcp(double b) { return (1.0 / b) * (1.0 + off); }
inline double __builtin_amdgcn_rsq(double b) { return (1.0 / std::sqrt(b)) * (1.0 + off); }
using std::fma;
#include "vsm_geo.h"
using namespace vsm::geo;
typedef unsigned __int128 u128;

static std::mt19937_64 gen(11);
static void estimate(int i)
{
    const double e = 0x1p-24;
    off = i == 0 ? e : i == 1 ? -e : e * (2.0 * (gen() * 0x1p-64) - 1.0);
}
static long bad = 0, quotients = 0, roots = 0, missed = 0, missed_roots = 0, next_to = 0;
static void check_quotient(double a, double b)
{
    for (int i = 0; i < 3; ++i) {
        estimate(i);
        const double q = quotient(a, b);
        const __float128 r = (__float128)q * b - a;                  // exact: 106 bits
        const double ulp = std::nextafter(std::fabs(q), INFINITY) - std::fabs(q);
        const __float128 err = (r < 0 ? -r : r) / (__float128)std::fabs(b) / ulp;
        ++quotients;
        missed += q != a / b;
        if (!(err <= (__float128)0.5 + 0x1p-50)) { if (bad++ < 5) printf("%a / %a: %a\n", a, b, q); }
    }
}
static void check_root(double x)
{
    for (int i = 0; i < 3; ++i) {
        estimate(i);
        ++roots;
        const double g = root(x);
        const __float128 r = (__float128)x - (__float128)g * g;      // exact: 106 bits
        const __float128 err = (r < 0 ? -r : r) / (2 * (__float128)g) / (std::nextafter(g, INFINITY) - g);
        missed_roots += g != std::sqrt(x);
        if (!(err <= (__float128)0.5 + 0x1p-46)) { if (bad++ < 5) printf("root %a: %a\n", x, g); }
    }
}

int main()
{
    for (long it = 0; it < 400000; ++it) {
        // a divisor, then a dividend that makes the quotient one part in 2^106 or so
        // from a 54-bit number: divisors near powers of two on both sides among them
        uint64_t B = (1ull << 52) | (gen() >> 12) | 1;
        if (it % 3 == 0) B = (1ull << 53) - 1 - 2 * (gen() % (1ull << (gen() % 40)));
        if (it % 3 == 1) B = (1ull << 52) + 1 + 2 * (gen() % (1ull << (gen() % 40)));
        uint64_t inv = B;
        for (int k = 0; k < 6; ++k) inv *= 2 - B * inv;              // 1 / B modulo 2^64
        const bool above = gen() & 1;
        for (int bits = 53; bits <= 55; ++bits) {
            const uint64_t M = (above ? inv : 0 - inv) & ((1ull << bits) - 1);
            if (M >> 53 != 1) continue;
            const u128 P = (u128)B * M;
            const uint64_t A = (uint64_t)((above ? P - 1 : P + 1) >> bits);
            if (A == 0 || A >= 1ull << 53) continue;
            check_quotient(std::ldexp((double)A, (int)(gen() % 120) - 112), std::ldexp((double)B, (int)(gen() % 120) - 112));
        }
        const double a = std::exp(46.0 * (2.0 * (gen() * 0x1p-64) - 1.0)), b = std::exp(46.0 * (2.0 * (gen() * 0x1p-64) - 1.0));
        check_quotient(a, -b);
        check_root(a);
        // roots next to a 54-bit number K: K^2 = c modulo 2^54 or 2^55, c small
        const int64_t c = 8 * ((int64_t)(gen() % 2000001) - 1000000) + 1;
        uint64_t K = 1;
        for (int k = 3; k < 63; ++k)
            if ((K * K - (uint64_t)c) >> k & 1) K += 1ull << (k - 1);
        for (int flip = 0; flip < 4; ++flip)
            for (int bits = 54; bits <= 55; ++bits) {
                const uint64_t L = (((flip & 1) ? 0 - K : K) + ((flip & 2) ? 1ull << (bits - 1) : 0)) & ((1ull << 54) - 1);
                if (L >> 53 != 1) continue;
                const u128 P = (u128)L * L - (u128)(__int128)c;
                if ((uint64_t)P & ((1ull << bits) - 1)) continue;
                const uint64_t X = (uint64_t)(P >> bits);
                if (X >> 52 == 1) { check_root(std::ldexp((double)X, bits & 1)); ++next_to; }
            }
        check_root(b * b);
    }
    printf("%ld quotients (%ld not correctly rounded), %ld roots (%ld), %ld next to a middle\n", quotients, missed,
           roots, missed_roots, next_to);
    return bad != 0 || quotients < 2000000 || next_to < 400000;
}
"""


def test_quotient_and_root_round_as_stated(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = str(tmp_path / "rounding")
    subprocess.run(["g++", "-std=gnu++17", "-O2", "-ffp-contract=off", "-I", build.CSRC, "-I", build.INCLUDE,
                    str(tmp_path / "main.cpp"), "-o", exe], check=True, timeout=120)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
