"""Scalar formulas of the kernels whose rounding is relied on (cloudrendering_amd/csrc/rounded.hpp), compiled for the
host."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cloudrendering_amd", "csrc")
HEAD = r'''
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>
#include "rounded.hpp"
using namespace crvpt;
'''


def _run(tmp_path, body):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not found")
    src, exe = tmp_path / "rounded.cpp", tmp_path / "rounded"
    src.write_text(HEAD + body)
    subprocess.run([cxx, "-O2", "-std=c++17", "-ffp-contract=off", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr


def test_quotient_is_the_divisions(tmp_path):
    """Random mantissas and exponents within 2^-40 .. 2^40, then the values a depth or a variance can hold otherwise."""
    _run(tmp_path, r'''
static bool same(float x, float y) { return x == y || (std::isnan(x) && std::isnan(y)); }
int main() {
    std::mt19937_64 g(5);
    long bad = 0;
    for (int i = 0; i < (1 << 22); i++) {
        const uint64_t r = g();
        const float a = std::ldexp(float((r & 0x7fffff) | 0x800000), int((r >> 46) % 40) - 43);
        const float c = std::ldexp(float(((r >> 23) & 0x7fffff) | 0x800000), int((r >> 52) % 40) - 43);
        bad += quotient(a, c, 1.0f / c) != a / c;
    }
    const float inf = INFINITY, nan = NAN;
    for (float a : {0.0f, 1e-30f, 1.0f, 3.0f, 1e30f, inf, nan})
        for (float c : {1e-4f, 0.1f, 10.0f, 1e10f, nan}) bad += !same(quotient(a, c, 1.0f / c), a / c);
    // a zero divisor, and an infinite one: infinite, or no number where the weight's fmaxf makes it 0 as the division's 0
    for (float a : {1.0f, inf}) bad += !same(quotient(a, 0.0f, inf), inf);
    for (float a : {0.0f, 1.0f, nan}) bad += std::fmax(quotient(a, inf, 0.0f), 0.0f) != 0.0f;
    std::printf("%ld mismatches\n", bad);
    return bad != 0;
}
''')


def test_sky_divisions_are_exact(tmp_path):
    """Every mantissa over each divisor of the default sky: the segments' widths and the two of the sRGB curve."""
    _run(tmp_path, r'''
int main() {
    const float stops[] = {-1.0f, -0.1f, 0.0f, 0.4f, 1.0f};
    float div[] = {12.92f, 1.055f, 0.0f, 0.0f, 0.0f, 0.0f};
    for (int i = 0; i < 4; i++) div[2 + i] = stops[i + 1] - stops[i];
    long bad = 0;
    for (float c : div) {
        const float rc = 1.0f / c;
        for (uint32_t m = 0; m < (1u << 23); m++) {
            const uint32_t bits = 0x3f800000u | m;
            float a;
            std::memcpy(&a, &bits, 4);
            bad += divRounded(a, c, rc) != a / c;
        }
        for (float a : {0.0f, -0.0f, -0.7f, 2.0f, 1e-20f}) bad += divRounded(a, c, rc) != a / c;
    }
    std::printf("%ld mismatches\n", bad);
    return bad != 0;
}
''')


def test_power_2_4(tmp_path):
    """Start values up to two units of float and reciprocals up to one unit off, as the hardware's exp2, log2 and rcp
    give them, against the power in long double. Bound: half a unit from the last rounding; the start's relative error e
    of 2^-22 leaves 2 e^2 = 2^-43 after the step, the float correction's own rounding e 2^-22 = 2^-44: 2^-18 units."""
    _run(tmp_path, r'''
int main() {
    std::mt19937 g(3);
    double worst = 0.0;
    auto one = [&](float x) {
        for (int off = -2; off <= 2; off++) {
            float y = float(powl((long double)x, 0.4L));
            for (int k = 0; k < (off < 0 ? -off : off); k++) y = nextafterf(y, off < 0 ? 0.0f : 2.0f);
            const double yd = y, y4 = (yd * yd) * (yd * yd);
            float r = 1.0f / (5.0f * float(y4));
            if (off & 1) r = nextafterf(r, 0.0f);
            const float p = pow24From(double(x) * double(x), yd, y4, r);
            const long double want = powl((long double)x, 2.4L);
            const double ulp = std::ldexp(1.0, std::ilogb(double(want)) - 23);
            const double e = double(fabsl((long double)p - want)) / ulp;
            if (e > worst) worst = e;
        }
    };
    for (int i = 0; i < 400000; i++) one(0.0625f + 1.9375f * float(g() >> 8) * (1.0f / 16777216.0f));
    for (float x : {0.0625f, 0.0904f, 1.0f, 0.99999994f, 2.0f}) one(x);
    std::printf("worst %f units\n", worst);
    return !(worst <= 0.501);
}
''')
