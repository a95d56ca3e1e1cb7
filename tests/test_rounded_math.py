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
