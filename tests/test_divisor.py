"""The tracker's quotients by a value that stays the same (csrc/sg_divisor.hpp),
compiled for the host, against the division itself: every bit, over the exponents
they are used for, with random mantissas, mantissas at the ends of their range and
numerators whose quotient lies next to a rounding boundary."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <cstdint>
#include <cstdio>
#include <cstring>
#include "sg_divisor.hpp"
static uint64_t state = 88172645463325252ull;
static uint64_t next() { state ^= state << 13; state ^= state >> 7; state ^= state << 17; return state; }
static double make(uint64_t mantissa, int e) {  // 1.mantissa * 2^e
    uint64_t u = (uint64_t)(1023 + e) << 52 | (mantissa & 0xFFFFFFFFFFFFFull);
    double v; memcpy(&v, &u, 8); return v;
}
static uint64_t mantissa() {
    switch (next() % 8) {
        case 0: return next() % 4;                 // just above a power of two
        case 1: return ~(next() % 4);              // just below the next
        case 2: return 0x8000000000000ull + next() % 8 - 4;
        default: return next();
    }
}
static long wrong = 0, total = 0;
static void check(const sg::Divisor& D, double a) {
    const double q = D(a), want = a / D.d;
    ++total;
    if (memcmp(&q, &want, 8) && wrong++ < 5) printf("%a / %a = %a, not %a\n", a, D.d, want, q);
}
int main() {
    for (int n = 0; n < 400000; ++n) {
        const double s = next() & 1 ? -1.0 : 1.0;
        const double d = s * make(mantissa(), (int)(next() % 119) - 59);
        if (!sg::Divisor::safe(d)) { printf("%a is not safe\n", d); return 1; }
        const sg::Divisor D(d);
        for (int k = 0; k < 4; ++k) check(D, (next() & 1 ? -1.0 : 1.0) * make(mantissa(), (int)(next() % 401) - 200));
        // next to a boundary: the product of d with a quotient and with one half a unit away
        const double q = make(mantissa(), (int)(next() % 201) - 100), a = q * d;
        const double h = (__builtin_nextafter(q, 1e300) - q) / 2 * d;
        check(D, a);
        check(D, a + h);
        check(D, a - h);
        check(D, __builtin_nextafter(a + h, 0.0));
        check(D, __builtin_nextafter(a + h, 1e300 * a));
    }
    printf("%ld of %ld quotients differ\n", wrong, total);
    const double out[] = {0x1p-60, 0x1p60, 0.0, -0x1p61, __builtin_inf(), __builtin_nan("")};
    for (double v : out) if (sg::Divisor::safe(v)) { printf("%a is safe\n", v); return 1; }
    return wrong != 0;
}
"""


def test_quotients_are_those_of_the_division(tmp_path):
    src, exe = tmp_path / "divisor.cpp", tmp_path / "divisor"
    src.write_text(DRIVER)
    r = subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-D__device__=", "-D__forceinline__=inline",
                        "-I" + os.path.join(ROOT, "simcoflow_amd", "csrc"), str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
