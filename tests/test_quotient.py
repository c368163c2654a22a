"""The quotients that the triangular sweeps form from a reciprocal (csrc/quotient.hpp), on the CPU against the
division: operands at random, near powers of two and with nearly equal mantissas, where a quotient lies next to a
rounding boundary; magnitudes at both ends of the range; zeros, infinities and NaN."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include <limits>
#include <random>
#include "quotient.hpp"
using namespace pfem;
static bool same(double a, double b) { return (a != a && b != b) || std::memcmp(&a, &b, 8) == 0; }
static double ulps(double q, double t)
{
    const double u = std::nextafter(std::fabs(t), std::numeric_limits<double>::infinity()) - std::fabs(t);
    return std::fabs(q - t) / u;
}
int main()
{
    std::mt19937_64 g(7);
    long wrong = 0, far = 0, n = 0;
    auto mantissa = [&](int kind) {
        uint64_t m = g() >> 12;
        if (kind == 1) m &= 15u;                            // just above a power of two
        if (kind == 2) m = ((1ull << 52) - 1) - (m & 15u);  // just below the next
        m |= 0x3ff0000000000000ull;
        double d;
        std::memcpy(&d, &m, 8);
        return d;
    };
    for (long i = 0; i < 30000000; ++i) {
        double d = mantissa(i % 3), s = mantissa(i / 3 % 3);
        if (i % 7 == 0) s = d * mantissa(1);
        const int e = (int)(g() % 199) - 99, f = (int)(g() % 1300) - 650;
        d = std::ldexp(g() & 1 ? d : -d, e);
        s = std::ldexp(s, f);
        const double t = s / d, q = quotient(s, d, 1.0 / d), p = quotient_near(s, d, 1.0 / d);
        ++n;
        if (quotient_ok(q) && !same(q, t)) ++wrong;
        if (ulps(p, t) > 1.0) ++far;
    }
    const double inf = std::numeric_limits<double>::infinity(), nan = std::numeric_limits<double>::quiet_NaN();
    long special = 0;
    for (double s : {0.0, -0.0, 1.0, -3.0, 1e300, -1e308, 5e-324, inf, -inf, nan})
        for (double d : {1.0, -2.5, 1e-20, 1e-160, 1e150, 0.0}) {
            const double t = s / d, p = quotient_near(s, d, 1.0 / d);
            // signed zeros, infinities and NaN as the division's; a subnormal's last bits are not corrected
            const bool fine = same(p, t) || (std::fabs(t) < 1e-290 && std::fabs(p - t) <= 1e-320) || (t == 0.0 && p == 0.0);
            if (!fine) {
                ++special;
                std::printf("%g / %g: %g, not %g\n", s, d, p, t);
            }
        }
    std::printf("%ld of %ld wrong, %ld far, %ld special\n", wrong, n, far, special);
    return wrong || far || special;
}
"""


def test_quotients(tmp_path):
    src, exe = tmp_path / "q.cpp", tmp_path / "q"
    src.write_text(PROGRAM)
    p = subprocess.run(["g++", "-O2", "-std=c++17", "-march=native", "-ffp-contract=off", "-I" + os.path.join(ROOT, "gpupfem2_amd", "csrc"),
                        str(src), "-o", str(exe)], capture_output=True, text=True)
    assert p.returncode == 0, p.stderr
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
