"""The shared-reciprocal quotients and roots of the FP64 pair sums (csrc/sphfem_fpmath.h) on the CPU:
equal to the correctly rounded operators for random operands over 120 binades and for divisors just
below a power of two, from seeds with 20 good bits (the hardware's approximations have more)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include "%s/sph_fem_2d_cutting_gpu_amd/csrc/sphfem_fpmath.h"
using namespace sphfem;
int main() {
    std::mt19937_64 g(3);
    std::uniform_real_distribution<double> u(-1, 1);
    long bad = 0;
    for (long k = 0; k < 4000000; k++) {
        double b = std::ldexp(1.5 + 0.5 * u(g), (int)(60 * u(g)));
        const double a = std::ldexp(u(g), (int)(60 * u(g)));
        if (k %% 5 == 0) {
            const unsigned long long m = 0x3ff0000000000000ull | ((1ull << 52) - 1 - (g() %% 64));
            std::memcpy(&b, &m, 8);
        }
        const double s = 1 + u(g) * std::ldexp(1, -20);
        double h;
        bad += quot(a, recip_from(b, 1 / b * s)) != a / b;
        const double q = sqrt_from(b, 1 / std::sqrt(b) * s, h);
        bad += q != std::sqrt(b);
        bad += quot(a, recip_from(q, 2 * h)) != a / q;
        const double x = (double)(float)b;     // the seed belongs to b, as in the pair term
        const double f = sqrtf_from(x, 1 / std::sqrt(b) * s, h);
        bad += f != (double)(float)std::sqrt(x);
        const Recip r = recip_from(f, 2 * h);
        bad += r.y != 1 / f || quot(a, r) != a / f;
    }
    std::printf("%%ld\n", bad);
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_quotients_and_roots_are_correctly_rounded(tmp_path):
    src = tmp_path / "q.cpp"
    src.write_text(SOURCE % ROOT)
    exe = tmp_path / "q"
    subprocess.run(["g++", "-O2", "-mfma", "-ffp-contract=off", "-std=c++17", str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.strip() == "0"


ROUNDED = r"""
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include "%s/sph_fem_2d_cutting_gpu_amd/csrc/sphfem_fpmath.h"
using namespace sphfem;
int main() {
    std::mt19937_64 g(4);
    std::uniform_real_distribution<double> u(-1, 1);
    long bad = 0, plain = 0;
    for (long k = 0; k < 4000000; k++) {
        // roots whose fraction bits are random, or all ones but for up to 63 units
        unsigned long long m = (1ull << 52) - 1 - (k %% 2 ? g() %% 64 : g() >> 12);
        m |= (unsigned long long)(1023 + (int)(60 * u(g))) << 52;
        double b, h;
        std::memcpy(&b, &m, 8);
        const double x = b * b;
        const double q = sqrt_from(x, 1 / std::sqrt(x) * (1 + u(g) * std::ldexp(1, -20)), h);
        bad += q != std::sqrt(x);
        const Recip r = recip_rounded(q, 2 * h);
        const double a = k %% 3 ? q * u(g) : std::ldexp(1, (int)(60 * u(g)));
        bad += r.y != 1 / q;
        bad += quot(a, r) != a / q;
        plain += recip_from(q, 2 * h).y != 1 / q;
    }
    std::printf("%%ld %%d\n", bad, plain > 0);
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_reciprocals_of_double_roots_are_correctly_rounded(tmp_path):
    """1 / distance of the heat term, which is used itself and not only in quotients; the unrounded form
    differs at the divisors of all ones that the test holds."""
    src = tmp_path / "r.cpp"
    src.write_text(ROUNDED % ROOT)
    exe = tmp_path / "r"
    subprocess.run(["g++", "-O2", "-mfma", "-ffp-contract=off", "-std=c++17", str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split() == ["0", "1"]


RANGE = r"""
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include "%s/sph_fem_2d_cutting_gpu_amd/csrc/sphfem_fpmath.h"
using namespace sphfem;
int main() {
    std::mt19937_64 g(6);
    std::uniform_real_distribution<double> u(-1, 1);
    long bad = 0, held = 0, n = 4000000;
    for (long k = 0; k < n; k++) {
        unsigned long long m = g();                        // every exponent: subnormal, infinite, NaN
        if (k %% 64 == 0) m &= 1ull << 63;                 // zeros
        double a;
        std::memcpy(&a, &m, 8);
        const double b = std::pow(10., 100 * u(g));
        if (!quot_holds(a)) continue;
        held++;
        bad += quot(a, recip_from(b, 1 / b * (1 + u(g) * std::ldexp(1, -20)))) != a / b;
    }
    const double end[] = {0., -0., 5e-324, 1e-308, 1e-200, 1e200, 1.7e308, INFINITY, -INFINITY, NAN};
    for (double a : end) bad += quot_holds(a);
    std::printf("%%ld %%d\n", bad, held > n / 2);
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_dividends_that_the_quotient_is_used_for(tmp_path):
    """Dividends of any exponent by the densities that the in-support sums take: those that quot_holds lets
    through are divided correctly, and zeros, subnormal, infinite and NaN ones are not let through."""
    src = tmp_path / "d.cpp"
    src.write_text(RANGE % ROOT)
    exe = tmp_path / "d"
    subprocess.run(["g++", "-O2", "-mfma", "-ffp-contract=off", "-std=c++17", str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split() == ["0", "1"]
