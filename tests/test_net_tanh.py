"""The FP64 tanh of the networks, its host build against the C library's
extended-precision tanh (64-bit significand), with a reciprocal that is off by up to
four units as the device's may be: at most 0.7 units in the last place over all
magnitudes, the limits and NaN as they are."""
import os
import subprocess

import pytest

from conftest import PKG_DIR

PROG = r"""
#include <cmath>
#include <cstdio>
#include <random>
#include "ptmc_tanh.hpp"

int main()
{
    std::mt19937_64 g(1);
    std::uniform_real_distribution<double> u(0.0, 1.0);
    double worst = 0.0, at = 0.0;
    auto check = [&](double x) {
        const double off = (u(g) * 2.0 - 1.0) * 0x1.0p-50;  // the reciprocal's error, up to four units
        const double v = ptmc::net_tanh(x, [&](double d) { return (1.0 + off) / d; });
        const long double w = tanhl((long double)x);
        const double ulp = std::nextafter(std::fabs((double)w), 2.0) - std::fabs((double)w);
        const double e = (double)(fabsl((long double)v - w) / (long double)ulp);
        if (!(e <= worst)) { worst = e; at = x; }
    };
    for (int i = 0; i < 1500000; ++i) {
        check((u(g) < 0.5 ? -1 : 1) * std::exp(u(g) * (std::log(25.0) - std::log(1e-9)) + std::log(1e-9)));
        check(u(g) * 2.0);
        check(std::ldexp(u(g), -(int)(u(g) * 1070)));
    }
    // about the steps of k and the clamp
    for (int k = 0; k < 60; ++k)
        for (int i = -2000; i <= 2000; ++i) check((k + 0.5) * 0.34657359027997264 + i * 1e-12);
    std::printf("%.4f ulp at %.17g\n", worst, at);
    const double inf = INFINITY;
    auto f = [](double x) { return ptmc::net_tanh(x, [](double d) { return 1.0 / d; }); };
    bool ok = f(0.0) == 0.0 && std::signbit(f(-0.0)) && f(inf) == 1.0 && f(-inf) == -1.0 && std::isnan(f(NAN)) &&
              f(1e300) == 1.0;
    return ok && worst <= 0.7 ? 0 : 1;
}
"""


def test_error_in_ulp(tmp_path):
    import build

    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    (tmp_path / "t.hip").write_text(PROG)
    subprocess.run([build.HIPCC, f"--offload-arch={build.ARCH}", "-O2", "-std=c++17", "-ffp-contract=off",
                    f"-I{PKG_DIR / 'csrc'}", str(tmp_path / "t.hip"), "-o", str(tmp_path / "t")], check=True,
                   capture_output=True)
    p = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True, timeout=100)
    assert p.returncode == 0, p.stdout
    print(p.stdout)
