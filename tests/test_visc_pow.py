"""The FP64 viscosity law's power T^n (visc_pow, visc_pow2 of cns_device.hpp),
compiled for the CPU with the emulation header and compared with long double
powl: at most 2 ulp where |n log2 T| <= 1 and 1 ulp more per further unit
(the rounding of the exponent n log2 T, which exp2(n log2 T) has as well),
over T in [0.05, 20], near 1 and at the ends of the mantissa's range; and the
values of exp2(n log2 T) where T is no positive finite number."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include "hip/hip_runtime.h"
#include "cns_device.hpp"
#include <cstdio>
#include <limits>
static long bad = 0;
static void one(double t, double n) {
    const long double ref = powl((long double)t, (long double)n);
    const double ulp = std::nextafter((double)ref, 1e300) - (double)ref;
    const double bound = 2.0 + std::fmax(0.0, std::fabs(n * std::log2(t)) - 1.0);
    double p, q;
    cns::visc_pow2(t, 1.0, n, p, q);
    const double v = cns::visc_pow(t, n), e = (double)fabsl(v - ref) / ulp;
    if (!(e <= bound) || p != v || q != 1.0) {
        if (bad++ < 5) std::printf("T %.17g n %g: %.17g, %.2f ulp (bound %.2f), pair %.17g %.17g\n", t, n, v, e, bound, p, q);
    }
}
int main() {
    const double ns[] = {0.5, 0.666, 0.7, 0.76, 1.0, 1.3, 1.5, 2.0, -0.5};
    const double mid = 0.70710678118654752440;
    for (double n : ns) {
        for (int i = 0; i <= 200000; i++) one(std::exp(-3.0 + 6.0 * i / 200000.0), n);
        for (int i = -20000; i <= 20000; i++) one(1.0 + i * 1e-9, n);
        for (double b : {mid, 2.0 * mid, 0.5, 1.0, 2.0, 4.0})
            for (int i = -50; i <= 50; i++) one(b * (1.0 + i * 1.2e-16), n);
    }
    const double inf = std::numeric_limits<double>::infinity(), nan = std::numeric_limits<double>::quiet_NaN();
    for (double t : {0.0, -0.0, -1.0, inf, -inf, nan})
        for (double n : {0.7, -0.7, 0.0}) {
            const double v = cns::visc_pow(t, n), w = exp2(n * log2(t));
            double p, q;
            cns::visc_pow2(t, 1.25, n, p, q);
            if (!(v == w || (std::isnan(v) && std::isnan(w))) || !(p == w || (std::isnan(p) && std::isnan(w)))) {
                bad++;
                std::printf("T %g n %g: %g, %g (expected %g)\n", t, n, v, p, w);
            }
        }
    for (double t : {5e-324, 1e-310, 1.7e308}) one(t, 0.001);
    std::printf("%ld bad\n", bad);
    return bad != 0;
}
"""


def test_visc_pow_against_powl(tmp_path):
    src, exe = tmp_path / "vp.cpp", tmp_path / "vp"
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++20", "-O2", "-pthread", "-I", os.path.join(ROOT, "tests", "emu"), "-I",
                    os.path.join(ROOT, "cudanavierstokes_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
