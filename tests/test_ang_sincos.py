"""The series sine and cosine of the angular kernel, as written in the kernel source, in a CPU build
against long double (64-bit significand) arithmetic.

With u = 2^-53: the sine is r + E, E = r z a + t w, where r z, a and the sum carry about 5 u |E| of
rounding and E is at most 0.079 at r = pi / 4, next to a result of at least 0.7 in units of u: 0.39 units in
the last place and the final half: 0.89 (below r = 0.52, where the units are half as large, 0.23 more
than the half).  The cosine is w + F with F below 0.016: less.  So 0.9 units bound both.  All
products that a compiler could contract are exact or arguments of fma, so the GPU forms the
same values."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
CLANG = os.path.join(ROCM, "llvm", "bin", "clang++")

DRIVER = r"""
#include <cmath>
#include <cstdio>
#include <cstdlib>
#define __device__
#define __forceinline__ inline
#define __any(x) (x)
%s
static double worst = 0.0, where = 0.0;
static void one(double x) {
    double s, c;
    ang_sincos(x, &s, &c);
    const long double es = sinl((long double)x), ec = cosl((long double)x);
    const long double v[2] = {es, ec};
    const double g[2] = {s, c};
    for (int k = 0; k < 2; ++k) {
        int e;
        (void)frexpl(v[k], &e);  // v in [2^(e-1), 2^e): a unit in the last place is 2^(e-53)
        const double err = (double)fabsl(ldexpl((long double)g[k] - v[k], 53 - e));
        if (!(err <= worst)) worst = err, where = x;
    }
}
int main() {
    srand48(7);
    for (int k = 0; k < 1000000; ++k) one((2.0 * drand48() - 1.0) * 1e5);
    for (int k = 0; k < 1000000; ++k) one((2.0 * drand48() - 1.0) * pow(10.0, 5.0 - 16.0 * drand48()));
    for (long n = -63661; n <= 63661; ++n) {  // next to the multiples of pi / 2 and midway between them
        double x = (double)((long double)n * 1.57079632679489661923132169163975144L);
        for (int d = 0; d < 3; ++d) one(x), x = nextafter(x, 1e9);
        x = ((double)n + 0.5) * 1.57079632679489661923;
        for (int d = 0; d < 3; ++d) one(x), x = nextafter(x, -1e9);
    }
    one(0.0), one(-0.0), one(99999.999), one(-99999.999);
    printf("worst %%.6f at %%.17g\n", worst, where);
    // outside the series' range: the library
    const double big[] = {1e5, -1e5, 1e300, HUGE_VAL, -HUGE_VAL, NAN};
    for (double x : big) {
        double s, c;
        ang_sincos(x, &s, &c);
        const double rs = sin(x), rc = cos(x);
        if (!(s == rs || (s != s && rs != rs)) || !(c == rc || (c != c && rc != rc))) return 1;
    }
    return 0;
}
"""


@pytest.mark.skipif(not os.path.exists(CLANG), reason="ROCm's clang not installed")
def test_series_sine_and_cosine(tmp_path):
    src = open(os.path.join(ROOT, "ggbtddft_amd", "csrc", "ggbtd.hip")).read()
    fn = re.search(r"static __device__ __forceinline__ void ang_sincos\(.*?\n}\n", src, re.S).group(0)
    cpp = tmp_path / "drive.cpp"
    cpp.write_text(DRIVER.replace("%s", fn, 1).replace("%%", "%"))
    exe = tmp_path / "drive"
    r = subprocess.run([CLANG, "-std=c++17", "-O2", "-mfma", "-ffp-contract=off", "-D_GNU_SOURCE", str(cpp), "-o", str(exe),
                        "-lm"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
    assert float(r.stdout.split()[1]) < 0.9, r.stdout
