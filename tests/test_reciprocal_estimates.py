"""The sequences of snac_amd/csrc/snh_math.h that the GPU runs from its
hardware estimates, on the CPU from estimates off by up to 2^-23: root,
reciprocal and quotients against sqrt and the division, with mantissas at
random, of few bits, and next to one, 3/2 and two, where reciprocals and
quotients come closest to rounding midpoints; either sign of the divisor, and
the ends of the stated range.  And the bound on the root of the yield test,
which takes the estimate itself."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <stdint.h>
#include <stdio.h>
#include <string.h>
#include "snh_math.h"
static uint64_t st = 2024;
static uint64_t rnd(void) {
    st += 0x9E3779B97F4A7C15ull;
    uint64_t z = st;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
static double uni(void) { return (double)(rnd() >> 11) * 0x1p-53; }
static double make(unsigned kind, int exponent) {
    uint64_t m;
    switch (kind % 5) {
    case 0: m = rnd() >> 12; break;
    case 1: m = rnd() % 64; break;
    case 2: m = 0xFFFFFFFFFFFFFull - rnd() % 64; break;
    case 3: m = 0x7FFFFFFFFFFC0ull + rnd() % 128; break;
    default: m = (rnd() >> 12) & ~((1ull << (rnd() % 52)) - 1);
    }
    const uint64_t u = ((uint64_t)(1023 + exponent) << 52) | m;
    double d;
    memcpy(&d, &u, 8);
    return d;
}
static int within(int n) { return (int)(rnd() % (unsigned)(2 * n + 1)) - n; }
static int is_pow2(double a) { int e; return frexp(fabs(a), &e) == 0.5; }
static int all_ones(double b) { int e; return frexp(fabs(b), &e) == 1.0 - 0x1p-53; }
static double estimate(double exact) { return exact * (1.0 + (uni() - 0.5) * 0x1p-22); }
int main(void) {
    long root = 0, recip = 0, faithful = 0, quot = 0, quot_root = 0, bound = 0;
    for (int i = 0; i < 3000000; i++) {
        const double a = make((unsigned)rnd(), within(40)) * (rnd() & 1 ? 1.0 : -1.0);
        const double b = make((unsigned)i, within(i & 8 ? 60 : 400)) * (rnd() & 1 ? 1.0 : -1.0), x = fabs(b);
        const snh_recip r = snh_recip_refine(b, estimate(1.0 / b));
        recip += snh_recip_rn(r) != 1.0 / b;
        faithful += fabs(r.hi - 1.0 / b) > fabs(1.0 / b) * 0x1p-52;
        /* 2^n over the largest number below a power of two is the known exception */
        if (!(is_pow2(a) && all_ones(b))) quot += snh_quot(a, r) != a / b;
        snh_recip rs;
        const double s = snh_sqrt_refine(x, estimate(1.0 / sqrt(x)), &rs);
        root += s != sqrt(x);
        recip += snh_recip_rn(rs) != 1.0 / sqrt(x);
        if (!(is_pow2(a) && all_ones(sqrt(x)))) quot_root += snh_quot(a, rs) != a / sqrt(x);
        /* q rsq(q) (1 + 1e-6) is not below the root */
        bound += x * estimate(1.0 / sqrt(x)) * (1.0 + 1e-6) < sqrt(x);
    }
    for (int k = 1; k < 200000; k++) {   /* every divisor just below a power of two */
        const double b = 2.0 - k * 0x1p-52;
        recip += snh_recip_rn(snh_recip_refine(b, estimate(1.0 / b))) != 1.0 / b;
    }
    const double ends[] = {0x1p-918, 0x1.fffffffffffffp-918, 0x1.5p-917, 0x1p1022, 0x1.fffffffffffffp1021, 0x1.7p1022};
    for (int k = 0; k < 6; k++) {
        snh_recip rs;
        root += snh_sqrt_refine(ends[k], estimate(1.0 / sqrt(ends[k])), &rs) != sqrt(ends[k]);
        recip += snh_recip_rn(rs) != 1.0 / sqrt(ends[k]);
    }
    printf("%ld %ld %ld %ld %ld %ld\n", root, recip, faithful, quot, quot_root, bound);
    return 0;
}
"""


def test_refined_estimates_equal_sqrt_and_division(tmp_path):
    src, exe = tmp_path / "r.c", tmp_path / "r"
    src.write_text(SRC)
    subprocess.check_call(["gcc", "-O2", "-ffp-contract=off", "-I", os.path.join(ROOT, "snac_amd", "csrc"), "-o",
                           str(exe), str(src), "-lm"])
    assert subprocess.check_output([str(exe)]).split() == [b"0"] * 6
