"""snh_math.h's reciprocal pairs and scaled divisions by three against the
division, on the CPU: quotients by a pair refined from an estimate as coarse
as the GPU's (2^-23), the scaled div3 forms, and the root of the host form."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <stdint.h>
#include <stdio.h>
#include "snh_math.h"
static uint64_t st = 12345;
static uint64_t rnd(void) {
    st += 0x9E3779B97F4A7C15ull;
    uint64_t z = st;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
static double uni(void) { return (double)(rnd() >> 11) * 0x1p-53; }
static double val(int range) {
    return ldexp(1.0 + uni(), (int)(rnd() % (unsigned)(2 * range + 1)) - range) * ((rnd() & 1) ? 1.0 : -1.0);
}
int main(void) {
    long bad = 0;
    for (int i = 0; i < 2000000; i++) {
        const double a = val(40), b = fabs(val(60));
        /* an estimate off by up to 2^-23, one Newton step, then the pair */
        double y = (1.0 / b) * (1.0 + (uni() - 0.5) * 0x1p-22);
        y = fma(fma(-b, y, 1.0), y, y);
        const snh_recip r = snh_recip_of(b, y);
        bad += snh_quot(a, r) != a / b;
        bad += r.hi != 1.0 / b;
        snh_recip rs;
        const double s = snh_sqrt_recip(b, &rs);
        bad += s != sqrt(b) || snh_quot(a, rs) != a / sqrt(b);
        bad += snh_div3(a) != a / 3.0 || snh_div6(a) != a / 6.0 || snh_div12(a) != a / 12.0;
        bad += snh_ndiv6(a) != -a / 6.0 || snh_ndiv12(a) != -a / 12.0;
    }
    printf("%ld\n", bad);
    return 0;
}
"""


def test_quotients_equal_the_division(tmp_path):
    src, exe = tmp_path / "q.c", tmp_path / "q"
    src.write_text(SRC)
    subprocess.check_call(["gcc", "-O2", "-ffp-contract=off", "-I", os.path.join(ROOT, "snac_amd", "csrc"), "-o",
                           str(exe), str(src), "-lm"])
    assert int(subprocess.check_output([str(exe)])) == 0
