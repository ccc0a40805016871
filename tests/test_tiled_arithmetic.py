"""Short forms of the tiled 3D kernel's float32 arithmetic, restated in C and
checked against the IEEE operations they stand for (the kernel's own results
are compared bit for bit with the oracle in the GPU tests)."""
import subprocess

import pytest

QUOTIENT = r"""
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <stdint.h>
static float f(uint32_t u) { float x; memcpy(&x, &u, 4); return x; }
static long bad, seen;
static void one(float a, float b, double y)
{
    const float q = (float)((double)a * y);
    if (fpclassify(q) == FP_SUBNORMAL) return;   /* the kernel divides there */
    seen++;
    const float w = a / b;
    if (memcmp(&q, &w, 4)) bad++;
}
int main(int argc, char **argv)
{
    const float b = strtof(argv[1], 0);
    const double y = 1.0 / (double)b;
    /* every numerator whose quotient is subnormal or just above: up to 4 b 2^-126 */
    uint32_t top; float t = 4 * b * 0x1p-126f; memcpy(&top, &t, 4);
    for (uint32_t u = 0; u <= top; u += 1) { one(f(u), b, y); one(-f(u), b, y); }
    /* every significand at three exponents */
    for (int e = 1; e < 255; e += 84)
        for (uint32_t m = 0; m < (1u << 23); m++) one(f(((uint32_t)e << 23) | m), b, y);
    printf("%ld %ld\n", bad, seen);
    return 0;
}
"""

RECIPROCAL = r"""
#include <math.h>
#include <stdio.h>
#include <string.h>
#include <stdint.h>
int main(void)
{
    long bad = 0;
    for (uint32_t m = 0; m < (1u << 23); m++) {
        uint32_t u = (127u << 23) | m; float d; memcpy(&d, &u, 4);
        const double b = d, want = 1.0 / b;
        float est = (float)(1.0 / b);            /* the hardware estimate: within 1 ulp */
        est = nextafterf(nextafterf(est, 0.0f), 0.0f);
        for (int k = 0; k < 5; k++, est = nextafterf(est, 2.0f)) {
            double y = est, r = fma(-b, y, 1.0);
            y = fma(y, r, y); r = fma(-b, y, 1.0); y = fma(y, r, y);
            bad += memcmp(&y, &want, 8) != 0;
        }
    }
    printf("%ld\n", bad);
    return 0;
}
"""


def _run(tmp_path, text, *args):
    src, exe = tmp_path / "c.c", tmp_path / "c"
    src.write_text(text)
    subprocess.run(["gcc", "-O2", "-mfma", "-ffp-contract=off", "-o", str(exe), str(src), "-lm"],
                   check=True)
    return [int(x) for x in subprocess.run([str(exe), *args], capture_output=True, text=True,
                                           check=True, timeout=600).stdout.split()]


@pytest.mark.parametrize("b", ["100", "400", "6", "156.25"])
def test_f64_product_is_the_quotient_unless_subnormal(tmp_path, b):
    """RN32(a RN64(1/b)) that is not subnormal is the IEEE quotient a/b for
    divisors with even factors too (h = 10 m: 100, and 400 = 4 h2)."""
    bad, seen = _run(tmp_path, QUOTIENT, b)
    assert bad == 0 and seen > 0


def test_two_newton_steps_give_the_rounded_reciprocal(tmp_path):
    """recip_f64 for every float significand and every estimate within two
    units in the last place."""
    with open("/proc/cpuinfo") as f:
        if "fma" not in f.read():
            pytest.skip("no fused multiply-add on this CPU")
    assert _run(tmp_path, RECIPROCAL) == [0]
