"""The fp8 page writer's quotient (csrc/kernels/fp8_page.hpp, fp8_quotient): a
product with the reciprocal and one residual step, r = 1 / scale,

    q = x * r;  copysign(fma(fma(-q, scale, x), r, q), x) clamped to +-448,

gives the e4m3 code of x / scale for the inputs of both its callers and the
scales for which the header uses it:

  rows written:   x any finite bf16 with |x| <= amax, scale >= amax / 448;
  rows re-encoded: x = (value of any code) * old in fp32, old any positive
                  float below scale.

Restated in C (fmaf and division are the IEEE operations there), swept on the
CPU; the kernel's own bytes are compared in test_gpu_kv_write.py."""
import re
import subprocess
from pathlib import Path

HEADER = Path(__file__).resolve().parent.parent / "lattice_amd/csrc/kernels/fp8_page.hpp"

SOURCE = r"""
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

static float f32(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
static uint32_t bits(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
static uint64_t state = 88172645463325252ull;
static uint64_t rnd(void) { state ^= state << 13; state ^= state >> 7; state ^= state << 17; return state; }

/* e4m3 code of f, round to nearest even, saturating */
static uint32_t encode(float f) {
    const uint32_t sign = bits(f) >> 24 & 0x80u;
    const float a = fabsf(f);
    if (a >= 448.0f) return sign | 0x7e;
    if (a < 0.015625f) return sign | (uint32_t)rintf(a * 512.0f);
    uint32_t u = bits(a);
    u += 0x7ffff + (u >> 20 & 1);
    return sign | ((u >> 20) - (120u << 3));
}
static float decode(uint32_t c) {
    const uint32_t e = c >> 3 & 15, m = c & 7;
    const float a = e ? ldexpf(8 + m, (int)e - 10) : ldexpf(m, -9);
    return c & 0x80 ? -a : a;
}
static float quotient(float x, float scale, float r) {
    const float q = x * r;
    return fminf(fmaxf(copysignf(fmaf(fmaf(-q, scale, x), r, q), x), -448.0f), 448.0f);
}
static long bad, done;
static void check(float x, float scale, float r) {
    ++done;
    if (encode(quotient(x, scale, r)) != encode(x / scale) && ++bad < 10)
        printf("x %a scale %a: %a, x / scale %a\n", x, scale, quotient(x, scale, r), x / scale);
}
/* a positive float with an exponent of lo .. hi */
static float any(int lo, int hi) {
    return f32((uint32_t)(127 + lo + (int)(rnd() % (uint64_t)(hi - lo + 1))) << 23 | (rnd() & 0x7fffff));
}
static void rows(float scale) {
    const float r = 1.0f / scale;
    for (uint32_t h = 0; h < 0x7f80; ++h) {
        const float x = f32(h << 16);
        if (x / 448.0f > scale) break;      /* |x| <= amax, scale >= amax / 448 */
        check(x, scale, r);
        check(-x, scale, r);
    }
}
static void codes(float old, float scale) {
    const float r = 1.0f / scale;
    if (!(old < scale)) return;
    for (uint32_t c = 0; c < 256; ++c)
        if ((c & 0x7f) != 0x7f) check(decode(c) * old, scale, r);
}
int main(void) {
    const float lo = LO, hi = HI;
    for (uint32_t c = 0; c < 256; ++c)
        if ((c & 0x7f) != 0x7f && encode(decode(c)) != c) return printf("code %u\n", c), 1;
    /* rows: every bf16 amax's scale in the range, then any */
    for (uint32_t h = 1; h < 0x7f80; h += 23) {
        const float s = f32(h << 16) / 448.0f;
        if (s >= lo && s <= hi) rows(s);
    }
    for (int i = 0; i < 300; ++i) rows(any(ilogbf(lo), ilogbf(hi) - 1));
    for (uint32_t d = 0; d < 40; ++d) {
        rows(f32(bits(lo) + d));
        rows(f32(bits(hi) - d));
        rows(f32((127u << 23) + d));
        rows(f32((127u << 23) - d));
    }
    /* codes: old over the whole range, near the scale, and subnormal */
    for (int i = 0; i < 60000; ++i) {
        const float s = i % 8 ? any(ilogbf(lo), ilogbf(hi) - 1) : f32(i % 16 ? bits(lo) + i / 16 : bits(hi) - i / 16);
        codes(any(-126, 99), s);
        codes(f32(bits(s) - 1 - rnd() % 64), s);
        codes(s * (float)(rnd() % 4096) / 4096.0f, s);
        codes(ldexpf(s, -(int)(rnd() % 24)), s);
        codes(f32(1 + rnd() % 0x7fffff), s);
    }
    printf("%ld of %ld differ\n", bad, done);
    return bad != 0;
}
"""


def test_quotient_gives_the_code_of_the_division(tmp_path):
    src = tmp_path / "quotient.c"
    lo, hi = re.search(r"kFp8QuotientMin = (\S+), kFp8QuotientMax = (\S+);",
                       HEADER.read_text()).groups()
    src.write_text(SOURCE.replace("LO", lo).replace("HI", hi))
    exe = tmp_path / "quotient"
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", "-o", str(exe), str(src), "-lm"], check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert p.returncode == 0, p.stdout
    print(p.stdout)
