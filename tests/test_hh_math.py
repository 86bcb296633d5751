"""The shortened forms of the HH substeps (nemo_amd/csrc/plugins/HH.hip)
against the host C library, at every float they can meet: expf without its
special cases on [-104, 89], and the exponents -y / c as a product with 1 / c
in two floats, through expf, for |y| <= 256."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <math.h>
#include <stdio.h>
#include <stdint.h>
#include <string.h>
#include "glibc_math.h"
using namespace nemo_math;
static uint32_t bits(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
int main() {
    uint64_t tab[32 * EXPF_REPEATS];
    for (unsigned i = 0; i < 32 * EXPF_REPEATS; i++) tab[i] = expf_table(i);
    long bad_exp = 0, n_exp = 0, bad_div = 0, n_div = 0;
    const float cs[] = {18.0f, 20.0f, 80.0f};
    #pragma omp parallel for reduction(+:bad_exp, n_exp, bad_div, n_div) schedule(dynamic, 1 << 20)
    for (int64_t u = 0; u < (int64_t(1) << 32); u += 1) {
        uint32_t w = (uint32_t)u;
        float x; memcpy(&x, &w, 4);
        if (x >= -104.0f && x <= 89.0f) { n_exp++; if (bits(expf(x)) != bits(expf_main_tab(x, tab))) bad_exp++; }
        if (!(fabsf(x) <= 256.0f)) continue;
        for (float c : cs) {
            const float inv = 1.0f / c, rest = float(1.0 / double(c) - double(inv));
            const float q = __builtin_fmaf(-inv, x, 0.0f - rest * x), a = -x / c;
            n_div++;
            if (bits(q) != bits(a) && bits(expf(q)) != bits(expf(a))) bad_div++;
        }
    }
    printf("%ld %ld %ld %ld\n", bad_exp, n_exp, bad_div, n_div);
    return 0;
}
"""


def test_every_float(tmp_path):
    src, exe = tmp_path / "m.cpp", tmp_path / "m"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-mfma", "-fopenmp", "-std=c++17", "-ffp-contract=off",
                    "-I" + os.path.join(ROOT, "nemo_amd", "csrc"), str(src), "-o", str(exe), "-lm"], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()
    bad_exp, n_exp, bad_div, n_div = map(int, out)
    assert n_exp > 2e9 and n_div > 6e9
    assert bad_exp == 0 and bad_div == 0
