"""The branch-free logf and sinf of the Box-Muller transform (logf_unit and
sinf_turn of nemo_amd/csrc/glibc_math.h) against the host C library, bit for
bit: logf over 0 and every float in [2^-24, 1], which holds every 1 - b the
transform forms, and sinf over every float in [0, 8)."""
import os
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <math.h>
#include <stdio.h>
#include "glibc_math.h"
using namespace nemo_math;
int main() {
    auto entry = [](unsigned i, double* a, double* b) { *a = logf_invc(i); *b = logf_logc(i); };
    long bad_log = asuint(logf_unit(0.0f, entry)) != asuint(logf(0.0f)), bad_sin = 0;
    #pragma omp parallel for reduction(+:bad_log)
    for (long u = 0x33800000; u <= 0x3f800000; ++u) {
        const float x = asfloat((uint32_t)u);
        if (asuint(logf_unit(x, entry)) != asuint(logf(x))) ++bad_log;
    }
    #pragma omp parallel for reduction(+:bad_sin)
    for (long u = 0; u < 0x41000000; ++u) {
        const float x = asfloat((uint32_t)u);
        if (asuint(sinf_turn(x)) != asuint(sinf(x))) ++bad_sin;
    }
    /* the extremes of 1 - b and of the angle */
    const float top = (float)0xffffffffu;
    const bool range = 1.0f - top * 0.00000000023283064365386962890625f >= 0.0f
        && top * 1.4629180792671596810513378043098e-9f < 8.0f;
    printf("%ld %ld %d\n", bad_log, bad_sin, (int)range);
    return 0;
}
"""


def test_branch_free_logf_and_sinf_match_the_c_library():
    with tempfile.TemporaryDirectory() as d:
        src, exe = os.path.join(d, "t.cpp"), os.path.join(d, "t")
        with open(src, "w") as f:
            f.write(PROGRAM)
        subprocess.run(["g++", "-O2", "-std=c++17", "-fopenmp", "-ffp-contract=off", "-mfma",
                        "-I" + os.path.join(ROOT, "nemo_amd", "csrc"), src, "-o", exe, "-lm"], check=True)
        out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split()
    assert out == ["0", "0", "1"]
