"""Forms of esth_math.h that stand in for one another give the same bits
(compiled as the host compiles them, no floating-point contraction)."""
import os
import subprocess

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <stdio.h>
#include "esth_math.h"
static const float edge[] = {0.0f, -0.0f, 1e-45f, -1e-45f, 1e-38f, -3e-39f, 9.9e-31f, 1e-30f, -1e-30f, 1.1e-30f, 1e-22f,
                             1e-10f, 0.02f, -0.5f, 1.0f, -1.0f, 3.0f, 70.0f, -70.0f, 1e10f, 1e19f, -1e30f, INFINITY,
                             -INFINITY, NAN};
enum { N = sizeof(edge) / sizeof(edge[0]) };
int main(void) {
    /* esth_polar_floor for esth_polar_abs in (z - r)^2 added to an accumulator, and the angle itself */
    long bad = 0;
    for (int i = 0; i < N; ++i)
        for (int j = 0; j < N; ++j) {
            float r, a, rf, af;
            esth_polar_abs(edge[i], edge[j], &r, &a);
            esth_polar_floor(edge[i], edge[j], &rf, &af);
            if (esth_f2u(a) != esth_f2u(af) && !(a != a && af != af)) ++bad;
            for (int k = 0; k < N; ++k)
                for (int l = 0; l < N; ++l) {
                    const float acc = fabsf(edge[l]);
                    const float x = esth_fma(edge[k] - r, edge[k] - r, acc), y = esth_fma(edge[k] - rf, edge[k] - rf, acc);
                    if (esth_f2u(x) != esth_f2u(y) && !(x != x && y != y)) ++bad;
                }
        }
    printf("%ld\n", bad);
    return 0;
}
"""


def test_polar_floor_in_a_squared_residual(tmp_path):
    src, exe = tmp_path / "forms.c", tmp_path / "forms"
    src.write_text(SOURCE)
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", "-I", os.path.join(REPO, "esthera_amd", "csrc"), str(src), "-lm",
                    "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.strip() == "0"
