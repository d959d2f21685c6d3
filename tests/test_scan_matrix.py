"""The candidate scan's matrix-core distances (ivp_grid.hip, seg_pop_scan): e = |b|^2 - 2 a.b +
(|a|^2 - h^2) in float32 about a segment's centre, decided by its sign outside |e| < 2^-14 h^2 and
by the reference's own test inside.

The bound that the band rests on, by a C restatement: for coordinates within 4 h of the centre
and pairs a few 10^-4 around the support radius, every order of the four products' sum (fused
or rounded one by one) stays within 2^-15 h^2, half the band, of the exact value, and the decision
equals sqrtf(d^2) < h on the unfused d^2.  Without the band it does not.
"""

import shutil
import subprocess

import pytest

SRC = r"""
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
static uint64_t s = 88172645463325252ull;
static inline uint64_t nx(void) { s ^= s << 13; s ^= s >> 7; s ^= s << 17; return s; }
static inline double u01(void) { return (nx() >> 11) * (1.0 / 9007199254740992.0); }
int main(int argc, char** argv) {
    long N = atol(argv[1]), bad = 0, bare = 0, band = 0, inside = 0;
    double worst = 0.0;
    for (long t = 0; t < N; ++t) {
        float h = (float)(0.003 + 0.3 * u01());
        if (t % 7 == 0) h = 0.02f; else if (t % 7 == 1) h = 0.04f; else if (t % 7 == 2) h = 0.01f;
        const float h2 = (float)((double)h * (double)h), far2 = 16.0f * h2, eps = h2 * (1.0f / 16384.0f);
        float o[3], xi[3], xj[3];
        double z = 2 * u01() - 1, ph = 6.283185307179586 * u01(), q = sqrt(1 - z * z);
        double R = h * (1.0 + 4e-4 * (u01() - 0.5));
        double dir[3] = {R * q * cos(ph), R * q * sin(ph), R * z};
        for (int c = 0; c < 3; ++c) {
            o[c] = (float)(4.0 * u01());
            xi[c] = (float)(o[c] + 2.4 * h * (2 * u01() - 1));
            xj[c] = (float)(xi[c] - dir[c]);
        }
        float a[3], b[3], r[3];
        for (int c = 0; c < 3; ++c) { a[c] = xi[c] - o[c]; b[c] = xj[c] - o[c]; r[c] = xi[c] - xj[c]; }
        const float a2 = fmaf(a[2], a[2], fmaf(a[1], a[1], a[0] * a[0]));
        const float b2 = fmaf(b[2], b[2], fmaf(b[1], b[1], b[0] * b[0]));
        if (!(a2 <= far2) || !(b2 <= far2)) continue;      /* the exact test throughout */
        const int ref = sqrtf(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]) < h;
        double d2 = 0.0;
        for (int c = 0; c < 3; ++c) { double w = (double)xi[c] - (double)xj[c]; d2 += w * w; }
        const float c0 = a2 - h2;
        const float p[4] = {b[0] * (-2.0f * a[0]), b[1] * (-2.0f * a[1]), b[2] * (-2.0f * a[2]), b2};
        float e[4];
        e[0] = fmaf(b2, 1.0f, fmaf(b[2], -2.0f * a[2], fmaf(b[1], -2.0f * a[1], fmaf(b[0], -2.0f * a[0], c0))));
        e[1] = fmaf(b[0], -2.0f * a[0], fmaf(b[1], -2.0f * a[1], fmaf(b[2], -2.0f * a[2], b2 + c0)));
        e[2] = c0 + ((p[0] + p[1]) + (p[2] + p[3]));
        e[3] = (((c0 + p[0]) + p[1]) + p[2]) + p[3];
        for (int k = 0; k < 4; ++k) {
            const double err = fabs((double)e[k] - (d2 - (double)h * (double)h)) / ((double)h * h);
            if (err > worst) worst = err;
            const int near = fabsf(e[k]) < eps;
            band += near;
            bad += (near ? ref : e[k] < 0.0f) != ref;
            bare += (e[k] < 0.0f) != ref;
        }
        inside += ref;
    }
    printf("%ld %ld %ld %ld %.17g\n", inside, band, bad, bare, worst);
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("gcc") is None, reason="gcc not available")
def test_matrix_distances_decide_outside_the_band(tmp_path):
    src, exe = tmp_path / "m.c", tmp_path / "m"
    src.write_text(SRC)
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", "-o", str(exe), str(src), "-lm"], check=True)
    n = 10_000_000
    out = subprocess.run([str(exe), str(n)], check=True, capture_output=True, text=True).stdout.split()
    inside, band, bad, bare = (int(v) for v in out[:4])
    assert float(out[4]) < 2.0 ** -15       # half the band
    assert bad == 0
    assert bare > 0 and band > n // 20      # the band is needed, and reached
    assert 0.3 * n < inside < 0.6 * n
