"""The bound on the columns under a block of windows (csrc/owm_axis.h), by which the
host sizes the windows' LDS, against the blocks of random axes, far ones among them."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))

SOURCE = """
#include <algorithm>
#include <cstdio>
#include <random>
#include "%s/owm_axis.h"
static double round2d(double z) { return std::round(z * 100.0) / 100.0; }
int main()
{
    std::mt19937_64 r(1);
    auto uni = [&](double a, double b) { return a + (b - a) * (double)(r() >> 11) * 0x1p-53; };
    long axes = 0, far = 0, refused = 0, bad = 0;
    for (double mag : {1e2, 1e4, 1e6, 1e8, 1e10, 1e11, 1e12, 3e12, 1e13, 1e17})
        for (int it = 0; it < 4000; ++it) {
            const int W = 1 + (int)(r() %% 20), B = (int)(r() %% 25), h = W / 2, hb = B / 2;
            const double some[] = {0, 0.5, 0.8, 0.9};
            const double O = r() %% 2 ? uni(0, 0.95) : some[r() %% 4], minx = uni(0.5, 1) * mag;
            const double width = round2d((minx + uni(1, 400)) - minx), D = round2d(W * (1 - O));
            if (!(width > 0) || !(D > 0))
                continue;
            const double c = O > 0 ? std::round((width + 2 * W * O) / D) - 1 : std::floor(width / W) + 1;
            if (!(c >= 1 && c <= 65535))
                continue;
            const uint32_t n = (uint32_t)c;
            GridAxis A;
            grid_edges(A.w, minx - h + D, D, (double)(float)h, n, false, 64);
            grid_edges(A.g, minx + hb, B ? B : 1, (double)(float)hb, B ? (uint32_t)(std::floor(width / B) + 1) : 0,
                       true, 1);
            grid_axis(A);
            if (A.w.tol > 0.125 || A.g.tol > 0.125) {
                ++refused;
                continue;
            }
            ++axes;
            far += mag >= 1e11;
            for (uint32_t bw : {8u, 16u, 32u})
                for (uint32_t i = 0; i < n; i += bw) {
                    int a, b, c, d;
                    axis_window_cols(A, i, a, b);
                    axis_window_cols(A, std::min(n, i + bw) - 1, c, d);
                    bad += d - a + 1 > axis_cols_of(A, bw);
                }
        }
    std::printf("%%ld %%ld %%ld %%ld\\n", axes, far, refused, bad);
}
"""


def test_bound(tmp_path):
    src, exe = str(tmp_path / "cols.cpp"), str(tmp_path / "cols")
    with open(src, "w") as f:
        f.write(SOURCE % os.path.join(os.path.dirname(HERE), "fastowm_amd", "csrc"))
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-o", exe, src], check=True)
    axes, far, refused, bad = map(int, subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split())
    assert bad == 0 and axes > 20_000 and far > 3000 and refused > 3000
