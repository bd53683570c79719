// Columns of owm_axis.h against direct compares: for random and edge
// coordinates of random window and cell grids, the fast column equals the exact
// one, a point's window and cell ranges are those whose open intervals hold it,
// and a point with a column lies in exactly the windows and cells that list the
// column.  Prints the counts; exits 1 on any difference.
#include <cstdio>
#include <random>
#include <vector>

#include "../fastowm_amd/csrc/owm_axis.h"

static double round2d(double z) { return std::round(z * 100.0) / 100.0; }

int main()
{
    std::mt19937_64 r(1);
    long bad = 0, points = 0, slow = 0, none = 0, pairs = 0;
    auto uni = [&](double a, double b) { return a + (b - a) * (double)(r() >> 11) * 0x1p-53; };
    for (int it = 0; it < 4000; ++it) {
        const int W = it % 5 == 0 ? 1 + (int)(r() % 8) : 5 + (int)(r() % 16);
        const double ov[] = {0, 0.5, 0.6, 0.75, 0.8, 0.9, 0.7, uni(0, 0.95)};
        const double O = ov[r() % 8], width = round2d(uni(1, 60 + W * 4));
        const int B = it % 7 == 0 ? (int)(r() % 6) : 10 + (int)(r() % 21);
        const double mins[] = {0, 512000.0, 4700000.12, -1234.56, uni(-10, 10), 1e9 + 0.25, -4e6};
        const double minx = mins[r() % 7], D = round2d(W * (1 - O));
        const double c = O > 0 ? std::round((width + 2 * W * O) / D) - 1 : std::floor(width / W) + 1;
        if (!(D > 0) || c < 1)
            continue;
        const uint32_t n = (uint32_t)c, ng = B ? (uint32_t)(std::floor(width / B) + 1) : 0;
        const int h = W / 2, hb = B / 2;
        GridAxis A;
        grid_edges(A.w, minx - h + D, D, (double)(float)h, n, false, 32);
        grid_edges(A.g, minx + hb, B ? B : 1, (double)(float)hb, ng, true, 1);
        grid_axis(A);
        pairs += A.w.pair != 0;
        std::vector<double> L, R, GL, GR, all;
        for (uint32_t i = 0; i < n; ++i) {
            const double m = (minx - h + D) + (double)(int)i * D;
            L.push_back(m - h), R.push_back(m + h);
        }
        for (uint32_t i = 0; i < ng; ++i) {
            const double m = (minx + hb) + (double)(int)(i * B);
            GL.push_back(m - hb), GR.push_back(m + hb);
        }
        for (auto *v : {&L, &R, &GL, &GR})
            all.insert(all.end(), v->begin(), v->end());
        std::vector<int> w0(n), w1(n), g0(ng), g1(ng);
        for (uint32_t i = 0; i < n; ++i)
            axis_window_cols(A, i, w0[i], w1[i]);
        for (uint32_t i = 0; i < ng; ++i)
            axis_cell_cols(A, i, g0[i], g1[i]);
        auto check = [&](double x) {
            uint32_t col, fast;
            const AxisPassed p = axis_passed(A, x);
            const bool ok = axis_col_exact(A, p, col), f = axis_col_fast(A, x, fast);
            ++points, slow += !f, none += !ok;
            bad += col >= A.ncol || fast >= A.ncol || (f && (!ok || fast != col));
            for (uint32_t i = 0; i < n; ++i) {
                const bool in = L[i] < x && x < R[i];
                bad += (i >= p.w_lo && i < p.w_hi) != in;
                bad += ok && ((int)col >= w0[i] && (int)col <= w1[i]) != in;
            }
            for (uint32_t i = 0; i < ng; ++i) {
                const bool in = GL[i] < x && x < GR[i];
                bad += (i >= p.g_lo && i < p.g_hi) != in;
                bad += ok && ((int)col >= g0[i] && (int)col <= g1[i]) != in;
            }
        };
        for (int k = 0; k < 60; ++k) {
            check(uni(minx - 3 * W, minx + width + 3 * W));
            check(round2d(uni(minx - W, minx + width + W)));
        }
        for (double e : all) {
            if (all.size() >= 60 && r() % 3)
                continue;
            double a = e, b = e;
            check(e);
            for (int k = 0; k < 3; ++k) {
                check(a = std::nextafter(a, 1e300));
                check(b = std::nextafter(b, -1e300));
            }
            check(e + 1e-9), check(e - 1e-9), check(e + 1e-6);
        }
        for (double x : {(double)NAN, (double)INFINITY, -(double)INFINITY, 1e300, -1e300, 0.0, -0.0})
            check(x);
    }
    std::printf("points %ld slow %ld without column %ld paired grids %ld bad %ld\n", points, slow, none,
                pairs, bad);
    return bad != 0;
}
