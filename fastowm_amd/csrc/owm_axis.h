// One axis of a tile's column grid: the exact partition of a coordinate axis by
// every edge of stage 1's windows and of stage 3's cells (plain C++, used by the
// device kernels and by the CPU test).
//
// Edges, in the reference's arithmetic (src/optim3_func.cpp:541-561, 627-662,
// makeBox): window i is the open interval (L_i, R_i), cell k the open interval
// (GL_k, GR_k).  A coordinate x has "passed" L and GL edges when e < x and R
// and GR edges when e <= x, so the windows holding x are exactly
// [#R passed, #L passed) and the cells [#GR passed, #GL passed), and the number
// of passed edges is monotone in x.  Points with equal passed counts lie in
// the same windows and cells: they share a column, numbered by the count.
//
// Two edges that coincide up to rounding would leave an (almost) empty column
// between them, so such pairs count once: when the window side is m steps,
// L_j and R_{j-m} form the pair E_j (E_j = R_{j-m} alone for j >= n), and when
// Bsize is even, GL_k and GR_{k-1} form the pair GE_k.  A coordinate that has
// passed one edge of a pair and not the other (it lies on or within rounding of
// both) has no column; axis_col_exact says so and the caller takes its
// window and cell ranges from axis_passed.
#pragma once
#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#endif
#include <math.h>
#include <stdint.h>

#ifdef __HIPCC__
#define OWM_HD __host__ __device__ __forceinline__
#else
#define OWM_HD inline
#endif

// n intervals centred at fl(init + fl(i * step)) with half side `half`
// (rounded per operation; compiled without fused multiply-add).
struct GridEdges {
    double init, step, inv, half;
    double e0, cr;  // first left edge; right edges' offset (R_0 - L_0) / step
    double tol;     // estimates this close to a whole number are not trusted
    uint32_t n;
    // windows: m when every R_i pairs with L_{i+m}, else 0; cells: 1 when every
    // GR_k pairs with GL_{k+1}, else 0
    uint32_t pair;
};

struct GridAxis {
    GridEdges w, g;  // windows, stage-3 cells (g.n == 0: none)
    uint32_t ncol;   // columns
    uint32_t pad;
};

OWM_HD double axis_edge(const GridEdges &E, int i, bool right)
{
    const double c = E.init + (double)i * E.step;
    return right ? c + E.half : c - E.half;
}

// Edges of one side passed by v: e < v, or e <= v with `equal`.  The estimate
// is off by rounding only, so the walk ends after a step or two.
OWM_HD uint32_t axis_count(const GridEdges &E, double v, bool right, bool equal)
{
    const int n = (int)E.n;
    const double f = (v - E.e0) * E.inv - (right ? E.cr : 0.0);
    int k = f >= 0.0 ? (f < (double)n ? (int)f + 1 : n) : 0;
    for (;;) {
        const double e = k > 0 ? axis_edge(E, k - 1, right) : 0.0;
        if (k > 0 && !(e < v || (equal && e == v)))
            --k;
        else
            break;
    }
    for (;;) {
        const double e = k < n ? axis_edge(E, k, right) : 0.0;
        if (k < n && (e < v || (equal && e == v)))
            ++k;
        else
            break;
    }
    return (uint32_t)k;
}

struct AxisPassed {
    uint32_t w_lo, w_hi;  // windows [w_lo, w_hi) hold x
    uint32_t g_lo, g_hi;  // cells [g_lo, g_hi) hold x
};

OWM_HD AxisPassed axis_passed(const GridAxis &A, double x)
{
    AxisPassed p;
    p.w_hi = axis_count(A.w, x, false, false);
    p.w_lo = axis_count(A.w, x, true, true);
    p.g_hi = A.g.n ? axis_count(A.g, x, false, false) : 0u;
    p.g_lo = A.g.n ? axis_count(A.g, x, true, true) : 0u;
    return p;
}

// The column of a coordinate with these passed counts; false when it has
// none (col is then that of a neighbouring column).
OWM_HD bool axis_col_exact(const GridAxis &A, const AxisPassed &p, uint32_t &col)
{
    bool ok = true;
    if (A.w.pair) {
        const uint32_t n = A.w.n, m = A.w.pair;  // m <= n
        const uint32_t c = p.w_hi < n ? p.w_hi : (p.w_lo + m > n ? p.w_lo + m : n);
        ok = p.w_lo == (c > m ? c - m : 0u);
        col = c;
    } else {
        col = p.w_hi + p.w_lo;
    }
    if (A.g.n) {
        if (A.g.pair) {
            const uint32_t ng = A.g.n;
            ok = ok && (p.g_hi == p.g_lo + 1u || (p.g_hi == 0u && p.g_lo == 0u) ||
                        (p.g_hi == ng && p.g_lo == ng));
            col += p.g_hi + (p.g_lo == ng ? 1u : 0u);
        } else {
            col += p.g_hi + p.g_lo;
        }
    }
    return ok;
}

// Edges of one side (or pairs) passed by x when the estimate is exact: farther
// than tol from every whole number (see grid_edges for tol).  `last` = edges.
OWM_HD uint32_t axis_fast1(double f, double last, double tol, bool &ok)
{
    const double i = floor(f), d = f - i;
    ok = ok && d > tol && d < 1.0 - tol;
    return (uint32_t)(int)fmin(fmax(i + 1.0, 0.0), last);
}

// The column by arithmetic; false where it is not certain (near an edge, NaN).
OWM_HD bool axis_col_fast(const GridAxis &A, double x, uint32_t &col)
{
    bool ok = true;
    const double f = (x - A.w.e0) * A.w.inv;
    uint32_t c = axis_fast1(f, (double)(A.w.n + A.w.pair), A.w.tol, ok);
    if (!A.w.pair)
        c += axis_fast1(f - A.w.cr, (double)A.w.n, A.w.tol, ok);
    if (A.g.n) {
        const double fg = (x - A.g.e0) * A.g.inv;
        c += axis_fast1(fg, (double)(A.g.n + A.g.pair), A.g.tol, ok);
        if (!A.g.pair)
            c += axis_fast1(fg - A.g.cr, (double)A.g.n, A.g.tol, ok);
    }
    col = c;
    return ok;
}

// Edges of F (pairs once) at or before v (equal) or before v.
OWM_HD uint32_t axis_edges_before(const GridEdges &F, bool cells, double v, bool equal)
{
    if (F.n == 0)
        return 0;
    const uint32_t l = axis_count(F, v, false, equal);
    const uint32_t r = axis_count(F, v, true, equal);
    if (!F.pair)
        return l + r;
    const uint32_t m = cells ? 1u : F.pair;  // R_i counts when it pairs with no L: i + m >= n
    const uint32_t first = F.n - m;
    return l + (r > first ? r - first : 0u);
}

// Columns [first, last] of window i: a point of column c lies in window i
// exactly when first <= c <= last (last < first: none).
OWM_HD void axis_window_cols(const GridAxis &A, uint32_t i, int &first, int &last)
{
    const double l = axis_edge(A.w, (int)i, false), r = axis_edge(A.w, (int)i, true);
    first = (int)(i + 1u + axis_edges_before(A.g, true, l, true));
    last = (int)(i + axis_edges_before(A.g, true, r, false));
    if (A.w.pair) {
        last += (int)A.w.pair;
    } else {
        first += (int)axis_count(A.w, l, true, true);
        last += (int)axis_count(A.w, r, false, false);
    }
}

// Columns [first, last] of stage-3 cell k.
OWM_HD void axis_cell_cols(const GridAxis &A, uint32_t k, int &first, int &last)
{
    const double l = axis_edge(A.g, (int)k, false), r = axis_edge(A.g, (int)k, true);
    first = (int)(k + 1u + axis_edges_before(A.w, false, l, true));
    last = (int)(k + axis_edges_before(A.w, false, r, false));
    if (A.g.pair) {
        last += 1;
    } else {
        first += (int)axis_count(A.g, l, true, true);
        last += (int)axis_count(A.g, r, false, false);
    }
}

// ------------------------------------------------------------- set-up ----

// The edges E_i = fl(fl(init + fl(i*step)) +- half) satisfy E_i = E_0 + i*step
// + e with |e| <= 2^-51 M for M bounding |init| and every edge, and for
// |x| <= M the estimate fl(fl(x - E_0) * inv) is within 3 * 2^-52 M / step of
// (x - E_0) / step (right edges, estimated by subtracting cr, at most
// 2^-50 M / step more); a pair's two edges differ by at most tol / 8 steps.
// With tol = 2^-45 M / step, an estimate farther than tol from every whole
// number therefore counts the passed edges exactly, and one beyond the last
// edge by more than a step clamps to the exact count for every x.
inline void grid_edges(GridEdges &E, double init, double step, double half, uint32_t n,
                       bool cells, uint32_t max_pair)
{
    E.init = init;
    E.step = step;
    E.inv = 1.0 / step;
    E.half = half;
    E.n = n;
    E.pair = 0;
    E.e0 = E.cr = E.tol = 0.0;
    if (!n)
        return;
    const double r0 = axis_edge(E, 0, true), last = axis_edge(E, (int)n - 1, true);
    E.e0 = axis_edge(E, 0, false);
    E.cr = (r0 - E.e0) * E.inv;
    const double m = fmax(fabs(init), fmax(fabs(E.e0), fabs(last))) + half + step;
    E.tol = ldexp(m, -45) * E.inv;
    const double w = round(E.cr);
    if (w >= 1.0 && w <= (double)max_pair && w <= (double)n && fabs(E.cr - w) <= 0.125 * E.tol &&
        E.tol < 1e-3)
        E.pair = (uint32_t)w;
    if (cells && E.pair > 1u)
        E.pair = 0;
}

inline void grid_axis(GridAxis &A)
{
    const uint32_t w = A.w.pair ? A.w.n + A.w.pair : 2u * A.w.n;
    const uint32_t g = A.g.pair ? A.g.n + 1u : 2u * A.g.n;
    A.ncol = w + g + 1u;
    A.pad = 0;
}

// An upper bound on the columns under bw neighbouring windows, for axes whose tol is at
// most 0.125 (rounding moves an edge by far less than a step).
inline double axis_cols_of(const GridAxis &A, uint32_t bw)
{
    const double len = (bw - 1) * A.w.step + 2.0 * A.w.half;
    double r = (len * A.w.inv + 1.0) * (A.w.pair ? 1.0 : 2.0);
    if (A.g.n)
        r += (len * A.g.inv + 1.0) * (A.g.pair ? 1.0 : 2.0);
    return ceil(r) + 4.0;
}
