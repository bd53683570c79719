// The column-grid chain of whole runs on gfx950: stages 1-3 of a tile whose
// tree nobody keeps, without building one.
//
// Every window and stage-3 cell is a rectangle of columns x rows of the tile's
// column grid (owm_axis.h), so a point matters only through the grid cell
// it lies in: its count and its (z, index).  The chain therefore streams the
// cloud twice and works on cells from there on:
//   k_grid_part     reads x, y, z once (24 B a point) and writes, per sort tile
//                   of GRID_PTS points, the points grouped by bucket (a rectangle
//                   of cells that fits LDS) as z key and cell (12 B a point), all
//                   writes linear, and where each bucket's run starts
//   k_grid_bin      gathers a bucket's runs (12 B a point), reduces them in LDS
//                   and writes the bucket's cells (16 B each)
//   k_grid_windows  per block of windows: the cells' rectangles reduced along x,
//                   then y; windows' minima mark the point bitmaps of stage 2
//   k_grid_cells    stage 3: the rectangle of each cell without an LLP
// Against the tree chain (56 B a point moved by each sort pass, 32 B by the leaf
// aggregates, about 35 B by stage 1 on window columns) a point moves 52 B after
// its box is known.  Measured on MI355X: 512 uneven tiles (329M points) 14.8 ->
// 6.1 ms (partition 2.1, bins 1.7, windows 0.5 ms), a 120M-point tile 6.6 ->
// 2.7 ms, 20M points with clusters 1.39 -> 0.63 ms, 1M points 0.32 -> 0.16 ms,
// 10k points 0.24 -> 0.13 ms.
// Points that lie on an edge (or between the two edges of a pair) have no
// column; k_grid_bin lists them with their exact window and cell ranges, and
// the last two kernels add them.
#include "owm_kernels.h"

namespace owm {

constexpr int GP_NT = 512, GP_K = GRID_PTS / GP_NT;
constexpr uint32_t KEY_NONE = 0xFFFFFFFFu, KEY_RARE = 0x80000000u;

// Table entry whose range of off[] holds v, found by the whole workgroup at
// once (off[t] <= v < off[t + 1]; s_t: one shared word).
__device__ __forceinline__ uint32_t find_entry(const uint32_t *__restrict__ off, uint32_t t0,
                                               uint32_t t1, uint32_t v, uint32_t *s_t)
{
    for (uint32_t t = t0 + threadIdx.x; t < t1; t += blockDim.x)
        if (off[t] <= v && v < off[t + 1])
            *s_t = t;
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(*s_t);
}

// Exclusive scan over the workgroup (NT threads); total of all.
template <int NT>
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t *s_w, uint32_t &total)
{
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t inc = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t u = __shfl_up(inc, o, 64);
        if (lane >= (uint32_t)o)
            inc += u;
    }
    if (lane == 63)
        s_w[w] = inc;
    __syncthreads();
    uint32_t add = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < NT / 64; ++k) {
        const uint32_t u = s_w[k];
        add += (uint32_t)k < w ? u : 0u;
        tot += u;
    }
    __syncthreads();
    total = tot;
    return add + inc - v;
}

// Bucket and cell within it of a column and row.
__device__ __forceinline__ uint32_t grid_key(const GridTile &T, uint32_t cx, uint32_t cy)
{
    const uint32_t b = (cy >> T.lh) * T.nbx + (cx >> T.lw);
    const uint32_t c = ((cy & ((1u << T.lh) - 1u)) << T.lw) | (cx & ((1u << T.lw) - 1u));
    return b << GRID_CELL_BITS | c;
}

// ------------------------------------------------------------- partition --

// Bound by HBM: 36 B a point at 5.5 TB/s (2.14 ms for 329M points; a plain copy
// reaches 4.9 TB/s).  The output of a sort tile is one linear stretch, so runs
// need no global offsets (no histogram pass, no look-back); the bins gather
// them.  4096 points (52 KB of LDS) leave room for three workgroups per CU, whose
// loads, ranking and writes overlap.
__global__ __launch_bounds__(GP_NT) void k_grid_part(GridDev G, const double *__restrict__ X,
                                                      const double *__restrict__ Y,
                                                      const double *__restrict__ Z)
{
    extern __shared__ unsigned long long s_part[];
    unsigned long long *sZ = s_part;                  // [GRID_PTS] z keys by bucket
    uint32_t *sW = (uint32_t *)(sZ + GRID_PTS);       // [GRID_PTS] cell and slot
    uint32_t *hist = sW + GRID_PTS;                   // [nb] counts, then offsets
    uint32_t *sList = (uint32_t *)sZ;                 // points near an edge
    __shared__ uint32_t s_t, s_n, s_w[GP_NT / 64];
    const uint32_t tid = threadIdx.x, u = blockIdx.x;
    if (tid == 0)
        s_n = 0;
    const uint32_t t = find_entry(G.st_off, 0, G.ntiles, u, &s_t);
    const GridTile &T = G.tiles[t];
    const uint32_t st = u - T.st_off;
    const uint32_t base = T.pt_off + st * GRID_PTS;
    const uint32_t cnt = min((uint32_t)GRID_PTS, T.n - st * GRID_PTS);
    const uint32_t nb = T.nb;
    double x[GP_K], y[GP_K], z[GP_K];
#pragma unroll
    for (int k = 0; k < GP_K; ++k) {
        const uint32_t i = base + min(tid + k * GP_NT, cnt - 1u);
        x[k] = X[i];
        y[k] = Y[i];
    }
#pragma unroll
    for (int k = 0; k < GP_K; ++k)
        z[k] = Z[base + min(tid + k * GP_NT, cnt - 1u)];
    for (uint32_t b = tid; b < nb; b += GP_NT)
        hist[b] = 0;
    uint32_t key[GP_K];
#pragma unroll
    for (int k = 0; k < GP_K; ++k) {
        uint32_t cx, cy;
        const bool okx = axis_col_fast(T.ax[0], x[k], cx);
        const bool oky = axis_col_fast(T.ax[1], y[k], cy);
        key[k] = okx && oky ? grid_key(T, cx, cy) : KEY_NONE;
    }
    // points near an edge: exact counts, the listed points spread over the
    // workgroup's lanes (in the loop above one such point would hold its wave)
#pragma unroll
    for (int k = 0; k < GP_K; ++k)
        if (key[k] == KEY_NONE && tid + k * GP_NT < cnt)
            sList[atomicAdd(&s_n, 1u)] = tid + k * GP_NT;
    __syncthreads();
    const uint32_t nl = s_n;
    if (nl) {
        for (uint32_t e = tid; e < nl; e += GP_NT) {
            const uint32_t slot = sList[e];
            uint32_t cx, cy;
            const bool okx = axis_col_exact(T.ax[0], axis_passed(T.ax[0], X[base + slot]), cx);
            const bool oky = axis_col_exact(T.ax[1], axis_passed(T.ax[1], Y[base + slot]), cy);
            sW[slot] = grid_key(T, cx, cy) | (okx && oky ? 0u : KEY_RARE);
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < GP_K; ++k)
            if (key[k] == KEY_NONE && tid + k * GP_NT < cnt)
                key[k] = sW[tid + k * GP_NT];
    }
    uint32_t rank[GP_K];
#pragma unroll
    for (int k = 0; k < GP_K; ++k)
        rank[k] = tid + k * GP_NT < cnt
                      ? atomicAdd(&hist[(key[k] & ~KEY_RARE) >> GRID_CELL_BITS], 1u)
                      : 0u;
    __syncthreads();
    // exclusive offsets of the buckets, nb / GP_NT consecutive ones per thread
    const uint32_t per = (nb + GP_NT - 1) / GP_NT, b0 = min(tid * per, nb), b1 = min(b0 + per, nb);
    uint32_t sum = 0;
    for (uint32_t b = b0; b < b1; ++b)
        sum += hist[b];
    uint32_t total;
    uint32_t run = block_scan<GP_NT>(sum, s_w, total);
    uint16_t *tab = G.tab + T.tab_off + (uint64_t)st * (nb + 1);
    for (uint32_t b = b0; b < b1; ++b) {
        const uint32_t h = hist[b];
        hist[b] = run;
        run += h;
    }
    __syncthreads();
    for (uint32_t b = tid; b < nb; b += GP_NT)
        tab[b] = (uint16_t)hist[b];
    if (tid == 0)
        tab[nb] = (uint16_t)cnt;
#pragma unroll
    for (int k = 0; k < GP_K; ++k) {
        const uint32_t slot = tid + k * GP_NT;
        if (slot < cnt) {
            const uint32_t pos = hist[(key[k] & ~KEY_RARE) >> GRID_CELL_BITS] + rank[k];
            sZ[pos] = owm_eligible(z[k]) ? owm_zkey(z[k]) : OWM_ZKEY_NONE;
            sW[pos] = (key[k] & KEY_RARE) | (key[k] & GRID_CELL_MASK) << GRID_SLOT_BITS | slot;
        }
    }
    __syncthreads();
    for (uint32_t i = tid; i < cnt; i += GP_NT) {
        G.zk[base + i] = sZ[i];
        G.cw[base + i] = sW[i];
    }
}

// ----------------------------------------------------------------- bins ----

constexpr int GB_NT = 512;   // threads
constexpr int GB_RUNS = 1024;  // run segments per pass
constexpr int GB_SEG = 4;    // points per lane and segment
constexpr int GB_TWO = 2;    // segments per lane group and round
constexpr int GB_KK = GB_SEG * GB_TWO;
constexpr uint32_t GB_RARE = 1024;  // points without a column listed in LDS before a flush

// Appends the listed points to the pool with their exact ranges; links the
// block of entries in front of `head`.  Every thread of the workgroup calls it.
__device__ void flush_rare(const GridDev &G, const GridTile &T, uint32_t item,
                           const double *__restrict__ X, const double *__restrict__ Y,
                           const double *__restrict__ Z, const uint32_t *list, uint32_t n,
                           uint32_t *s_base, uint32_t &head)
{
    const uint32_t sub = item & (GRID_POOLS - 1u);
    if (threadIdx.x == 0) {
        const uint32_t at = atomicAdd(G.pool_used + sub * 16, n + 1u);
        *s_base = at + n + 1u <= G.pool_cap ? sub * G.pool_cap + at : OWM_NONE;
        if (*s_base == OWM_NONE)
            atomicOr(G.err, GRID_ERR_POOL);
    }
    __syncthreads();
    const uint32_t base = *s_base;
    if (base != OWM_NONE) {
        if (threadIdx.x == 0) {
            GridRare h = {};
            h.id = n;
            h.next = head;
            G.pool[base] = h;
        }
        for (uint32_t e = threadIdx.x; e < n; e += GB_NT) {
            const uint32_t id = list[e];
            const AxisPassed px = axis_passed(T.ax[0], X[id]), py = axis_passed(T.ax[1], Y[id]);
            const double z = Z[id];
            GridRare r;
            r.zk = owm_eligible(z) ? owm_zkey(z) : OWM_ZKEY_NONE;
            r.id = id;
            r.next = 0;
            r.wx0 = (uint16_t)px.w_lo;
            r.wx1 = (uint16_t)px.w_hi;
            r.wy0 = (uint16_t)py.w_lo;
            r.wy1 = (uint16_t)py.w_hi;
            r.gx0 = (uint16_t)px.g_lo;
            r.gx1 = (uint16_t)px.g_hi;
            r.gy0 = (uint16_t)py.g_lo;
            r.gy1 = (uint16_t)py.g_hi;
            G.pool[base + 1 + e] = r;
        }
        head = base;
    }
    __syncthreads();
}

// One workgroup per item: a bucket's runs in one share of the tile's sort tiles.
// Cells keep (count, lowest z key, lowest index at that key); a round reads
// GB_KK points per lane, and its two barriers order the count and minimum, the
// reset of the index where the minimum dropped, and the index minimum.
__global__ __launch_bounds__(GB_NT) void k_grid_bin(GridDev G, const double *__restrict__ X,
                                                     const double *__restrict__ Y,
                                                     const double *__restrict__ Z, uint32_t t0,
                                                     uint32_t t1, uint32_t item0, uint32_t items,
                                                     uint32_t cells)
{
    extern __shared__ unsigned long long s_bin[];
    unsigned long long *sZ = s_bin;
    uint32_t *sId = (uint32_t *)(sZ + cells);
    uint32_t *sCnt = sId + cells;
    __shared__ uint32_t s_t, s_base, s_nr, s_w[GB_NT / 64];
    __shared__ uint2 sRun[GB_RUNS];
    __shared__ uint32_t sRare[GB_RARE];
    const uint32_t tid = threadIdx.x;
    // consecutive items (neighbouring buckets, whose runs share cache lines)
    // on one XCD: workgroups go round the eight XCDs
    const uint32_t per = (items + 7u) / 8u;
    const uint32_t rel = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    if (rel >= items || (blockIdx.x >> 3) >= per)
        return;
    const uint32_t item = item0 + rel;
    if (tid == 0)
        s_nr = 0;
    const uint32_t t = find_entry(G.item_off, t0, t1, item, &s_t);
    const GridTile &T = G.tiles[t];
    const uint32_t lc = T.lw + T.lh, nc = 1u << lc;
    const uint32_t q = item - T.item_off, bucket = q / T.split, part = q - bucket * T.split;
    const uint32_t st0 = (uint32_t)((uint64_t)T.nst * part / T.split);
    const uint32_t st1 = (uint32_t)((uint64_t)T.nst * (part + 1) / T.split);
    const uint32_t nb1 = T.nb + 1, lpr = T.lpr, seg_pts = (uint32_t)GB_SEG << lpr;
    for (uint32_t c = tid; c < nc; c += GB_NT) {
        sZ[c] = OWM_ZKEY_NONE;
        sId[c] = OWM_NONE;
        sCnt[c] = 0;
    }
    uint32_t head = OWM_NONE;
    const uint32_t grp = tid >> lpr, ngrp = GB_NT >> lpr, gl = tid & ((1u << lpr) - 1u);
    for (uint32_t s0 = st0; s0 < st1; s0 += GB_NT) {
        // this thread's sort tile: the bucket's run, in segments of seg_pts
        const uint32_t s = s0 + tid;
        uint32_t o0 = 0, o1 = 0;
        if (s < st1) {
            const uint16_t *row = G.tab + T.tab_off + (uint64_t)s * nb1 + bucket;
            o0 = row[0];
            o1 = row[1];
        }
        const uint32_t nseg = (o1 - o0 + seg_pts - 1) / seg_pts;
        uint32_t total;
        const uint32_t first = block_scan<GB_NT>(nseg, s_w, total);
        for (uint32_t p0 = 0; p0 < total; p0 += GB_RUNS) {
            for (uint32_t e = max(first, p0); e < min(first + nseg, p0 + GB_RUNS); ++e) {
                const uint32_t a = o0 + (e - first) * seg_pts;
                // first point of the segment (sort tiles start at multiples of
                // GRID_PTS within the tile), points in it
                sRun[e - p0] = make_uint2(T.pt_off + s * GRID_PTS + a,
                                          min(seg_pts, o1 - a) | (a << 16));
            }
            __syncthreads();
            const uint32_t here = min((uint32_t)GB_RUNS, total - p0);
            for (uint32_t r0 = 0; r0 < here; r0 += ngrp * GB_TWO) {
                unsigned long long zk[GB_KK];
                uint32_t cw[GB_KK], id0[GB_TWO];
#pragma unroll
                for (int h = 0; h < GB_TWO; ++h) {
                    const uint32_t e = r0 + h * ngrp + grp;
                    const uint2 run = e < here ? sRun[e] : make_uint2(0u, 0u);
                    const uint32_t len = run.y & 0xFFFFu;
                    id0[h] = run.x - (run.y >> 16);  // first point of the sort tile
#pragma unroll
                    for (int k = 0; k < GB_SEG; ++k) {
                        const uint32_t i = gl + ((uint32_t)k << lpr);
                        cw[h * GB_SEG + k] = KEY_NONE;
                        zk[h * GB_SEG + k] = OWM_ZKEY_NONE;
                        if (i < len) {
                            zk[h * GB_SEG + k] = G.zk[run.x + i];
                            cw[h * GB_SEG + k] = G.cw[run.x + i];
                        }
                    }
                }
                uint32_t cand = 0, drop = 0, pend = 0;
#pragma unroll
                for (int k = 0; k < GB_KK; ++k) {
                    const uint32_t w = cw[k];
                    if (w == KEY_NONE)
                        continue;
                    if (w & KEY_RARE) {
                        const uint32_t e = atomicAdd(&s_nr, 1u);
                        if (e < GB_RARE)
                            sRare[e] = id0[k / GB_SEG] + (w & GRID_SLOT_MASK);
                        else
                            pend |= 1u << k;
                        continue;
                    }
                    const uint32_t c = w >> GRID_SLOT_BITS;
                    atomicAdd(&sCnt[c], 1u);
                    if (zk[k] != OWM_ZKEY_NONE && zk[k] <= sZ[c]) {
                        const unsigned long long old = atomicMin(&sZ[c], zk[k]);
                        cand |= (zk[k] <= old ? 1u : 0u) << k;
                        drop |= (zk[k] < old ? 1u : 0u) << k;
                    }
                }
                // the list was full for some points: flushed until all are on it
                while (__syncthreads_or(pend != 0)) {
                    flush_rare(G, T, item, X, Y, Z, sRare, GB_RARE, &s_base, head);
                    if (tid == 0)
                        s_nr = 0;
                    __syncthreads();
#pragma unroll
                    for (int k = 0; k < GB_KK; ++k)
                        if ((pend >> k) & 1u) {
                            const uint32_t e = atomicAdd(&s_nr, 1u);
                            if (e < GB_RARE) {
                                sRare[e] = id0[k / GB_SEG] + (cw[k] & GRID_SLOT_MASK);
                                pend &= ~(1u << k);
                            }
                        }
                }
#pragma unroll
                for (int k = 0; k < GB_KK; ++k)
                    if (((drop >> k) & 1u) && sZ[cw[k] >> GRID_SLOT_BITS] == zk[k])
                        sId[cw[k] >> GRID_SLOT_BITS] = OWM_NONE;
                __syncthreads();
#pragma unroll
                for (int k = 0; k < GB_KK; ++k)
                    if (((cand >> k) & 1u) && sZ[cw[k] >> GRID_SLOT_BITS] == zk[k])
                        atomicMin(&sId[cw[k] >> GRID_SLOT_BITS],
                                  id0[k / GB_SEG] + (cw[k] & GRID_SLOT_MASK));
            }
            __syncthreads();  // sRun is rewritten
        }
    }
    __syncthreads();
    if (s_nr) {
        const uint32_t n = min(s_nr, GB_RARE);
        flush_rare(G, T, item, X, Y, Z, sRare, n, &s_base, head);
    }
    if (tid == 0)
        G.heads[item] = head;
    uint4 *out = G.cells + T.cell_off + ((uint64_t)q << lc);
    for (uint32_t c = tid; c < nc; c += GB_NT) {
        const unsigned long long zk = sZ[c];
        out[c] = make_uint4((uint32_t)zk, (uint32_t)(zk >> 32), sId[c], sCnt[c]);
    }
}

// -------------------------------------------------------------- windows --

constexpr int GW_NT = 256;
constexpr uint32_t GW_SEGS = 512;  // pool blocks a window block can meet
constexpr int GW_PER = 32 * 32 / GW_NT;  // windows per thread, at most

struct CellAgg {
    unsigned long long zk;
    uint32_t id, cnt;
};

__device__ __forceinline__ void agg_add(CellAgg &a, unsigned long long zk, uint32_t id, uint32_t cnt)
{
    a.cnt += cnt;
    if (owm_less(zk, id, a.zk, a.id)) {
        a.zk = zk;
        a.id = id;
    }
}

// Adds the cell of column c in the row whose cells of bucket column 0 start at
// `row` (all shares of the bucket).
__device__ __forceinline__ void cell_add(CellAgg &a, const GridTile &T, const uint4 *row, uint32_t c)
{
    const uint32_t lc = T.lw + T.lh;
    const uint4 *p = row + ((uint64_t)(c >> T.lw) * T.split << lc) + (c & ((1u << T.lw) - 1u));
    for (uint32_t k = 0; k < T.split; ++k, p += 1u << lc) {
        const uint4 v = *p;
        agg_add(a, (unsigned long long)v.y << 32 | v.x, v.z, v.w);
    }
}

__device__ __forceinline__ const uint4 *cell_row(const GridDev &G, const GridTile &T, uint32_t r)
{
    const uint32_t lc = T.lw + T.lh;
    return G.cells + T.cell_off + ((uint64_t)(r >> T.lh) * T.nbx * T.split << lc) +
           ((r & ((1u << T.lh) - 1u)) << T.lw);
}

// Buckets (as ranges of bucket columns and rows) whose listed points can lie in
// the columns and rows given: a point without a column is kept in the bucket
// of a column next to its place.
__device__ __forceinline__ void rare_buckets(const GridTile &T, int c0, int c1, int r0, int r1,
                                             uint32_t &bx0, uint32_t &bx1, uint32_t &by0,
                                             uint32_t &by1)
{
    bx0 = min((uint32_t)max(c0 - 2, 0) >> T.lw, T.nbx - 1u);
    by0 = min((uint32_t)max(r0 - 2, 0) >> T.lh, T.nby - 1u);
    bx1 = max(min((uint32_t)max(c1 + 2, 0) >> T.lw, T.nbx - 1u), bx0);
    by1 = max(min((uint32_t)max(r1 + 2, 0) >> T.lh, T.nby - 1u), by0);
}

// Marks `id` as an LLP; the first to do so marks the stage-3 cells that
// hold it (as k_s3_mark).
__device__ __forceinline__ void mark_llp(const GridDev &G, const GridTile &T, uint32_t id,
                                         const double *__restrict__ X, const double *__restrict__ Y)
{
    const uint32_t bit = 1u << (id & 31u);
    if ((atomicOr(G.llp + (id >> 5), bit) & bit) || T.ax[0].g.n == 0)
        return;
    const double x = X[id], y = Y[id];
    const uint32_t x0 = axis_count(T.ax[0].g, x, true, true), x1 = axis_count(T.ax[0].g, x, false, false);
    const uint32_t y0 = axis_count(T.ax[1].g, y, true, true), y1 = axis_count(T.ax[1].g, y, false, false);
    for (uint32_t j = y0; j < y1; ++j)
        for (uint32_t i = x0; i < x1; ++i)
            G.cell_flag[T.gcell_off + j * T.ax[0].g.n + i] = 1u;
}

// One workgroup per block of bw x bw windows: row sums of the cells per window
// column (k_stage1_pairs' separable reduction, here over cells in memory), then
// the windows, then the listed points, then stage 2's marks.
__global__ __launch_bounds__(GW_NT) void k_grid_windows(GridDev G, const double *__restrict__ X,
                                                         const double *__restrict__ Y,
                                                         uint32_t rows_cap)
{
    extern __shared__ unsigned long long s_win[];
    __shared__ uint32_t s_t, s_nseg;
    __shared__ int sx0[32], sx1[32], sy0[32], sy1[32];
    __shared__ uint2 sSeg[GW_SEGS];
    const uint32_t tid = threadIdx.x;
    if (tid == 0)
        s_nseg = 0;
    const uint32_t t = find_entry(G.blk_off, 0, G.ntiles, blockIdx.x, &s_t);
    const GridTile &T = G.tiles[t];
    const uint32_t lb = T.lbw, bw = 1u << lb;
    const uint32_t q0 = blockIdx.x - T.blk_off, bj = q0 / T.nblkx, bi = q0 - bj * T.nblkx;
    const uint32_t nx = T.ax[0].w.n, ny = T.ax[1].w.n;
    const uint32_t i0 = bi << lb, j0 = bj << lb;
    const uint32_t ni = min(bw, nx - i0), nj = min(bw, ny - j0);
    if (tid < ni)
        axis_window_cols(T.ax[0], i0 + tid, sx0[tid], sx1[tid]);
    else if (tid >= 64 && tid - 64 < nj)
        axis_window_cols(T.ax[1], j0 + tid - 64, sy0[tid - 64], sy1[tid - 64]);
    __syncthreads();
    const int c0 = sx0[0], c1 = sx1[ni - 1], r0 = sy0[0], r1 = sy1[nj - 1];
    uint32_t nr = r1 >= r0 ? (uint32_t)(r1 - r0 + 1) : 0u;
    unsigned long long *mZ = s_win;                       // [rows_cap * bw]
    uint32_t *mId = (uint32_t *)(mZ + (rows_cap << 5));
    uint32_t *mCnt = mId + (rows_cap << 5);
    if (nr > (rows_cap << 5) >> lb) {  // cannot happen (the host sizes rows_cap)
        if (tid == 0)
            atomicOr(G.err, GRID_ERR_ROWS);
        nr = (rows_cap << 5) >> lb;
    }
    // the listed points' pool blocks, while the cells are read
    uint32_t bx0, bx1, by0, by1;
    rare_buckets(T, c0, c1, r0, r1, bx0, bx1, by0, by1);
    {
        const uint32_t wx = (bx1 - bx0 + 1) * T.split, all = wx * (by1 - by0 + 1);
        for (uint32_t k = tid; k < all; k += GW_NT) {
            const uint32_t row = k / wx;
            uint32_t h = G.heads[T.item_off + ((by0 + row) * T.nbx + bx0) * T.split + (k - row * wx)];
            while (h != OWM_NONE) {
                const GridRare &r = G.pool[h];
                const uint32_t e = atomicAdd(&s_nseg, 1u);
                if (e < GW_SEGS)
                    sSeg[e] = make_uint2(h + 1, r.id);
                else
                    atomicOr(G.err, GRID_ERR_POOL);
                h = r.next;
            }
        }
    }
    for (uint32_t q = tid; q < nr << lb; q += GW_NT) {
        const uint32_t rr = q >> lb, w = q & (bw - 1u);
        if (w >= ni)
            continue;
        CellAgg a = {OWM_ZKEY_NONE, OWM_NONE, 0};
        const uint4 *row = cell_row(G, T, (uint32_t)r0 + rr);
        for (int c = sx0[w]; c <= sx1[w]; ++c)
            cell_add(a, T, row, (uint32_t)c);
        mZ[q] = a.zk;
        mId[q] = a.id;
        mCnt[q] = a.cnt;
    }
    __syncthreads();
    CellAgg win[GW_PER];
#pragma unroll
    for (int k = 0; k < GW_PER; ++k) {
        const uint32_t q = tid + k * GW_NT, v = q >> lb, w = q & (bw - 1u);
        win[k] = {OWM_ZKEY_NONE, OWM_NONE, 0};
        if (v < nj && w < ni)
            for (int r = sy0[v]; r <= sy1[v]; ++r) {
                const uint32_t m = ((uint32_t)(r - r0) << lb) + w;
                agg_add(win[k], mZ[m], mId[m], mCnt[m]);
            }
    }
    __syncthreads();  // the row sums are no longer needed: their memory holds the windows
    const uint32_t nseg = min(s_nseg, GW_SEGS);
    if (nseg) {
        const uint32_t lane = tid & 63, wv = tid >> 6;
#pragma unroll
        for (int k = 0; k < GW_PER; ++k) {
            const uint32_t q = tid + k * GW_NT;
            if (q < bw * bw) {
                mZ[q] = win[k].zk;
                mId[q] = win[k].id;
                mCnt[q] = win[k].cnt;
            }
        }
        __syncthreads();
        for (uint32_t sg = wv; sg < nseg; sg += GW_NT / 64)
            for (uint32_t e = lane; e < sSeg[sg].y; e += 64) {
                const GridRare r = G.pool[sSeg[sg].x + e];
                const uint32_t x0 = max((uint32_t)r.wx0, i0), x1 = min((uint32_t)r.wx1, i0 + ni);
                const uint32_t y0 = max((uint32_t)r.wy0, j0), y1 = min((uint32_t)r.wy1, j0 + nj);
                for (uint32_t y = y0; y < y1; ++y)
                    for (uint32_t x = x0; x < x1; ++x) {
                        const uint32_t q = ((y - j0) << lb) + (x - i0);
                        atomicAdd(&mCnt[q], 1u);
                        if (r.zk < mZ[q])
                            atomicMin(&mZ[q], r.zk);
                    }
            }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < GW_PER; ++k) {
            const uint32_t q = tid + k * GW_NT;
            if (q < bw * bw && mZ[q] < win[k].zk)
                mId[q] = OWM_NONE;
        }
        __syncthreads();
        for (uint32_t sg = wv; sg < nseg; sg += GW_NT / 64)
            for (uint32_t e = lane; e < sSeg[sg].y; e += 64) {
                const GridRare r = G.pool[sSeg[sg].x + e];
                if (r.zk == OWM_ZKEY_NONE)
                    continue;
                const uint32_t x0 = max((uint32_t)r.wx0, i0), x1 = min((uint32_t)r.wx1, i0 + ni);
                const uint32_t y0 = max((uint32_t)r.wy0, j0), y1 = min((uint32_t)r.wy1, j0 + nj);
                for (uint32_t y = y0; y < y1; ++y)
                    for (uint32_t x = x0; x < x1; ++x) {
                        const uint32_t q = ((y - j0) << lb) + (x - i0);
                        if (mZ[q] == r.zk)
                            atomicMin(&mId[q], r.id);
                    }
            }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < GW_PER; ++k) {
            const uint32_t q = tid + k * GW_NT;
            if (q < bw * bw)
                win[k] = {mZ[q], mId[q], mCnt[q]};
        }
        __syncthreads();
    }
    // stage 2 (as k_s2_mark): only the first window of a patch of windows that
    // share their minimum acts; one beside another of its patch marks the point
    // as an LLP at once, a single one when the point was a minimum elsewhere
    uint32_t *sMin = (uint32_t *)s_win;  // [bw * bw] minima
#pragma unroll
    for (int k = 0; k < GW_PER; ++k) {
        const uint32_t q = tid + k * GW_NT;
        if (q < bw * bw) {
            const bool valid = win[k].cnt >= T.min_num_points && win[k].zk != OWM_ZKEY_NONE;
            win[k].id = valid && (q >> lb) < nj && (q & (bw - 1u)) < ni ? win[k].id : OWM_NONE;
            sMin[q] = win[k].id;
        }
    }
    __syncthreads();
    uint32_t act[GW_PER], old[GW_PER];
#pragma unroll
    for (int k = 0; k < GW_PER; ++k) {
        const uint32_t q = tid + k * GW_NT, w = q & (bw - 1u), v = q >> lb, id = win[k].id;
        act[k] = 0;
        if (q < bw * bw && id != OWM_NONE && !(w > 0 && sMin[q - 1] == id) &&
            !(v > 0 && sMin[q - bw] == id))
            act[k] = T.stage2_need == 1u || (w + 1 < bw && sMin[q + 1] == id) ||
                             (v + 1 < bw && sMin[q + bw] == id)
                         ? 1u
                         : 2u;
    }
#pragma unroll
    for (int k = 0; k < GW_PER; ++k)
        old[k] = act[k] == 2 ? atomicOr(G.seen + (win[k].id >> 5), 1u << (win[k].id & 31u)) : 0u;
#pragma unroll
    for (int k = 0; k < GW_PER; ++k)
        if (act[k] == 1 || (act[k] == 2 && ((old[k] >> (win[k].id & 31u)) & 1u)))
            mark_llp(G, T, win[k].id, X, Y);
}

// --------------------------------------------------------------- cells ----

// One wave per stage-3 cell without an LLP: the lowest (z, index) of its
// columns and rows and of the listed points inside it joins the seeds' bitmap.
__global__ __launch_bounds__(256) void k_grid_cells(GridDev G)
{
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (uint32_t c = blockIdx.x * 4 + w; c < G.ngcell; c += gridDim.x * 4) {
        if (G.cell_flag[c])
            continue;
        const uint32_t t = owm_find_tile(G.gcell_off, G.ntiles, c);
        const GridTile &T = G.tiles[t];
        const uint32_t l = c - T.gcell_off, nx = T.ax[0].g.n;
        const uint32_t jj = l / nx, ii = l - jj * nx;
        // columns by the even lanes, rows by the odd ones
        int first, last;
        axis_cell_cols(T.ax[lane & 1u], lane & 1u ? jj : ii, first, last);
        const int c0 = __shfl(first, 0, 64), c1 = __shfl(last, 0, 64);
        const int r0 = __shfl(first, 1, 64), r1 = __shfl(last, 1, 64);
        CellAgg a = {OWM_ZKEY_NONE, OWM_NONE, 0};
        if (c1 >= c0 && r1 >= r0) {
            const uint32_t nc = (uint32_t)(c1 - c0 + 1), all = nc * (uint32_t)(r1 - r0 + 1);
            for (uint32_t q = lane; q < all; q += 64) {
                const uint32_t r = q / nc;
                cell_add(a, T, cell_row(G, T, (uint32_t)r0 + r), (uint32_t)c0 + (q - r * nc));
            }
        }
        uint32_t bx0, bx1, by0, by1;
        rare_buckets(T, c0, c1, r0, r1, bx0, bx1, by0, by1);
        const uint32_t wx = (bx1 - bx0 + 1) * T.split, all = wx * (by1 - by0 + 1);
        for (uint32_t k0 = 0; k0 < all; k0 += 64) {
            const uint32_t k = k0 + lane, row = k / wx;
            uint32_t h = k < all ? G.heads[T.item_off + ((by0 + row) * T.nbx + bx0) * T.split +
                                           (k - row * wx)]
                                 : OWM_NONE;
            // one list at a time, its entries over the wave
            unsigned long long some = __ballot(h != OWM_NONE);
            while (some) {
                const int src = __builtin_ctzll(some);
                some &= some - 1;
                uint32_t at = __shfl(h, src, 64);
                while (at != OWM_NONE) {
                    const uint32_t n = G.pool[at].id, next = G.pool[at].next;
                    for (uint32_t e = lane; e < n; e += 64) {
                        const GridRare r = G.pool[at + 1 + e];
                        if (ii >= r.gx0 && ii < r.gx1 && jj >= r.gy0 && jj < r.gy1)
                            agg_add(a, r.zk, r.id, 1);
                    }
                    at = next;
                }
            }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const unsigned long long zk = __shfl_xor(a.zk, o, 64);
            const uint32_t id = __shfl_xor(a.id, o, 64);
            agg_add(a, zk, id, 0);
        }
        if (lane == 0 && a.zk != OWM_ZKEY_NONE)
            atomicOr(G.llp + (a.id >> 5), 1u << (a.id & 31u));
    }
}

// ----------------------------------------------------------------- launch --

void launch_grid_part(hipStream_t s, const GridDev &G, const double *x, const double *y,
                      const double *z, uint32_t sort_tiles, uint32_t max_nb)
{
    if (!sort_tiles)
        return;
    const uint32_t lds = GRID_PTS * 12u + max_nb * 4u;
    hipLaunchKernelGGL(k_grid_part, dim3(sort_tiles), dim3(GP_NT), lds, s, G, x, y, z);
}

void launch_grid_bin(hipStream_t s, const GridDev &G, const double *x, const double *y,
                     const double *z, uint32_t t0, uint32_t t1, uint32_t item0, uint32_t items,
                     uint32_t cells)
{
    if (!items)
        return;
    const uint32_t g = (items + 7u) / 8u * 8u;
    hipLaunchKernelGGL(k_grid_bin, dim3(g), dim3(GB_NT), cells * 16u, s, G, x, y, z, t0, t1, item0,
                       items, cells);
}

void launch_grid_windows(hipStream_t s, const GridDev &G, const double *x, const double *y,
                         uint32_t blocks, uint32_t rows_cap)
{
    if (!blocks)
        return;
    hipLaunchKernelGGL(k_grid_windows, dim3(blocks), dim3(GW_NT), rows_cap * 32u * 16u, s, G, x, y,
                       rows_cap);
}

void launch_grid_cells(hipStream_t s, const GridDev &G)
{
    if (!G.ngcell)
        return;
    uint32_t g = (G.ngcell + 3) / 4;
    g = g > 16384 ? 16384 : g;
    hipLaunchKernelGGL(k_grid_cells, dim3(g), dim3(256), 0, s, G);
}

// LDS of more than 64 KB per workgroup is taken by dynamic size alone on
// gfx950; the attribute tells the runtime to expect it.
hipError_t grid_kernels_init()
{
    hipError_t e = hipFuncSetAttribute((const void *)k_grid_part,
                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                       GRID_PTS * 12 + GRID_MAX_BUCKETS * 4);
    if (e == hipSuccess)
        e = hipFuncSetAttribute((const void *)k_grid_bin, hipFuncAttributeMaxDynamicSharedMemorySize,
                                GRID_MAX_CELLS * 16);
    return e;
}

}  // namespace owm
