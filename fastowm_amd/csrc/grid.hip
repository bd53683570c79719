// The column-grid chain of whole runs on gfx950: stages 1-3 of a tile whose
// tree nobody keeps, without building one.
//
// Every window and stage-3 cell is a rectangle of columns x rows of the tile's
// column grid (owm_axis.h), so a point matters only through the grid cell
// it lies in: its count and its (z, index).  The chain therefore streams the
// cloud twice and works on cells from there on:
//   k_grid_part     reads x, y, z once (24 B a point) and writes, per sort tile
//                   of 2^lsp points, the points grouped by bucket (a rectangle
//                   of cells that fits LDS) as z key and cell (12 B a point), all
//                   writes linear, and where each bucket's run starts
//   k_grid_bin      gathers a bucket's runs (12 B a point), reduces them in LDS
//                   and writes the bucket's cells (16 B each)
//   k_grid_windows  per block of windows: the cells' rectangles reduced along x,
//                   then y; windows' minima mark the point bitmaps of stage 2
//   k_grid_cells    stage 3: the rectangle of each cell without an LLP
// Against the tree chain (56 B a point moved by each sort pass, 32 B by the leaf
// aggregates, about 35 B by stage 1 on window columns) a point moves 48 B after
// its box is known.  Measured on MI355X: 512 uneven tiles (329M points) 14.6 ->
// 5.3 ms (partition 2.3, bins 1.0, windows 0.3 ms), a 120M-point tile 6.6 ->
// 1.9 ms, 20M points with clusters 1.38 -> 0.43 ms, 1M points 0.32 -> 0.10 ms,
// 10k points 0.25 -> 0.07 ms.
// Points that lie on an edge (or between the two edges of a pair) have no
// column; k_grid_part puts their exact window and cell ranges into a pool,
// k_grid_bin lists each bucket's, and the last two kernels add them.
#include "owm_kernels.h"
#include <algorithm>
#include <utility>

namespace owm {

// threads of the partition
constexpr int gp_threads(int lsp) { return lsp == 13 ? 1024 : 512; }
constexpr uint32_t KEY_NONE = 0x7FFFFFFFu, KEY_RARE = 0x80000000u;

// Table entry whose range of off[] holds v, found by the whole workgroup at
// once (off[t] <= v < off[t + 1]; s_t: one shared word): each thread's look, then what
// one of them found.
__device__ __forceinline__ void look_for_entry(const uint32_t *__restrict__ off, uint32_t t0,
                                               uint32_t t1, uint32_t v, uint32_t *s_t)
{
    for (uint32_t t = t0 + threadIdx.x; t < t1; t += blockDim.x)
        if (off[t] <= v && v < off[t + 1])
            *s_t = t;
}

__device__ __forceinline__ uint32_t entry_found(const uint32_t *s_t)
{
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(*s_t);
}

// Bucket and cell within it of a column and row.
__device__ __forceinline__ uint32_t grid_key(const GridTile &T, uint32_t cx, uint32_t cy)
{
    const uint32_t b = (cy >> T.lh) * T.nbx + (cx >> T.lw);
    const uint32_t c = ((cy & ((1u << T.lh) - 1u)) << T.lw) | (cx & ((1u << T.lw) - 1u));
    return b << GRID_CELL_BITS | c;
}

// The same for a point of that column and row; bucket nb, which is not written, for
// one before an axis's first edge or behind its last (a window has two: ncol > 2).
__device__ __forceinline__ uint32_t point_key(const GridTile &T, uint32_t cx, uint32_t cy)
{
    const bool out = cx - 1u >= T.ax[0].ncol - 2u || cy - 1u >= T.ax[1].ncol - 2u;
    return out ? T.nb << GRID_CELL_BITS : grid_key(T, cx, cy);
}

// Everything the chain starts from: ranges that must be zero (blockIdx.y below
// their count), and the columns of every window of a tile, x then y.
// The table of a few tiles is read from host memory, and copied, here: an upload
// of its own would cost more.
__global__ __launch_bounds__(256) void k_grid_prep(GridDev G, FillRanges r, uint32_t windows,
                                                    const uint32_t *__restrict__ host_table,
                                                    uint32_t table_words)
{
    const uint32_t i0 = blockIdx.x * 256u + threadIdx.x;
    if (blockIdx.y < r.count) {
        uint32_t *p = r.ptr[blockIdx.y];
        const uint64_t n = r.len[blockIdx.y];
        for (uint64_t i = i0; i < n; i += gridDim.x * 256ull)
            p[i] = 0;
        return;
    }
    const uint32_t *own = (const uint32_t *)G.tiles;
    if (blockIdx.y > r.count) {
        for (uint32_t i = i0; i < table_words; i += gridDim.x * 256u)
            const_cast<uint32_t *>(own)[i] = host_table[i];
        return;
    }
    const uint32_t *table = host_table ? host_table : own;
    const uint32_t *axis_off = table + (G.axis_off - own);
    for (uint32_t i = i0; i < windows; i += gridDim.x * 256u) {
        const uint32_t t = owm_find_tile(axis_off, G.ntiles, i);
        const GridTile &T = ((const GridTile *)table)[t];
        const uint32_t q = i - axis_off[t], n = T.ax[0].w.n, a = q >= n ? 1u : 0u;
        int first, last;
        axis_window_cols(T.ax[a], a ? q - n : q, first, last);
        G.wcols[i] = make_int2(first, last);
    }
}

// ------------------------------------------------------------- partition --

// Word k of *p as other XCDs' atomics leave it (agent scope: sc1).  To the compiler an
// atomic load might write, and what follows it would not come by scalar loads: the
// partition would keep the tile's fields in lanes' registers and spill them (8M
// points 97 -> 154 us).
__device__ __forceinline__ uint32_t load_past_caches(uint32_t *p, uint32_t k)
{
    return __builtin_amdgcn_raw_buffer_load_b32(
        __builtin_amdgcn_make_buffer_rsrc(p, 0, 4 * k + 4, 0x00027000), 4 * k, 0, 16);
}

// Bound by HBM: 36 B a point at 5.2 TB/s (2.27 ms for 329M points; a plain copy
// reaches 4.9 TB/s).  The output of a sort tile is one linear stretch, so runs
// need no global offsets (no histogram pass, no look-back); the bins gather
// them.  4096 points (52 KB of LDS) leave room for three workgroups per CU, whose
// loads, ranking and writes overlap; that takes at most 80 registers (with 81, two
// workgroups per CU, centimetre coordinates and clusters ran slower: 8M points
// 78 us instead of 66, 96 mixed tiles 1.20 ms instead of 1.00; without points
// near edges it was 2.15 ms against 2.27 for the 329M points).
// TREE: the points come from a resident tree, whose order only groups them (33 us
// for its 3M points).
// Points before an axis's first edge or behind its last (of a box that holds a part
// of the tile) are in no window and no cell and get no record; kept, one workgroup
// of the bins would gather them (20M points, a box of a tenth of each side: bins
// 7.9 -> 0.02 ms, the whole run 8.3 -> 0.18 ms).  The test adds nothing measurable.
// LSP 13: 100 KB of LDS, one workgroup per CU, for runs that would else be short.
template <bool TREE, int LSP>
__global__ __launch_bounds__(gp_threads(LSP), LSP == 13 ? 4 : 6) void k_grid_part(GridDev G, const double *__restrict__ X,
                                                      const double *__restrict__ Y,
                                                      const double *__restrict__ Z)
{
    constexpr uint32_t PTS = 1u << LSP;
    constexpr int GP_NT = gp_threads(LSP), GP_K = PTS / GP_NT;
    extern __shared__ uint4 s_part[];
    uint32_t *sRec = (uint32_t *)s_part;              // [PTS] records by bucket
    uint32_t *hist = sRec + 3 * PTS;             // [nb + 1] counts, then offsets
    uint32_t *sList = sRec;                           // points near an edge
    uint32_t *sPool = sList + PTS;               // pool entry of a slot without a column
    uint32_t *sW = sPool + PTS;                  // exact key of a slot near an edge
    __shared__ uint32_t s_t, s_n, s_nr, s_base, s_stop, s_w[GP_NT / 64];
    const uint32_t tid = threadIdx.x, u = blockIdx.x;
    if (tid == 0)
        s_n = s_nr = 0;
    // (other workgroups may set it meanwhile: one thread reads it for all, the last,
    // which has no part in finding the tile of most launches)
    if (tid == GP_NT - 1)
        s_stop = load_past_caches(G.err, GRID_STOP_PART);
    look_for_entry(G.st_off, 0, G.ntiles, u, &s_t);
    const uint32_t t = entry_found(&s_t);
    if (s_stop)
        return;
    const GridTile &T = G.tiles[t];
    const uint32_t st = u - T.st_off;
    const uint32_t base = T.pt_off + st * PTS;
    const uint32_t cnt = min(PTS, T.n - st * PTS);
    const uint32_t nb = T.nb;
    double x[GP_K], y[GP_K], z[GP_K];
#pragma unroll
    for (int k = 0; k < GP_K; ++k) {
        const uint32_t i = base + min(tid + k * GP_NT, cnt - 1u);
        if (TREE) {
            const double2 v = G.xy[i];
            x[k] = v.x;
            y[k] = v.y;
        } else {
            x[k] = X[i];
            y[k] = Y[i];
        }
    }
#pragma unroll
    for (int k = 0; k < GP_K; ++k) {
        const uint32_t i = base + min(tid + k * GP_NT, cnt - 1u);
        z[k] = TREE ? G.zi[i].z : Z[i];
    }
    for (uint32_t b = tid; b <= nb; b += GP_NT)
        hist[b] = 0;
    uint32_t key[GP_K];
#pragma unroll
    for (int k = 0; k < GP_K; ++k) {
        uint32_t cx, cy;
        const bool okx = axis_col_fast(T.ax[0], x[k], cx);
        const bool oky = axis_col_fast(T.ax[1], y[k], cy);
        key[k] = okx && oky ? point_key(T, cx, cy) : KEY_NONE;
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
            const double xs = TREE ? G.xy[base + slot].x : X[base + slot];
            const double ys = TREE ? G.xy[base + slot].y : Y[base + slot];
            const bool okx = axis_col_exact(T.ax[0], axis_passed(T.ax[0], xs), cx);
            const bool oky = axis_col_exact(T.ax[1], axis_passed(T.ax[1], ys), cy);
            sW[slot] = okx && oky ? point_key(T, cx, cy) : grid_key(T, cx, cy) | KEY_RARE;
            if (!(okx && oky))
                atomicAdd(&s_nr, 1u);
        }
        __syncthreads();
        const uint32_t nr = s_nr;
        if (nr) {
            // their ranges go to the pool (counted again: few points take this)
            __syncthreads();
            if (tid == 0) {
                // (a share asked for more than it has left is closed, and some others are
                // asked: points on edges may lie in few sort tiles; 64 tries in a row
                // kept the last sort tiles of a full pool 25 us)
                s_base = OWM_NONE;
                for (uint32_t k = 0; k < 8 && s_base == OWM_NONE; ++k) {
                    const uint32_t share = (u + 9 * k) & (GRID_POOLS - 1u);
                    const uint32_t at = atomicAdd(G.pool_used + share * 32, nr);
                    s_base = at + nr <= G.pool_cap ? share * G.pool_cap + at : OWM_NONE;
                }
                const bool many = nr * 6 > cnt && atomicAdd(G.pool_used + 8, 1u) >= G.many_cap;
                if (s_base == OWM_NONE || many) {
                    atomicOr(G.err, GRID_ERR_POOL);
                    atomicOr(G.err + GRID_STOP_PART, 1u);
                }
                s_nr = 0;
            }
            __syncthreads();
            const uint32_t pbase = s_base;
            for (uint32_t e = tid; e < nl; e += GP_NT) {
                const uint32_t slot = sList[e], i = base + slot;
                if (!(sW[slot] & KEY_RARE))
                    continue;
                if (pbase == OWM_NONE) {  // no room: nobody may read a place for it
                    sW[slot] = nb << GRID_CELL_BITS;
                    continue;
                }
                const uint32_t at = pbase + atomicAdd(&s_nr, 1u);
                sPool[slot] = at;
                const AxisPassed px = axis_passed(T.ax[0], TREE ? G.xy[i].x : X[i]);
                const AxisPassed py = axis_passed(T.ax[1], TREE ? G.xy[i].y : Y[i]);
                const double zi = TREE ? G.zi[i].z : Z[i];
                GridRare r;
                r.zk = owm_eligible(zi) ? owm_zkey(zi) : OWM_ZKEY_NONE;
                r.id = TREE ? G.zi[i].id : i;
                r.pad = 0;
                r.wx0 = (uint16_t)px.w_lo;
                r.wx1 = (uint16_t)px.w_hi;
                r.wy0 = (uint16_t)py.w_lo;
                r.wy1 = (uint16_t)py.w_hi;
                r.gx0 = (uint16_t)px.g_lo;
                r.gx1 = (uint16_t)px.g_hi;
                r.gy0 = (uint16_t)py.g_lo;
                r.gy1 = (uint16_t)py.g_hi;
                G.pool[at] = r;
            }
            __syncthreads();
        }
#pragma unroll
        for (int k = 0; k < GP_K; ++k)
            if (key[k] == KEY_NONE && tid + k * GP_NT < cnt)
                key[k] = sW[tid + k * GP_NT];
        // the pool entry travels in place of the z key
#pragma unroll
        for (int k = 0; k < GP_K; ++k)
            if (tid + k * GP_NT < cnt && (key[k] & KEY_RARE))
                z[k] = __hiloint2double(0, (int)sPool[tid + k * GP_NT]);
    }
    uint32_t rank[GP_K];
#pragma unroll
    for (int k = 0; k < GP_K; ++k)
        rank[k] = tid + k * GP_NT < cnt && key[k] != nb << GRID_CELL_BITS
                      ? atomicAdd(&hist[(key[k] & ~KEY_RARE) >> GRID_CELL_BITS], 1u)
                      : 0u;
    __syncthreads();
    // exclusive offsets of the buckets, nb / GP_NT consecutive ones per thread
    const uint32_t per = (nb + GP_NT - 1) / GP_NT, b0 = min(tid * per, nb), b1 = min(b0 + per, nb);
    uint32_t sum = 0;
    for (uint32_t b = b0; b < b1; ++b)
        sum += hist[b];
    uint32_t total;
    uint32_t run = owm_block_scan<GP_NT>(sum, s_w, total);
    uint16_t *tab = G.tab + T.tab_off + (uint64_t)st * (nb + 1);
    for (uint32_t b = b0; b < b1; ++b) {
        const uint32_t h = hist[b];
        hist[b] = run;
        run += h;
    }
    if (tid == 0)
        hist[nb] = total;  // (the unwritten points share the place behind the others)
    __syncthreads();
    for (uint32_t b = tid; b <= nb; b += GP_NT)
        tab[b] = (uint16_t)hist[b];
#pragma unroll
    for (int k = 0; k < GP_K; ++k) {
        const uint32_t slot = tid + k * GP_NT;
        if (slot < cnt) {
            const uint32_t pos = hist[(key[k] & ~KEY_RARE) >> GRID_CELL_BITS] + rank[k];
            const unsigned long long zk = key[k] & KEY_RARE
                                              ? (unsigned long long)__double_as_longlong(z[k])
                                          : owm_eligible(z[k]) ? owm_zkey(z[k])
                                                               : OWM_ZKEY_NONE;
            sRec[3 * pos] = (uint32_t)zk;
            sRec[3 * pos + 1] = (uint32_t)(zk >> 32);
            sRec[3 * pos + 2] =
                (key[k] & KEY_RARE) | (key[k] & GRID_CELL_MASK) << GRID_SLOT_BITS | slot;
        }
    }
    __syncthreads();
    // four records are three 16-byte words; a tile's records start at a multiple
    // of four, and the words behind its last record are its own padding
    uint4 *out = (uint4 *)G.rec + ((uint64_t)T.rec_off + st * PTS) / 4 * 3;
    const uint32_t words = (total + 3) / 4 * 3;
    for (uint32_t i = tid; i < words; i += GP_NT)
        out[i] = s_part[i];
}

// ----------------------------------------------------------------- bins ----

constexpr int GB_RUNS = 1024;  // run segments per pass
constexpr int GB_SEG = 4;     // points per lane and segment
// 16 bytes of records, at any multiple of four bytes
struct __attribute__((packed, aligned(4))) RecWord {
    uint32_t x, y, z, w;
};
constexpr uint32_t GB_RARE = 512;   // points without a column listed before a flush

// Appends the listed pool entries to the item's chain of blocks {count, next
// block, entries}, whose head is kept in `head` (SUB: in memory, other workgroups
// append too).  Every thread of the workgroup calls it.
template <int NT, bool SUB>
__device__ __forceinline__ void flush_rare(const GridDev &G, uint32_t item, const uint32_t *list,
                                           uint32_t n, uint32_t *s_base, uint32_t &head)
{
    if (threadIdx.x == 0) {
        // (the first entry spreads an item's blocks over the shares: most listed points
        // may lie in one bucket)
        const uint32_t share = (item + list[0]) & (GRID_POOLS - 1u);
        const uint32_t at = atomicAdd(G.pool_used + share * 32 + 16, n + 2u);
        *s_base = at + n + 2u <= G.list_cap ? share * G.list_cap + at : OWM_NONE;
        if (*s_base == OWM_NONE) {
            atomicOr(G.err, GRID_ERR_POOL);
            G.err[SUB ? GRID_STOP_HEAVY : GRID_STOP_BIN] = 1u;
        }
    }
    __syncthreads();
    const uint32_t base = *s_base;
    if (base != OWM_NONE) {
        if (threadIdx.x == 0) {
            G.list[base] = n;
            G.list[base + 1] = SUB ? atomicExch(G.heads + item, base) : head;
        }
        for (uint32_t e = threadIdx.x; e < n; e += NT)
            G.list[base + 2 + e] = list[e];
        head = base;
    }
    __syncthreads();
}

// Queues an item's points in the sort tiles [s0, s0 + len), pts at most.  own: its
// owner, last group, number of stretches and tile.  Every thread of the workgroup calls it.
template <int NT>
__device__ __forceinline__ void queue_rest(const GridDev &G, const GridTile &T, uint32_t item,
                                           uint32_t s0, uint32_t len, uint32_t pts, uint32_t *own,
                                           uint32_t *s_base)
{
    const GridHeavy H(G, T.heavy_cap);
    const uint32_t ns = min((pts + T.heavy_sub - 1) / T.heavy_sub, len);
    if (threadIdx.x == 0) {
        const uint32_t at = atomicAdd(H.n, ns);
        const bool room = at + ns <= T.heavy_cap;
        *s_base = room ? at : OWM_NONE;
        if (room) {
            own[0] = min(own[0], at);
            H.grp[at] = make_uint2(ns, own[1]);
            own[1] = at;
            own[2] += ns;
        } else {
            atomicOr(G.err, GRID_ERR_POOL);
            G.err[GRID_STOP_BIN] = 1u;
        }
    }
    __syncthreads();
    const uint32_t at = *s_base, owner = own[0];
    if (at != OWM_NONE)
        for (uint32_t i = threadIdx.x; i < ns; i += NT)
            H.q[at + i] = make_uint4(item, s0 + len * i / ns, s0 + len * (i + 1) / ns, owner);
    __syncthreads();
}

// One workgroup per item: a bucket's runs in one share of the tile's sort tiles.
// Cells keep the count, the lowest z key and the lowest index at that key.  A
// round takes GB_SEG points per lane, without branches (a lane without a
// point, or whose point has no column, works on one spare cell), so that the
// round's LDS operations are in flight together: counts and key minima; after a
// barrier the points that still hold their cell's minimum, of which those that
// lowered it reset the index; after another the index minimum.
// Bound by instruction issue (64 % of the cycles issue vector instructions at
// 329M points) and, where runs are short, by the scattered loads: 12-byte records
// read four at a time by 16-byte loads took 120M points (runs of 8) from 0.94 to
// 0.83 ms against separate key and cell streams, two lanes a segment instead of
// four to eight 0.74, lane masks instead of bit sets 0.71 ms.  One spare cell for
// all idle lanes instead of one per lane: 3.1 instead of 1.3 ms (329M points).
//
// A share of more than T.heavy points (clouds with most points in a few square
// metres) would keep one workgroup busy long after the others: further stretches
// of its sort tiles are queued and binned by the launch below (SUB), each into
// cells of its own, which the last of an item's adds up.  95 % of 20M points in
// 5 m x 5 m: 64 -> 0.48 ms; density falling with the distance from a scanner:
// 0.66 -> 0.29 ms; clouds without such shares pay the empty launch and the test
// (20M points 100 -> 105 us, 120M 0.61 -> 0.64 ms).
template <int NT, bool TREE, bool SUB>
__device__ __forceinline__ void bin_range(const GridDev &G, uint32_t t, uint32_t item,
                                          uint32_t cells, uint32_t st0, uint32_t st1, uint4 *out)
{
    extern __shared__ unsigned long long s_bin[];
    unsigned long long *sZ = s_bin;                 // [cells + 64]
    uint32_t *sId = (uint32_t *)(sZ + cells + 64);  // [cells + 64]
    uint32_t *sCnt = sId + cells + 64;              // [cells + 64]
    __shared__ uint32_t s_base, s_nr, s_w[NT / 64], s_own[4];
    __shared__ uint2 sRun[GB_RUNS];
    __shared__ uint32_t sRare[GB_RARE];
    const uint32_t tid = threadIdx.x;
    if (tid == 0) {
        s_nr = 0;
        s_own[0] = s_own[1] = OWM_NONE;
        s_own[2] = 0;
        s_own[3] = t;
    }
    const GridTile &T = G.tiles[t];
    const uint32_t lc = T.lw + T.lh, nc = 1u << lc, pt_off = T.pt_off, rec_off = T.rec_off;
    const uint32_t bucket = (item - T.item_off) / T.split;
    const uint32_t nb1 = T.nb + 1, lpr = T.lpr, seg_pts = (uint32_t)GB_SEG << lpr;
    const uint32_t lsp = T.lsp;
    uint32_t left = T.heavy;  // points until the item is heavy
    for (uint32_t c = tid; c < nc + 64; c += NT) {
        sZ[c] = OWM_ZKEY_NONE;
        sId[c] = OWM_NONE;
        sCnt[c] = 0;
    }
    uint32_t head = OWM_NONE;
    const uint32_t spare = nc + (tid & 63);
    const uint32_t grp = tid >> lpr, ngrp = NT >> lpr;
    const uint32_t first = (tid & ((1u << lpr) - 1u)) * GB_SEG;  // the lane's points of a segment
    for (uint32_t s0 = st0; s0 < st1; s0 += NT) {
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
        const uint32_t at0 = owm_block_scan<NT>(nseg, s_w, total);
        if (!SUB) {
            const uint32_t pts = __builtin_amdgcn_readfirstlane(total) * seg_pts;
            if (__builtin_expect(pts > left, 0)) {
                queue_rest<NT>(G, T, item, s0, min((uint32_t)NT, st1 - s0), pts, s_own, &s_base);
                total = 0;
            } else {
                left -= pts;
            }
        }
        for (uint32_t p0 = 0; p0 < total; p0 += GB_RUNS) {
            for (uint32_t e = max(at0, p0); e < min(at0 + nseg, p0 + GB_RUNS); ++e) {
                const uint32_t a = o0 + (e - at0) * seg_pts;
                sRun[e - p0] = make_uint2((s << lsp) + a, min(seg_pts, o1 - a));
            }
            __syncthreads();
            const uint32_t here = min((uint32_t)GB_RUNS, total - p0);
            for (uint32_t r0 = 0; r0 < here; r0 += ngrp) {
                unsigned long long zk[GB_SEG], cur[GB_SEG];
                uint32_t cw[GB_SEG], cell[GB_SEG], all = 0;
                const uint2 run = r0 + grp < here ? sRun[r0 + grp] : make_uint2(0u, 0u);
                const uint32_t id0 = pt_off + (run.x >> lsp << lsp);
                RecWord w[3] = {};
                if (first < run.y) {
                    // four records in three loads (the last may hold the next
                    // run's, or the padding behind the tile's)
                    const RecWord *p =
                        (const RecWord *)(G.rec + ((uint64_t)rec_off + run.x + first) * 3);
                    w[0] = p[0];
                    w[1] = p[1];
                    w[2] = p[2];
                }
                const uint32_t v[12] = {w[0].x, w[0].y, w[0].z, w[0].w, w[1].x, w[1].y,
                                        w[1].z, w[1].w, w[2].x, w[2].y, w[2].z, w[2].w};
#pragma unroll
                for (int k = 0; k < GB_SEG; ++k) {
                    zk[k] = (unsigned long long)v[3 * k + 1] << 32 | v[3 * k];
                    cw[k] = first + k < run.y ? v[3 * k + 2] : KEY_NONE;
                }
#pragma unroll
                for (int k = 0; k < GB_SEG; ++k) {
                    cell[k] = min(cw[k] >> GRID_SLOT_BITS, spare);
                    all |= cw[k];
                    atomicAdd(&sCnt[cell[k]], 1u);
                    cur[k] = sZ[cell[k]];
                }
                bool low[GB_SEG], eq[GB_SEG];
#pragma unroll
                for (int k = 0; k < GB_SEG; ++k) {
                    low[k] = zk[k] < cur[k];
                    if (low[k])
                        atomicMin(&sZ[cell[k]], zk[k]);
                }
                uint32_t pend = 0;  // points without a column not listed: the list was full
                if ((int32_t)all < 0) {
#pragma unroll
                    for (int k = 0; k < GB_SEG; ++k)
                        if ((int32_t)cw[k] < 0) {
                            const uint32_t e = atomicAdd(&s_nr, 1u);
                            if (e < GB_RARE)
                                sRare[e] = (uint32_t)zk[k];
                            else
                                pend |= 1u << k;
                        }
                }
                __syncthreads();
                // (no thread appends between the two barriers: the test is uniform)
                if (s_nr > GB_RARE) {
                    do {
                        flush_rare<NT, SUB>(G, item, sRare, GB_RARE, &s_base, head);
                        if (tid == 0)
                            s_nr = 0;
                        __syncthreads();
#pragma unroll
                        for (int k = 0; k < GB_SEG; ++k)
                            if ((pend >> k) & 1u) {
                                const uint32_t e = atomicAdd(&s_nr, 1u);
                                if (e < GB_RARE) {
                                    sRare[e] = (uint32_t)zk[k];
                                    pend &= ~(1u << k);
                                }
                            }
                    } while (__syncthreads_or(pend != 0));
                }
#pragma unroll
                for (int k = 0; k < GB_SEG; ++k)
                    cur[k] = sZ[cell[k]];
#pragma unroll
                for (int k = 0; k < GB_SEG; ++k) {
                    eq[k] = zk[k] == cur[k];
                    if (eq[k] && low[k])
                        sId[cell[k]] = OWM_NONE;
                }
                __syncthreads();
#pragma unroll
                for (int k = 0; k < GB_SEG; ++k)
                    if (eq[k]) {
                        const uint32_t i = id0 + (cw[k] & GRID_SLOT_MASK);
                        // (idle lanes may point anywhere: theirs is the spare cell)
                        if (!TREE)
                            atomicMin(&sId[cell[k]], i);
                        else if (cell[k] < nc)
                            atomicMin(&sId[cell[k]], G.zi[i].id);
                    }
            }
            __syncthreads();  // sRun is rewritten
        }
    }
    __syncthreads();
    const uint32_t n_r = min(s_nr, GB_RARE);
    if (n_r)
        flush_rare<NT, SUB>(G, item, sRare, n_r, &s_base, head);
    if (!SUB && tid == 0) {
        G.heads[item] = head;
        if (s_own[0] != OWM_NONE)
            ((uint4 *)GridHeavy(G, T.heavy_cap).own)[s_own[0]] = make_uint4(s_own[1], s_own[2], 0u, s_own[3]);
    }
    if (!SUB)
        out = G.cells + T.cell_off + ((uint64_t)(item - T.item_off) << lc);
    for (uint32_t c = tid; c < nc; c += NT) {
        const unsigned long long zk = sZ[c];
        out[c] = make_uint4((uint32_t)zk, (uint32_t)(zk >> 32), sId[c], sCnt[c]);
    }
}

template <int NT, bool TREE>
__global__ __launch_bounds__(NT) void k_grid_bin(GridDev G, uint32_t t0, uint32_t t1,
                                                 uint32_t item0, uint32_t items, uint32_t cells)
{
    __shared__ uint32_t s_t;
    const uint32_t stop = G.err[GRID_STOP_PART];
    // consecutive items (neighbouring buckets, whose runs share cache lines)
    // on one XCD: workgroups go round the eight XCDs
    const uint32_t per = (items + 7u) / 8u;
    const uint32_t rel = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    if (rel >= items)
        return;
    const uint32_t item = item0 + rel;
    look_for_entry(G.item_off, t0, t1, item, &s_t);
    if (stop)  // (its load went beside the table's)
        return;
    const uint32_t t = entry_found(&s_t);
    const GridTile &T = G.tiles[t];
    const uint32_t q = item - T.item_off, part = q % T.split;
    bin_range<NT, TREE, false>(G, t, item, cells, (uint32_t)((uint64_t)T.nst * part / T.split),
                               (uint32_t)((uint64_t)T.nst * (part + 1) / T.split), nullptr);
}

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

// The queued stretches (none for most clouds: 4 us).
template <int NT, bool TREE>
__global__ __launch_bounds__(NT) void k_grid_heavy(GridDev G, uint32_t cap,
                                                   uint32_t cells)
{
    __shared__ uint32_t s_last;
    const uint32_t tid = threadIdx.x;
    // An overfull queue has entries that were never written.  (Not *G.err, which this
    // launch may set: a workgroup's waves that read it at different times could go
    // different ways, some into the barriers, some out.)
    if (G.err[GRID_STOP_PART] | G.err[GRID_STOP_BIN])
        return;
    const GridHeavy H(G, cap);
    const uint32_t n = min(*H.n, cap);
    for (uint32_t e = blockIdx.x; e < n; e += gridDim.x) {
        const uint4 v = H.q[e];
        uint32_t *own = H.own + 4 * v.w;
        const uint32_t t = own[3];
        bin_range<NT, TREE, true>(G, t, v.x, cells, v.y, v.z, H.cells + (uint64_t)e * cells);
        // the last of the item's adds them up: every wave's stores have reached
        // the L2, the fence makes them visible beyond this XCD
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0) {
            __threadfence();
            s_last = atomicAdd(own + 2, 1u) + 1u == own[1];
        }
        __syncthreads();
        const bool last = s_last;
        if (last) {
            __threadfence();
            const GridTile &T = G.tiles[t];
            const uint32_t lc = T.lw + T.lh;
            uint4 *out = G.cells + T.cell_off + ((uint64_t)(v.x - T.item_off) << lc);
            for (uint32_t c = tid; c < 1u << lc; c += NT) {
                const uint4 o = out[c];
                CellAgg a = {(unsigned long long)o.y << 32 | o.x, o.z, o.w};
                for (uint32_t g = own[0]; g != OWM_NONE;) {
                    const uint2 grp = H.grp[g];
                    const uint4 *p = H.cells + (uint64_t)g * cells + c;
#pragma unroll 4
                    for (uint32_t k = 0; k < grp.x; ++k) {
                        const uint4 w = p[(uint64_t)k * cells];
                        agg_add(a, (unsigned long long)w.y << 32 | w.x, w.z, w.w);
                    }
                    g = grp.y;
                }
                out[c] = make_uint4((uint32_t)a.zk, (uint32_t)(a.zk >> 32), a.id, a.cnt);
            }
        }
        __syncthreads();  // s_last and the cells in LDS are rewritten
    }
}

// -------------------------------------------------------------- windows --

constexpr int GW_NT = 512;
constexpr uint32_t GW_SEGS = 512;  // pool blocks a window block can meet
constexpr int GW_PER = 32 * 32 / GW_NT;  // windows per thread, at most

// The cell of column c and row r in its bucket's first share (the others follow
// at the bucket's size).
__device__ __forceinline__ const uint4 *cell_ptr(const GridDev &G, const GridTile &T, uint32_t c,
                                                 uint32_t r)
{
    const uint32_t k = grid_key(T, c, r);
    return G.cells + T.cell_off + ((uint64_t)(k >> GRID_CELL_BITS) * T.split << (T.lw + T.lh)) +
           (k & GRID_CELL_MASK);
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
    const double2 xy = G.pos ? G.xy[G.pos[id]] : make_double2(X[id], Y[id]);
    const double x = xy.x, y = xy.y;
    const uint32_t x0 = axis_count(T.ax[0].g, x, true, true), x1 = axis_count(T.ax[0].g, x, false, false);
    const uint32_t y0 = axis_count(T.ax[1].g, y, true, true), y1 = axis_count(T.ax[1].g, y, false, false);
    for (uint32_t j = y0; j < y1; ++j)
        for (uint32_t i = x0; i < x1; ++i)
            G.cell_flag[T.gcell_off + j * T.ax[0].g.n + i] = 1u;
}

// One workgroup per block of bw x bw windows: its columns x rows of cells go to
// LDS (each read once, the shares of a bucket summed), every row is reduced to
// the window columns in place, then the rows to windows, then come the listed
// points and stage 2's marks.  Bound by latency, a chain of dependent steps per
// block: 329M points in 512 tiles 0.48 ms with row sums taken from memory, 0.34
// through LDS with 512 threads and the windows' columns from a table (0.56 with
// 256 threads that computed them); 120M points in shares of 32768: 0.27 -> 0.08.
__global__ __launch_bounds__(GW_NT) void k_grid_windows(GridDev G, const double *__restrict__ X,
                                                         const double *__restrict__ Y,
                                                         uint32_t cells_cap)
{
    extern __shared__ unsigned long long s_win[];
    __shared__ uint32_t s_t, s_nseg;
    __shared__ int sx0[32], sx1[32], sy0[32], sy1[32];
    __shared__ uint2 sSeg[GW_SEGS];
    const uint32_t tid = threadIdx.x;
    const uint32_t stop = G.err[GRID_STOP_PART] | G.err[GRID_STOP_BIN] | G.err[GRID_STOP_HEAVY];
    if (tid == 0)
        s_nseg = 0;
    look_for_entry(G.blk_off, 0, G.ntiles, blockIdx.x, &s_t);
    if (stop)
        return;
    const uint32_t t = entry_found(&s_t);
    const GridTile &T = G.tiles[t];
    const uint32_t lb = T.lbw, bw = 1u << lb;
    const uint32_t q0 = blockIdx.x - T.blk_off, bj = q0 / T.nblkx, bi = q0 - bj * T.nblkx;
    const uint32_t nx = T.ax[0].w.n, ny = T.ax[1].w.n;
    const uint32_t i0 = bi << lb, j0 = bj << lb;
    const uint32_t ni = min(bw, nx - i0), nj = min(bw, ny - j0);
    const int2 *cols = G.wcols + G.axis_off[t];
    if (tid < ni) {
        const int2 v = cols[i0 + tid];
        sx0[tid] = v.x;
        sx1[tid] = v.y;
    } else if (tid >= 64 && tid - 64 < nj) {
        const int2 v = cols[nx + j0 + tid - 64];
        sy0[tid - 64] = v.x;
        sy1[tid - 64] = v.y;
    }
    __syncthreads();
    const int c0 = sx0[0], c1 = sx1[ni - 1], r0 = sy0[0], r1 = sy1[nj - 1];
    // pitch: a row of cells, and later of window columns
    const uint32_t nc = c1 >= c0 ? (uint32_t)(c1 - c0 + 1) : 0u, pitch = max(nc, bw);
    uint32_t nr = r1 >= r0 ? (uint32_t)(r1 - r0 + 1) : 0u;
    unsigned long long *mZ = s_win;  // [cells_cap]
    uint32_t *mId = (uint32_t *)(mZ + cells_cap);
    uint32_t *mCnt = mId + cells_cap;
    if (nr * pitch > cells_cap) {  // cannot happen (the host sizes cells_cap)
        if (tid == 0)
            atomicOr(G.err, GRID_ERR_ROWS);
        nr = 0;
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
                const uint32_t n = G.list[h], next = G.list[h + 1];
                const uint32_t e = atomicAdd(&s_nseg, 1u);
                if (e >= GW_SEGS) {
                    atomicOr(G.err, GRID_ERR_POOL);
                    break;
                }
                sSeg[e] = make_uint2(h + 2, n);
                h = next;
            }
        }
    }
    // four cells per thread in flight
    for (uint32_t q0 = tid; q0 < nr * nc; q0 += 4 * GW_NT) {
        const uint4 *p[4];
        uint4 v[4];
        uint32_t at[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const uint32_t q = min(q0 + u * GW_NT, nr * nc - 1u), rr = q / nc, c = q - rr * nc;
            p[u] = cell_ptr(G, T, (uint32_t)c0 + c, (uint32_t)r0 + rr);
            v[u] = *p[u];
            at[u] = rr * pitch + c;
        }
        if (T.split > 1) {
            CellAgg a[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                a[u] = {(unsigned long long)v[u].y << 32 | v[u].x, v[u].z, v[u].w};
            for (uint32_t k = 1; k < T.split; ++k) {
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    v[u] = p[u][k << (T.lw + T.lh)];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    agg_add(a[u], (unsigned long long)v[u].y << 32 | v[u].x, v[u].z, v[u].w);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                v[u] = make_uint4((uint32_t)a[u].zk, (uint32_t)(a[u].zk >> 32), a[u].id, a[u].cnt);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (q0 + u * GW_NT < nr * nc) {
                mZ[at[u]] = (unsigned long long)v[u].y << 32 | v[u].x;
                mId[at[u]] = v[u].z;
                mCnt[at[u]] = v[u].w;
            }
    }
    __syncthreads();
    if (s_nseg > GW_SEGS)  // (flagged above)
        return;
    // rows to window columns: a row belongs to bw lanes of one wave, whose
    // reads of it all precede its writes
    for (uint32_t rr = tid >> lb; rr < nr; rr += GW_NT >> lb) {
        const uint32_t w = tid & (bw - 1u), m = rr * pitch;
        CellAgg a = {OWM_ZKEY_NONE, OWM_NONE, 0};
        if (w < ni)
            for (int c = sx0[w] - c0; c <= sx1[w] - c0; ++c)
                agg_add(a, mZ[m + c], mId[m + c], mCnt[m + c]);
        __builtin_amdgcn_wave_barrier();
        mZ[m + w] = a.zk;
        mId[m + w] = a.id;
        mCnt[m + w] = a.cnt;
    }
    __syncthreads();
    CellAgg win[GW_PER];
#pragma unroll
    for (int k = 0; k < GW_PER; ++k) {
        const uint32_t q = tid + k * GW_NT, v = q >> lb, w = q & (bw - 1u);
        win[k] = {OWM_ZKEY_NONE, OWM_NONE, 0};
        if (v < nj && w < ni && nr)
            for (int r = sy0[v] - r0; r <= sy1[v] - r0; ++r)
                agg_add(win[k], mZ[r * pitch + w], mId[r * pitch + w], mCnt[r * pitch + w]);
    }
    __syncthreads();  // the row sums are no longer needed: their memory holds the windows
    const uint32_t nseg = s_nseg;
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
                const GridRare r = G.pool[G.list[sSeg[sg].x + e]];
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
                const GridRare r = G.pool[G.list[sSeg[sg].x + e]];
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
            const bool in = (q >> lb) < nj && (q & (bw - 1u)) < ni;
            win[k].id = valid && in ? win[k].id : OWM_NONE;
            sMin[q] = win[k].id;
            if (G.min_ids && in)
                G.min_ids[(uint64_t)(j0 + (q >> lb)) * nx + i0 + (q & (bw - 1u))] = win[k].id;
        }
    }
    if (G.min_ids)
        return;
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
    const uint32_t stop = *G.err;  // (this launch sets none)
    for (uint32_t c = blockIdx.x * 4 + w; c < G.ngcell; c += gridDim.x * 4) {
        if (G.cell_flag[c] | stop)
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
                const uint4 *p = cell_ptr(G, T, (uint32_t)c0 + (q - r * nc), (uint32_t)r0 + r);
                for (uint32_t k = 0; k < T.split; ++k, p += 1u << (T.lw + T.lh)) {
                    const uint4 v = *p;
                    agg_add(a, (unsigned long long)v.y << 32 | v.x, v.z, v.w);
                }
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
                    const uint32_t n = G.list[at], next = G.list[at + 1];
                    for (uint32_t e = lane; e < n; e += 64) {
                        const GridRare r = G.pool[G.list[at + 2 + e]];
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

void launch_grid_prep(hipStream_t s, const GridDev &G, const FillRanges &r, uint32_t windows,
                      const uint32_t *host_table, uint32_t table_words)
{
    uint64_t most = windows;
    for (uint32_t k = 0; k < r.count; ++k)
        most = r.len[k] > most ? r.len[k] : most;
    const uint64_t g = (most + 1023) / 1024;  // four words a thread, up to 2048 blocks
    hipLaunchKernelGGL(k_grid_prep,
                       dim3((uint32_t)(g < 1 ? 1 : g > 2048 ? 2048 : g),
                            r.count + (host_table ? 2 : 1)),
                       dim3(256), 0, s, G, r, windows, host_table, table_words);
}

void launch_grid_part(hipStream_t s, const GridDev &G, const double *x, const double *y,
                      const double *z, uint32_t sort_tiles, uint32_t lsp, uint32_t max_nb)
{
    if (!sort_tiles)
        return;
    const uint32_t lds = (12u << lsp) + (max_nb + 1) * 4u;
    const auto k = lsp == 10 ? (G.zi ? k_grid_part<true, 10> : k_grid_part<false, 10>)
                   : lsp == 13 ? k_grid_part<false, 13>  // (no tree of that size comes here)
                   : lsp == 11 ? (G.zi ? k_grid_part<true, 11> : k_grid_part<false, 11>)
                               : (G.zi ? k_grid_part<true, 12> : k_grid_part<false, 12>);
    hipLaunchKernelGGL(k, dim3(sort_tiles), dim3(gp_threads(lsp)), lds, s, G, x, y, z);
}

// LDS of the bins: the cells and 64 spare ones.
static constexpr int BIN_LDS(uint32_t cells) { return (int)(cells + 64u) * 16; }

void launch_grid_bin(hipStream_t s, const GridDev &G, uint32_t t0, uint32_t t1, uint32_t item0,
                     uint32_t items, uint32_t cells)
{
    if (!items)
        return;
    const uint32_t g = (items + 7u) / 8u * 8u;
    // 512 threads where LDS or the number of items leaves few workgroups to a CU
    // (120M points, 64 KB of cells: 1.50 ms with 256 threads, 1.13 with 512; 1M
    // points: 29 and 21 us; 329M points in 27,700 items: 1.00 and 1.04 ms)
    const bool wide = cells > 1024 || items <= 1024;
    const dim3 grid(g), block(wide ? 512 : 256);
    if (G.zi && wide)
        hipLaunchKernelGGL((k_grid_bin<512, true>), grid, block, BIN_LDS(cells), s, G, t0, t1,
                           item0, items, cells);
    else if (G.zi)
        hipLaunchKernelGGL((k_grid_bin<256, true>), grid, block, BIN_LDS(cells), s, G, t0, t1,
                           item0, items, cells);
    else if (wide)
        hipLaunchKernelGGL((k_grid_bin<512, false>), grid, block, BIN_LDS(cells), s, G, t0, t1,
                           item0, items, cells);
    else
        hipLaunchKernelGGL((k_grid_bin<256, false>), grid, block, BIN_LDS(cells), s, G, t0, t1,
                           item0, items, cells);
}

void launch_grid_heavy(hipStream_t s, const GridDev &G, uint32_t cap, uint32_t cells)
{
    const auto k = G.zi ? k_grid_heavy<512, true> : k_grid_heavy<512, false>;
    hipLaunchKernelGGL(k, dim3(std::min(cap, 256u)), dim3(512), BIN_LDS(cells), s, G, cap,
                       cells);
}

void launch_grid_windows(hipStream_t s, const GridDev &G, const double *x, const double *y,
                         uint32_t blocks, uint32_t cells_cap)
{
    if (!blocks)
        return;
    hipLaunchKernelGGL(k_grid_windows, dim3(blocks), dim3(GW_NT), cells_cap * 16u, s, G, x, y,
                       cells_cap);
}

void launch_grid_cells(hipStream_t s, const GridDev &G)
{
    if (!G.ngcell)
        return;
    uint32_t g = (G.ngcell + 3) / 4;
    g = g > 16384 ? 16384 : g;
    hipLaunchKernelGGL(k_grid_cells, dim3(g), dim3(256), 0, s, G);
}

__global__ void k_flags_out(const uint32_t *flags, uint32_t *host) { *host = *flags; }

void launch_flags_out(hipStream_t s, const uint32_t *flags, uint32_t *host)
{
    hipLaunchKernelGGL(k_flags_out, dim3(1), dim3(1), 0, s, flags, host);
}

// LDS of more than 64 KB per workgroup is taken by dynamic size alone on
// gfx950; the attribute tells the runtime to expect it.
hipError_t grid_kernels_init()
{
    const std::pair<const void *, int> k[] = {
        {(const void *)k_grid_part<false, 10>, (12 << 10) + (GRID_MAX_BUCKETS + 1) * 4},
        {(const void *)k_grid_part<true, 10>, (12 << 10) + (GRID_MAX_BUCKETS + 1) * 4},
        {(const void *)k_grid_part<false, 11>, (12 << 11) + (GRID_MAX_BUCKETS + 1) * 4},
        {(const void *)k_grid_part<true, 11>, (12 << 11) + (GRID_MAX_BUCKETS + 1) * 4},
        {(const void *)k_grid_part<false, 12>, (12 << 12) + (GRID_MAX_BUCKETS + 1) * 4},
        {(const void *)k_grid_part<true, 12>, (12 << 12) + (GRID_MAX_BUCKETS + 1) * 4},
        {(const void *)k_grid_part<false, 13>, (12 << 13) + (GRID_MAX_BUCKETS + 1) * 4},
        {(const void *)k_grid_bin<256, false>, BIN_LDS(GRID_MAX_CELLS)},
        {(const void *)k_grid_bin<512, false>, BIN_LDS(GRID_MAX_CELLS)},
        {(const void *)k_grid_bin<256, true>, BIN_LDS(GRID_MAX_CELLS)},
        {(const void *)k_grid_bin<512, true>, BIN_LDS(GRID_MAX_CELLS)},
        {(const void *)k_grid_heavy<512, false>, BIN_LDS(GRID_MAX_CELLS)},
        {(const void *)k_grid_heavy<512, true>, BIN_LDS(GRID_MAX_CELLS)},
        {(const void *)k_grid_windows, GRID_MAX_WIN_CELLS * 16}};
    for (const auto &f : k) {
        const hipError_t e =
            hipFuncSetAttribute(f.first, hipFuncAttributeMaxDynamicSharedMemorySize, f.second);
        if (e != hipSuccess)
            return e;
    }
    return hipSuccess;
}

}  // namespace owm
