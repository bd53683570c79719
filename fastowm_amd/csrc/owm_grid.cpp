// Host side of the column-grid chain (grid.hip): whole runs of tiles whose
// trees nobody keeps.  Plans each tile's column grid (owm_axis.h), buckets and
// work items, enqueues the chain and reads the seeds back.  Calls that it does
// not take go on to the tree chain (run_batch), with the boxes it took.
#include "owm_host.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>

namespace owm {

static inline uint64_t up256(uint64_t v) { return (v + 255) / 256 * 256; }

// The plan of one call: the device table and its totals.  Entries are ordered
// by the size class of their buckets' cells, so that each class is one launch
// of the bins with LDS for its own largest bucket.
struct GridPlan {
    std::vector<GridTile> t;
    std::vector<uint32_t> st_off, item_off, blk_off, gcell_off, axis_off;
    std::vector<uint32_t> pt_off;  // caller's tile order
    struct Class {
        uint32_t t0, t1, cells;
    };
    std::vector<Class> cls;
    uint64_t np = 0, recs = 0, cells = 0, tab = 0, nwin = 0, nleaf = 0, pool_cap = 0, list_cap = 0;
    uint32_t max_nb = 1, win_cells = 1024, heavy_cap = 0, heavy_cells = 0, many_cap = 0;
};

// Bucket cells up to which tiles share a launch of the bins: the LDS of the
// largest bucket of a launch bounds the workgroups per CU for all of them.
static int cell_class(uint32_t cells) { return cells <= 1024 ? 0 : cells <= 4096 ? 1 : 2; }

// Sort tiles of 2^lsp points, and what follows from them.
static void sort_tiles(GridTile &T, uint32_t lsp)
{
    T.lsp = lsp;
    T.nst = (uint32_t)((T.n + (1ull << T.lsp) - 1) >> T.lsp);
    const uint64_t mean = T.n / T.nb;
    // A bucket's points beyond 32768 are shared out: more workgroups, more partial
    // cells for the windows to add up (120M points: bins + windows 0.90 ms with
    // 16384, 0.69 with 32768, 0.75 with 65536).
    T.split = (uint32_t)std::min<uint64_t>(std::max<uint64_t>(mean / 32768, 1), 16);
    // A lane reads four consecutive points of a run, a segment is 2^lpr lanes:
    // small segments waste the fewest lanes at the ends of runs, larger ones cost
    // fewer list entries (10k points in 16 buckets: 19 us with one lane, 13 with
    // two; 96 mixed tiles: 0.67 ms with one, 0.69 with two, 0.72 with four; 100M
    // points in runs of three: 1.01 ms with one, 0.87 with two).
    const double run = T.nst ? (double)T.n / ((double)T.nst * T.nb) : 1.0;
    T.lpr = run <= 6.0 && T.n <= (8u << 20) ? 0 : run <= 64.0 ? 1 : run <= 128.0 ? 2 : 3;
    // An item is heavy at three times the mean (counted in whole segments), and not
    // below 65536 points: some 70 us of a workgroup's time.
    const double mean_item = ((double)mean + (double)T.nst * (2 << T.lpr)) / T.split;
    T.heavy = (uint32_t)std::max(65536.0, 3.0 * mean_item);
}

// Fills one tile's grid; false when the chain does not take it.
static bool plan_tile(GridTile &T, const owm_params &P, const Derived &D, uint64_t n,
                      uint64_t launch_points, uint32_t lsp)
{
    memset(&T, 0, sizeof T);
    T.n = (uint32_t)n;
    // the integer products of stage 3's centres must not wrap
    if (D.width >= 1e9 || D.height >= 1e9 || !D.ncols || !D.nrows)
        return false;
    const double hd = (double)(float)D.h, hb = (double)(float)D.hb;
    const double init[2] = {D.initx, D.inity}, initg[2] = {D.initxg, D.inityg};
    const uint32_t nw[2] = {D.ncols, D.nrows}, ng[2] = {D.ncolsg, D.nrowsg};
    for (int a = 0; a < 2; ++a) {
        grid_edges(T.ax[a].w, init[a], D.displace, hd, nw[a], false, 64);
        grid_edges(T.ax[a].g, initg[a], P.bsize ? (double)P.bsize : 1.0, hb, ng[a], true, 1);
        grid_axis(T.ax[a]);
        // coordinates so far from zero, in steps, that the arithmetic decides for few of
        // the points (and that axis_cols_of would not bound, further out)
        if (T.ax[a].w.tol > 0.125 || T.ax[a].g.tol > 0.125)
            return false;
    }
    T.min_num_points = D.min_num_points;
    T.stage2_need = P.overlap != 0.0 ? 2u : 1u;
    // Buckets: the smallest power-of-two rectangle of cells that leaves at most
    // this many of them.  More buckets give a small launch more workgroups (1M
    // points: bins 21 us with 8192 points a bucket, 11 us with 2048); fewer give
    // a large one longer runs, which cost fewer loads (20M points: 129 us with
    // 900 buckets, 98 us with 450, 84 with 225; 12M points: 70 and 64 us with 512
    // and 256) and fewer items (512 tiles, 329M points: 1.05 ms with 4096 points a
    // bucket, 0.99 ms with 8192).
    const uint32_t cx = T.ax[0].ncol, cy = T.ax[1].ncol;
    auto buckets = [&](uint32_t lw, uint32_t lh) {
        return ((uint64_t)(cx - 1) / (1u << lw) + 1) * ((uint64_t)(cy - 1) / (1u << lh) + 1);
    };
    const uint64_t per = launch_points <= (2u << 20) ? 2048 : launch_points <= (16u << 20) ? 4096 : 8192;
    const uint64_t want = std::min<uint64_t>(std::max<uint64_t>(n / per, 16), launch_points <= (8u << 20) ? 512 : 256);
    uint32_t lw = 3, lh = 3;
    while (buckets(lw, lh) > want && lw + lh < 12)
        (lw <= lh ? lw : lh) += 1;
    if (buckets(lw, lh) > GRID_MAX_BUCKETS)
        ++lw;
    if (buckets(lw, lh) > GRID_MAX_BUCKETS)
        return false;
    T.lw = lw;
    T.lh = lh;
    T.nbx = (cx - 1) / (1u << lw) + 1;
    T.nby = (cy - 1) / (1u << lh) + 1;
    T.nb = T.nbx * T.nby;
    sort_tiles(T, lsp);
    return true;
}

// An upper bound on the tree chain's device memory for the same call: a call
// that might not fit the budget there keeps that chain's answer.
static uint64_t tree_chain_bound(const GridPlan &P)
{
    return P.np * 112 + P.nleaf * 1000 + P.nwin * 32 + (64ull << 20);
}

static bool make_plan(owm_ctx *ctx, const owm_tile *tiles, uint32_t n_tiles,
                      const std::vector<std::array<double, 4>> &box, GridPlan &P)
{
    std::vector<GridTile> raw(n_tiles);
    uint64_t launch_points = 0;
    for (uint32_t t = 0; t < n_tiles; ++t)
        launch_points += tiles[t].n;
    // Sort tiles: 4096 points; a small launch takes its points in more workgroups of
    // less work each (10k points: partition 14.8 -> 9.6 us with 1024; 300k points: 14.8
    // -> 11.2 with 2048, bins 12.0 -> 11.9; 1M points: 16.7 -> 14.1, but bins 12.1 ->
    // 12.9 for the shorter runs, 102 us a run with either).
    uint32_t lsp = launch_points <= (1u << 17) ? 10 : launch_points <= (1u << 19) ? 11 : 12;
    P.pt_off.assign(n_tiles + 1, 0);
    for (uint32_t t = 0; t < n_tiles; ++t) {
        Derived D;
        std::string why;
        if (derive_params(tiles[t].params, tiles[t].n, box[t].data(), D, why) != OWM_OK)
            return false;  // the tree chain reports it
        if (!plan_tile(raw[t], tiles[t].params, D, tiles[t].n, launch_points, lsp))
            return false;
        raw[t].pt_off = P.pt_off[t];
        P.pt_off[t + 1] = P.pt_off[t] + (uint32_t)tiles[t].n;
        P.nwin += (uint64_t)D.ncols * D.nrows;
        P.nleaf += tiles[t].n / std::max(pick_leaf(ctx, tiles[t].n, 0), 1u) + 1;
    }
    // 8192 points where the runs of every tile would be short, in launches that fill
    // the device often (a workgroup has a CU to itself): partition and bins, 100M
    // points in runs of three 654 + 882 us with 4096, 733 + 595 with 8192; 120M in
    // runs of eight 805 + 637 and 869 + 492; 40M in runs of six 252 + 251 and 308 +
    // 199; 20M in runs of twenty 123 + 85 and 173 + 70.  341 buckets and more share a
    // sort tile of 4096 in runs of twelve and less, between the eight where the larger
    // tiles win and the twenty where they lose.
    bool brief = launch_points >= (48u << 20);
    for (const GridTile &T : raw)
        brief = brief && (T.n == 0 || T.nb > 341);
    if (brief)
        for (GridTile &T : raw)
            sort_tiles(T, 13);
    P.np = P.pt_off[n_tiles];
    // blocks of 32x32 windows where there are enough of them to occupy the
    // device and their cells fit (48 KB), else smaller
    uint64_t big = 0;
    for (const GridTile &T : raw)
        big += ((T.ax[0].w.n + 31ull) / 32) * ((T.ax[1].w.n + 31ull) / 32);
    for (GridTile &T : raw) {
        T.lbw = big < 512 || !T.ax[0].w.pair || !T.ax[1].w.pair ? 4 : 5;
        double cells;
        for (;; --T.lbw) {
            const uint32_t bw = 1u << T.lbw;
            cells = axis_cols_of(T.ax[1], bw) * std::max<double>(axis_cols_of(T.ax[0], bw), bw);
            if (cells <= 3072.0 || T.lbw == 3)
                break;
        }
        if (cells > GRID_MAX_WIN_CELLS)
            return false;  // window sides of very many steps
        P.win_cells = std::max(P.win_cells, (uint32_t)cells);
    }
    for (int c = 0; c < 3; ++c) {
        const uint32_t t0 = (uint32_t)P.t.size();
        uint32_t cells = 0;
        for (const GridTile &T : raw)
            if (cell_class(1u << (T.lw + T.lh)) == c) {
                P.t.push_back(T);
                cells = std::max(cells, 1u << (T.lw + T.lh));
            }
        if (P.t.size() > t0)
            P.cls.push_back({t0, (uint32_t)P.t.size(), cells});
    }
    P.st_off.assign(n_tiles + 1, 0);
    P.item_off.assign(n_tiles + 1, 0);
    P.blk_off.assign(n_tiles + 1, 0);
    P.gcell_off.assign(n_tiles + 1, 0);
    P.axis_off.assign(n_tiles + 1, 0);
    uint64_t st = 0, items = 0, blk = 0, gc = 0;
    for (uint32_t t = 0; t < n_tiles; ++t) {
        GridTile &T = P.t[t];
        T.st_off = (uint32_t)st;
        T.rec_off = (uint32_t)P.recs;
        P.recs += (T.n + 3ull) / 4 * 4;
        T.item_off = (uint32_t)items;
        T.blk_off = (uint32_t)blk;
        T.gcell_off = (uint32_t)gc;
        T.tab_off = P.tab;
        T.cell_off = P.cells;
        T.nblkx = ((T.ax[0].w.n - 1) >> T.lbw) + 1;
        st += T.nst;
        items += (uint64_t)T.nb * T.split;
        blk += (uint64_t)T.nblkx * (((T.ax[1].w.n - 1) >> T.lbw) + 1);
        gc += (uint64_t)T.ax[0].g.n * T.ax[1].g.n;
        P.tab += (uint64_t)T.nst * (T.nb + 1);
        P.cells += (uint64_t)T.nb * T.split << (T.lw + T.lh);
        if (items >= (1ull << 30) || blk >= (1ull << 30) || gc >= (1ull << 30))
            return false;
        P.st_off[t + 1] = (uint32_t)st;
        P.item_off[t + 1] = (uint32_t)items;
        P.blk_off[t + 1] = (uint32_t)blk;
        P.gcell_off[t + 1] = (uint32_t)gc;
        P.axis_off[t + 1] = P.axis_off[t] + T.ax[0].w.n + T.ax[1].w.n;
        P.max_nb = std::max(P.max_nb, T.nb);
    }
    if (P.nwin >= (1ull << 31))
        return false;  // the tree chain refuses it
    // heavy stretches: 256 of the whole launch's points, their share of the ends
    // of groups and of segments that are not full
    for (const GridTile &T : P.t) {
        P.heavy_cells = std::max(P.heavy_cells, 1u << (T.lw + T.lh));
        if (T.n > T.heavy)
            P.heavy_cap = (uint32_t)std::min<uint64_t>(64 + P.np / 8192, 2048);
    }
    for (GridTile &T : P.t) {
        if (!P.heavy_cap)  // (by the estimate a small tile's item may seem heavy)
            T.heavy = ~0u;
        T.heavy_sub = (uint32_t)std::max<uint64_t>(16384, P.np / 256);
        T.heavy_cap = P.heavy_cap;
    }
    // A quarter of the points may lie on edges before the tree chain takes over.  The
    // end of a share that a sort tile's points do not fit is lost, so every share has
    // room for one more; the lists' blocks are spread by chance, over twice the words.
    P.pool_cap = (P.np / 4 + 65536) / GRID_POOLS + (1u << P.t[0].lsp);
    P.list_cap = 2 * P.pool_cap + 2 * (items / GRID_POOLS + 1) + 1024;
    // A point without a column costs the windows 0.3 ns and more, ten times what the
    // chain takes for another, so beyond 4M points (where launches no longer bound the
    // tree chain) clouds with more than a sixth of them are the tree chain's (windows of
    // 5 m a metre apart, 12 % and 18 % of the points on edges: 8M points 0.66 and
    // 0.87 ms against 0.85 and 0.87 by the tree chain, 40M points 2.96 and 4.02
    // against 3.38 and 3.53).  A quarter of the sort tiles must say so: a raster's are
    // uneven (a line of it on an edge), and a part of a cloud may be gridded.
    P.many_cap = P.np > (4u << 20) ? (uint32_t)(st / 4) + 8u : ~0u;
    return true;
}

// The chain's results in page-locked host memory: count and error flags, tile
// ranges, the first indices (most calls' all: no copy follows the chain), and
// before it the boxes.
struct GridIo {
    static constexpr uint32_t IDS = 65536;
    uint32_t *head = nullptr, *off = nullptr, *ids = nullptr;
    double *box = nullptr;
    GridIo(owm_ctx *ctx, uint32_t n_tiles)
    {
        const uint64_t o = 256 + up256((n_tiles + 1) * 4ull), i = o + IDS * 4ull;
        uint8_t *h = ctx->pinned(ctx->h_io, ctx->h_io_cap,
                                 std::max<uint64_t>(i + n_tiles * 32ull, io_bytes(n_tiles)));
        if (!h)
            return;
        head = (uint32_t *)h;
        off = (uint32_t *)(h + 256);
        ids = (uint32_t *)(h + o);
        box = (double *)(h + i);
    }
};

// Boxes of at most BOX_TILES tiles: one launch that leaves them in io.box.
static owm_status take_few_boxes(owm_ctx *ctx, const double *dx, const double *dy,
                                 const owm_tile *tiles, uint32_t n_tiles, const GridIo &io,
                                 std::vector<std::array<double, 4>> &box)
{
    hipStream_t s = ctx->stream;
    if (!ctx->box_work.ptr) {
        HIP_TRY(ctx->grow(ctx->box_work, box_work_bytes()), "box work");
        launch_fill_u32(s, (uint32_t *)ctx->box_work.ptr, BOX_TILES, 0u);
    }
    BoxArgs a{};
    a.ntiles = n_tiles;
    uint64_t np = 0, want = 0;
    auto needed = [&](uint32_t t) {
        return tiles[t].n && !(tiles[t].params.flags & OWM_F_HAVE_BBOX);
    };
    for (uint32_t t = 0; t < n_tiles; ++t)
        if (needed(t)) {
            np += tiles[t].n;
            want += (tiles[t].n + BOX_POINTS - 1) / BOX_POINTS;
        }
    // a workgroup per BOX_POINTS points, and no more than four to a CU (their
    // tickets are atomics on one word)
    const double scale = want > 1024 ? 1024.0 / (double)want : 1.0;
    for (uint32_t t = 0; t < n_tiles; ++t) {
        uint32_t g = 0;
        if (needed(t))
            g = std::max(1u, (uint32_t)((double)((tiles[t].n + BOX_POINTS - 1) / BOX_POINTS) * scale));
        a.pt[t + 1] = a.pt[t] + (uint32_t)tiles[t].n;
        a.blk[t + 1] = a.blk[t] + g;
    }
    if (a.blk[n_tiles]) {
        const int pi = ctx->prof.begin(s, PH_BBOX);
        launch_boxes(s, a, dx, dy, ctx->box_work.ptr, io.box);
        ctx->prof.end(s, pi, 16ull * np, np);
        HIP_TRY(hipGetLastError(), "box launch");
        HIP_TRY(hipStreamSynchronize(s), "bbox sync");
        ctx->prof.collect();
    }
    for (uint32_t t = 0; t < n_tiles; ++t) {
        if (tiles[t].params.flags & OWM_F_HAVE_BBOX)
            continue;
        const double *b = io.box + 4 * t;  // min x, min y, max x, max y
        if (tiles[t].n == 0 || !(b[0] <= b[2]) || !(b[1] <= b[3])) {
            set_err(ctx, "tile %u: no finite points to take a bbox from", t);
            return OWM_E_ARG;
        }
        box[t] = {b[0], b[2], b[1], b[3]};
    }
    return OWM_OK;
}

// Exact boxes of the tiles that come without one (device reduction).
static owm_status take_boxes(owm_ctx *ctx, const double *dx, const double *dy,
                             const owm_tile *tiles, uint32_t n_tiles,
                             std::vector<std::array<double, 4>> &box)
{
    hipStream_t s = ctx->stream;
    uint64_t np = 0;
    for (uint32_t t = 0; t < n_tiles; ++t)
        np += tiles[t].n;
    const uint64_t bk_bytes = bbox_key_words(n_tiles) * 8, off_bytes = (n_tiles + 1) * 4ull;
    owm_status st = ctx->small.ensure(ctx, up256(bk_bytes) + up256(off_bytes));
    if (st != OWM_OK)
        return st;
    unsigned long long *bk = (unsigned long long *)ctx->small.take(bk_bytes);
    uint32_t *ptoff = (uint32_t *)ctx->small.take(off_bytes);
    uint8_t *h = ctx->pinned(ctx->h_io, ctx->h_io_cap, io_bytes(n_tiles));
    if (!bk || !ptoff || !h) {
        set_err(ctx, "pinned host allocation failed");
        return OWM_E_NOMEM;
    }
    uint32_t *ho = (uint32_t *)h;
    unsigned long long *hk = (unsigned long long *)(h + up256(off_bytes));
    ho[0] = 0;
    for (uint32_t t = 0; t < n_tiles; ++t)
        ho[t + 1] = ho[t] + (uint32_t)tiles[t].n;
    HIP_TRY(hipMemcpyAsync(ptoff, ho, off_bytes, hipMemcpyHostToDevice, s), "upload offsets");
    BatchDev B{};
    B.ntiles = n_tiles;
    B.np = (uint32_t)np;
    B.pt_off = ptoff;
    launch_bbox_init(s, bk, n_tiles);
    const int pi = ctx->prof.begin(s, PH_BBOX);
    launch_bbox(s, B, dx, dy, bk);
    ctx->prof.end(s, pi, 16ull * np, np);
    HIP_TRY(hipMemcpyAsync(hk, bk, n_tiles * 32ull, hipMemcpyDeviceToHost, s), "bbox D2H");
    HIP_TRY(hipStreamSynchronize(s), "bbox sync");
    ctx->prof.collect();
    auto dec = [](unsigned long long k) {
        const uint64_t b = (k >> 63) ? (k & 0x7FFFFFFFFFFFFFFFull) : ~k;
        double v;
        memcpy(&v, &b, 8);
        return v;
    };
    for (uint32_t t = 0; t < n_tiles; ++t) {
        if (tiles[t].params.flags & OWM_F_HAVE_BBOX)
            continue;
        if (tiles[t].n == 0 || hk[4 * t] == ~0ull || hk[4 * t + 1] == ~0ull) {
            set_err(ctx, "tile %u: no finite points to take a bbox from", t);
            return OWM_E_ARG;
        }
        box[t] = {dec(hk[4 * t]), dec(hk[4 * t + 2]), dec(hk[4 * t + 1]), dec(hk[4 * t + 3])};
    }
    return OWM_OK;
}

owm_status one_box(owm_ctx *ctx, const double *dx, const double *dy, uint64_t n, double *box,
                   bool &any)
{
    const GridIo io(ctx, 1);
    if (!io.head) {
        set_err(ctx, "pinned host allocation failed");
        return OWM_E_NOMEM;
    }
    owm_tile t{};
    t.n = n;
    std::vector<std::array<double, 4>> b(1);
    const owm_status st = take_few_boxes(ctx, dx, dy, &t, 1, io, b);
    any = st != OWM_E_ARG;
    memcpy(box, b[0].data(), sizeof b[0]);
    return any ? st : OWM_OK;
}

// Where a chain's points are, and what it is to give.
struct GridSrc {
    const double *x = nullptr, *y = nullptr, *z = nullptr;
    const TreeOut *tree = nullptr;  // a resident tree's instead
    bool minima = false;            // the windows' minima (qo.min_ids), not the seeds
};

// Everything the chain's launches depend on.
static void plan_key(owm_ctx *ctx, const GridSrc &src, const GridPlan &P, const GridIo &io,
                     std::vector<uint8_t> &key)
{
    auto put = [&key](const void *p, size_t n) {
        const uint8_t *b = (const uint8_t *)p;
        key.insert(key.end(), b, b + n);
    };
    key.clear();
    put("grid", 4);
    const void *ptrs[6] = {src.x, src.y, src.z, ctx->arena.buf.ptr, io.head, ctx->h_tab};
    put(ptrs, sizeof ptrs);
    put(P.t.data(), P.t.size() * sizeof(GridTile));
    put(P.pt_off.data(), P.pt_off.size() * 4);
}

// Runs the planned chain; its results are in io (and qo) when it comes back.  Not
// taken: it might not fit the budget where the tree chain would, there is no memory, or
// too many points lie on edges.
static owm_status exec_plan(owm_ctx *ctx, const GridPlan &P, const GridIo &io, const GridSrc &src,
                            uint32_t flags, QueryOut &qo, bool &taken)
{
    taken = false;
    const uint32_t T = (uint32_t)P.t.size();
    const uint64_t np = P.np;
    const uint64_t nwords = (np + 31) / 32, items = P.item_off[T], gcells = P.gcell_off[T];
    const uint64_t nseed = std::min<uint64_t>(np, P.nwin + gcells) + 1;
    const uint64_t table = up256(T * sizeof(GridTile)) + 6 * up256((T + 1) * 4ull);
    const uint64_t need = table + up256(P.recs * 12 + 64) + up256(P.tab * 2) +
                          up256(P.cells * 16) + up256(items * 4) + up256(P.axis_off[T] * 8ull) +
                          up256(P.pool_cap * GRID_POOLS * sizeof(GridRare)) +
                          up256(P.list_cap * GRID_POOLS * 4) + up256(GRID_POOLS * 128) + 2 * up256((nwords + 4) * 4) +
                          up256((gcells + 1) * 4) + up256((nwords / 4096 + 2) * 4) +
                          up256(nseed * 4) + up256((T + 1) * 4ull) +
                          up256(GridHeavy::bytes(P.heavy_cap, P.heavy_cells)) +
                          (src.minima ? up256(P.nwin * 4) : 0) + 4096;
    // (a tree's query may leave less room than the tree chain would for the
    // builds that follow: its scratch grows only where one of this size still fits)
    if (src.tree ? need > ctx->arena.buf.bytes && ctx->exceeds(need + tree_chain_bound(P))
                 : ctx->exceeds(std::max(need, tree_chain_bound(P)), &ctx->arena.buf))
        return OWM_OK;
    void *old_arena = ctx->arena.buf.ptr;
    owm_status st = ctx->arena.ensure(ctx, need);
    if (st == OWM_E_NOMEM)
        return OWM_OK;  // the tree chain may fit
    if (st != OWM_OK)
        return st;
    if (ctx->arena.buf.ptr != old_arena)
        ctx->graphs.clear();
    taken = true;

    Arena &A = ctx->arena;
    hipStream_t s = ctx->stream;
    // table
    uint8_t *d = A.take(table);
    (void)hipStreamSynchronize(s);  // the previous reads of this buffer must have completed
    uint8_t *h = ctx->pinned(ctx->h_tab, ctx->h_tab_cap, table);
    if (!d || !h) {
        set_err(ctx, "pinned host allocation failed");
        return OWM_E_NOMEM;
    }
    bool graph = (flags & OWM_B_GRAPH) != 0;
    std::vector<uint8_t> key;
    if (graph || (flags & B_AUTO_GRAPH))
        plan_key(ctx, src, P, io, key);
    if (!graph && (flags & B_AUTO_GRAPH))
        graph = ctx->graphs.last_grid.repeats(key) && !ctx->prof.on;
    GridDev G{};
    if (src.tree) {
        G.xy = src.tree->pts.xy;
        G.zi = src.tree->pts.zi;
        G.pos = src.tree->pos;
    }
    G.ntiles = T;
    G.ngcell = (uint32_t)gcells;
    G.tiles = (const GridTile *)d;
    memcpy(h, P.t.data(), T * sizeof(GridTile));
    const std::vector<uint32_t> *tabs[6] = {&P.st_off,    &P.item_off, &P.blk_off,
                                           &P.gcell_off, &P.axis_off, &P.pt_off};
    const uint32_t *off[6];
    uint64_t o = up256(T * sizeof(GridTile));
    for (int k = 0; k < 6; ++k, o += up256((T + 1) * 4ull)) {
        memcpy(h + o, tabs[k]->data(), (T + 1) * 4ull);
        off[k] = (const uint32_t *)(d + o);
    }
    G.st_off = off[0];
    G.item_off = off[1];
    G.blk_off = off[2];
    G.gcell_off = off[3];
    G.axis_off = off[4];
    BatchDev B{};
    B.ntiles = T;
    B.np = (uint32_t)np;
    B.pt_off = off[5];
    // a few tiles' table is fetched by the chain's first launch
    const bool fetch = T <= 8;
    if (!fetch)
        HIP_TRY(hipMemcpyAsync(d, h, table, hipMemcpyHostToDevice, s), "upload table");

    auto body = [&]() -> owm_status {
        // (a lane's last load may reach 36 bytes past its run)
        G.rec = (uint32_t *)A.take(P.recs * 12 + 64);
        G.tab = (uint16_t *)A.take(P.tab * 2);
        G.cells = (uint4 *)A.take(P.cells * 16);
        G.heads = (uint32_t *)A.take(items * 4);
        G.wcols = (int2 *)A.take(P.axis_off[T] * 8ull);
        G.pool = (GridRare *)A.take(P.pool_cap * GRID_POOLS * sizeof(GridRare));
        G.pool_cap = (uint32_t)P.pool_cap;
        G.many_cap = P.many_cap;
        G.list = (uint32_t *)A.take(P.list_cap * GRID_POOLS * 4);
        G.list_cap = (uint32_t)P.list_cap;
        G.pool_used = (uint32_t *)A.take(GRID_POOLS * 128);
        G.seen = (uint32_t *)A.take((nwords + 4) * 4);
        G.llp = (uint32_t *)A.take((nwords + 4) * 4);
        G.cell_flag = (uint32_t *)A.take((gcells + 1) * 4);
        G.heavy = (uint4 *)A.take(GridHeavy::bytes(P.heavy_cap, P.heavy_cells));
        uint32_t *lookback = (uint32_t *)A.take((nwords / 4096 + 2) * 4);
        uint32_t *out = (uint32_t *)A.take(nseed * 4);
        uint32_t *seed_off = (uint32_t *)A.take((T + 1) * 4ull);
        if (src.minima)
            G.min_ids = (uint32_t *)A.take(P.nwin * 4);
        uint32_t *cnt = (uint32_t *)A.take(1024);
        if (!cnt) {
            set_err(ctx, "scratch arena exhausted (grid)");
            return OWM_E_INTERNAL;
        }
        G.err = cnt + 3;
        FillRanges z;
        auto zero = [&](uint32_t *p, uint64_t words) {
            z.ptr[z.count] = p;
            z.len[z.count++] = words;
        };
        zero(cnt, 16);
        zero(G.pool_used, GRID_POOLS * 32);
        zero(G.seen, nwords + 4);
        zero(G.llp, nwords + 4);
        zero(G.cell_flag, gcells + 1);
        zero(lookback, nwords / 4096 + 2);
        launch_grid_prep(s, G, z, P.axis_off[T], fetch ? (const uint32_t *)h : nullptr,
                         (uint32_t)(table / 4));
        int pi = ctx->prof.begin(s, PH_GRID_PART);
        launch_grid_part(s, G, src.x, src.y, src.z, P.st_off[T], P.t[0].lsp, P.max_nb);
        // x, y and z read; a record written
        ctx->prof.end(s, pi, 36ull * np, np);
        pi = ctx->prof.begin(s, PH_GRID_BIN);
        for (const GridPlan::Class &c : P.cls)
            launch_grid_bin(s, G, c.t0, c.t1, P.item_off[c.t0],
                            P.item_off[c.t1] - P.item_off[c.t0], c.cells);
        if (P.heavy_cap)
            launch_grid_heavy(s, G, P.heavy_cap, P.heavy_cells);
        ctx->prof.end(s, pi, 12ull * np + 16ull * P.cells, np, (uint32_t)P.cls.size());
        pi = ctx->prof.begin(s, PH_GRID_WIN);
        launch_grid_windows(s, G, src.x, src.y, P.blk_off[T], P.win_cells);
        ctx->prof.end(s, pi, 16ull * P.cells + 8ull * P.nwin, P.nwin);
        if (src.minima) {
            launch_flags_out(s, cnt + 3, io.head + 1);
            HIP_TRY(hipGetLastError(), "grid chain launch");
            qo.min_ids = G.min_ids;
            return OWM_OK;
        }
        if (gcells) {
            pi = ctx->prof.begin(s, PH_STAGE3);
            launch_grid_cells(s, G);
            ctx->prof.end(s, pi, 12ull * gcells, gcells);
        }
        pi = ctx->prof.begin(s, PH_MERGE);
        SeedOut S;
        S.ntiles = T;
        S.pt_off = B.pt_off;
        S.err = cnt + 3;
        S.host = io.head;
        S.host_off = io.off;
        S.host_ids = io.ids;
        S.host_cap = GridIo::IDS;
        launch_seeds(s, B, G.llp, (uint32_t)nwords, out, (uint32_t)nseed, seed_off, cnt + 2,
                     lookback, cnt + 7, S);
        ctx->prof.end(s, pi, 4ull * nwords, nwords);
        HIP_TRY(hipGetLastError(), "grid chain launch");
        qo.cnt = cnt;
        qo.seeds = out;
        return OWM_OK;
    };
    st = run_chain(ctx, graph, std::move(key), A, qo, body);
    if (st != OWM_OK)
        return st;
    HIP_TRY(hipStreamSynchronize(s), "pipeline");
    ctx->prof.collect();
    const uint32_t err = io.head[1];
    if (err & ~GRID_ERR_POOL) {
        set_err(ctx, "device capacity guard tripped (flags %u)", err);
        return OWM_E_INTERNAL;
    }
    taken = !(err & GRID_ERR_POOL);
    return OWM_OK;
}

// The seeds of a finished chain.
static owm_status copy_seeds(owm_ctx *ctx, const GridIo &io, const QueryOut &qo, uint32_t n_tiles,
                             uint32_t *seeds, uint64_t cap, uint64_t *seed_off_host)
{
    const uint64_t ns = io.head[0];
    for (uint32_t t = 0; t <= n_tiles; ++t)
        seed_off_host[t] = io.off[t];
    if (ns > cap) {
        set_err(ctx, "seed buffer holds %llu, %llu needed", (unsigned long long)cap,
                (unsigned long long)ns);
        return OWM_E_CAPACITY;
    }
    if (ns <= GridIo::IDS)
        memcpy(seeds, io.ids, ns * 4);
    else
        HIP_TRY(hipMemcpy(seeds, qo.seeds, ns * 4, hipMemcpyDeviceToHost), "seeds D2H");
    return OWM_OK;
}

owm_status run_grid(owm_ctx *ctx, const double *dx, const double *dy, const double *dz,
                    const owm_tile *tiles, uint32_t n_tiles, uint32_t flags, uint32_t *seeds,
                    uint64_t cap, uint64_t *seed_off_host, std::vector<owm_tile> &boxed,
                    bool &handled)
{
    handled = false;
    owm_status st = check_tiles(ctx, tiles, n_tiles);
    if (st != OWM_OK)
        return st;
    uint64_t np = 0;
    bool need_box = false;
    std::vector<std::array<double, 4>> box(n_tiles);
    for (uint32_t t = 0; t < n_tiles; ++t) {
        if (tiles[t].params.leaf_size)
            return OWM_OK;  // the caller asks for a tree with such leaves
        if (tiles[t].offset != np)
            return OWM_OK;  // the tree chain reports it
        np += tiles[t].n;
        if (tiles[t].params.flags & OWM_F_HAVE_BBOX)
            memcpy(box[t].data(), tiles[t].params.bbox, sizeof(double) * 4);
        else
            need_box = true;
    }
    if (np == 0)
        return OWM_OK;
    // Many tiles of few points are the tree chain's: its box pass counts the sort's
    // digits on the way, where this one's is a pass of its own through tile after
    // tile, and a tile takes 16 workgroups of the bins at least (500 tiles of 200
    // points 1.02 ms by the tree chain, 1.75 here; 3000 of 300 2.5 and 3.6; 20000 of
    // 1000 15.4 and 20.1; 500 of 5000 0.83 and 0.73, 3000 of 5000 3.5 and 2.7).
    if (n_tiles > BOX_TILES && np / n_tiles < 4096)
        return OWM_OK;
    const GridIo io(ctx, n_tiles);
    if (!io.head) {
        set_err(ctx, "pinned host allocation failed");
        return OWM_E_NOMEM;
    }
    if (need_box) {
        st = n_tiles <= BOX_TILES ? take_few_boxes(ctx, dx, dy, tiles, n_tiles, io, box)
                                  : take_boxes(ctx, dx, dy, tiles, n_tiles, box);
        if (st != OWM_OK)
            return st;
    }
    // what a call that is not taken hands on: its tiles with their boxes
    auto hand_on = [&]() {
        if (need_box) {
            boxed.assign(tiles, tiles + n_tiles);
            for (uint32_t t = 0; t < n_tiles; ++t) {
                boxed[t].params.flags |= OWM_F_HAVE_BBOX;
                memcpy(boxed[t].params.bbox, box[t].data(), sizeof(double) * 4);
            }
        }
        return OWM_OK;
    };
    GridPlan P;
    if (!make_plan(ctx, tiles, n_tiles, box, P))
        return hand_on();
    GridSrc src;
    src.x = dx;
    src.y = dy;
    src.z = dz;
    QueryOut qo;
    st = exec_plan(ctx, P, io, src, flags, qo, handled);
    if (st != OWM_OK)
        return st;
    if (!handled)
        return hand_on();
    return copy_seeds(ctx, io, qo, n_tiles, seeds, cap, seed_off_host);
}

owm_status tree_grid(owm_ctx *ctx, const owm_tree &tree, const owm_params &params, bool minima,
                     uint32_t *out, uint64_t cap, uint64_t *n_out, bool &handled)
{
    handled = false;
    if (!tree.n || ctx->tuner.forced || getenv("OWM_NO_GRID"))
        return OWM_OK;
    owm_tile t{};
    t.n = tree.n;
    t.params = params;
    std::vector<std::array<double, 4>> box(1);
    if (params.flags & OWM_F_HAVE_BBOX)
        memcpy(box[0].data(), params.bbox, sizeof(double) * 4);
    else
        box[0] = tree.P.box[0];
    // The chain reads every point, the tree chain the leaves under the windows'
    // edges: a query of a part of the tree stays there.  So do large trees with
    // small windows, whose order leaves the partition's runs uneven (minima and
    // seeds, windows of 600 points, 3M points: 125 us against 183 by the tree
    // chain, 8M 231 and 325, 16M 434 and 537, 60M 3450 and 1829; windows of 2400
    // points, 3M points: 172 and 595 us, 16M 418 and 807, 60M 1566 and 1182).
    const std::array<double, 4> &tb = tree.P.box[0];
    for (int a = 0; a < 4; a += 2)
        if (!(box[0][a] <= tb[a] && tb[a + 1] <= box[0][a + 1]))
            return OWM_OK;
    const double per_window = (double)tree.n * params.wsize * params.wsize /
                              ((tb[1] - tb[0]) * (tb[3] - tb[2]));
    if (tree.n > (8u << 20) && !(tree.n <= (32u << 20) && per_window >= 2000.0))
        return OWM_OK;
    GridPlan P;
    if (!make_plan(ctx, &t, 1, box, P))
        return OWM_OK;
    if (minima && P.nwin > cap)
        return OWM_OK;  // the tree chain reports it
    const GridIo io(ctx, 1);
    if (!io.head) {
        set_err(ctx, "pinned host allocation failed");
        return OWM_E_NOMEM;
    }
    GridSrc src;
    src.tree = &tree.T;
    src.minima = minima;
    QueryOut qo;
    owm_status st = exec_plan(ctx, P, io, src, 0, qo, handled);
    if (st != OWM_OK || !handled)
        return st;
    if (minima) {
        *n_out = P.nwin;
        HIP_TRY(hipMemcpy(out, qo.min_ids, P.nwin * 4, hipMemcpyDeviceToHost), "min_ids D2H");
        return OWM_OK;
    }
    uint64_t off[2] = {0, 0};
    st = copy_seeds(ctx, io, qo, 1, out, cap, off);
    *n_out = off[1];
    return st;
}

}  // namespace owm
