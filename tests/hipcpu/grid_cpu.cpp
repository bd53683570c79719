// The column-grid chain on the CPU (hip/hip_runtime.h here): csrc/grid.hip, whose
// text comes in as GRID_SOURCE, under the library's own planning and launch code.
//   grid_cpu IN OUT
// IN: doubles {mode, poke, calls, tiles, then per tile {n, wsize, bsize,
// overlap, has box, box[4]}}, then x, y, z.  Modes: 0 a whole run, 1 the seeds and
// 2 the minima of a resident tree (one tile, its points in reverse); 3 whole runs that
// may replay, each followed by the tree chain's look at its own key.  poke: 1, every
// workgroup of k_grid_heavy finds GRID_ERR_POOL set by another one of the launch
// before its wave 4 first runs; 2, the queue of heavy stretches holds two; 3, the device
// has 2 MB; 4 and 5, a share of the lists holds 600 words (5: from k_grid_heavy on).
// OUT: int64 {status, taken, flags, count, stray marks, barriers passed by launches that
// began after the flag was raised, by k_grid_part, its workgroups, replays of the chain,
// calls in which the tree chain's key repeats, the largest allocation asked for}, tile
// ranges (tiles + 1 of them), ids.
#include "../../fastowm_amd/csrc/owm_host.h"
#include <math.h>

namespace owm {
uint4 s_part[10240];  // dynamic LDS
unsigned long long s_bin[20480], s_win[20480];
}  // namespace owm
#include GRID_SOURCE

namespace owm {

static int64_t stray = 0;  // bits behind the last point

void launch_fill_u32(hipStream_t, uint32_t *p, uint64_t n, uint32_t v)
{
    for (uint64_t i = 0; i < n; ++i)
        p[i] = v;
}
uint64_t box_work_bytes() { return 256 + BOX_BLOCKS * 32ull; }
void launch_boxes(hipStream_t, const BoxArgs &a, const double *x, const double *y, void *, double *box)
{
    for (uint32_t t = 0; t < a.ntiles; ++t) {
        double *b = box + 4 * t;
        b[0] = b[1] = INFINITY;
        b[2] = b[3] = -INFINITY;
        for (uint32_t i = a.pt[t]; i < a.pt[t + 1]; ++i) {
            b[0] = fmin(b[0], x[i]);
            b[1] = fmin(b[1], y[i]);
            b[2] = fmax(b[2], x[i]);
            b[3] = fmax(b[3], y[i]);
        }
    }
}
void launch_seeds(hipStream_t, const BatchDev &B, const uint32_t *words, uint32_t nwords, uint32_t *out,
                  uint32_t n_max, uint32_t *, uint32_t *d_count, uint32_t *, uint32_t *, const SeedOut &S)
{
    uint32_t n = 0, t = 0;
    S.host_off[0] = 0;
    for (uint32_t i = 0; i < B.np; ++i) {
        while (t + 1 < B.ntiles && B.pt_off[t + 1] <= i)
            S.host_off[++t] = n;
        if (((words[i >> 5] >> (i & 31)) & 1u) && n < n_max) {
            out[n] = i - B.pt_off[t];
            if (n < S.host_cap)
                S.host_ids[n] = out[n];
            ++n;
        }
    }
    while (t < B.ntiles)
        S.host_off[++t] = n;
    for (uint32_t i = B.np; i < (nwords + 4) * 32; ++i)
        stray += (words[i >> 5] >> (i & 31)) & 1u;
    S.host[0] = *d_count = n;
    S.host[1] = *S.err;
}

}  // namespace owm

owm_ctx::~owm_ctx() {}

int main(int argc, char **argv)
{
    using namespace owm;
    FILE *f = argc == 3 ? fopen(argv[1], "rb") : nullptr;
    if (!f)
        return 2;
    double head[4];
    if (fread(head, 8, 4, f) != 4)
        return 2;
    const int mode = (int)head[0], calls = (int)head[2];
    const uint32_t T = (uint32_t)head[3];
    std::vector<owm_tile> tiles(T);
    uint64_t np = 0;
    for (owm_tile &t : tiles) {
        double v[9];
        if (fread(v, 8, 9, f) != 9)
            return 2;
        t = owm_tile{};
        t.offset = np;
        t.n = (uint64_t)v[0];
        t.params.wsize = (uint32_t)v[1];
        t.params.bsize = (uint32_t)v[2];
        t.params.overlap = v[3];
        t.params.flags = v[4] ? OWM_F_HAVE_BBOX : 0;
        memcpy(t.params.bbox, v + 5, 32);
        np += t.n;
    }
    std::vector<double> c(3 * np);
    if (fread(c.data(), 8, 3 * np, f) != 3 * np)
        return 2;
    fclose(f);
    const double *x = c.data(), *y = x + np, *z = y + np;
    // memory that was never written reads as a low point of every window and cell, whose
    // index lies behind every cloud
    GridRare low{};
    low.zk = 1;
    low.id = 0x7FFFFFF0u;
    low.wx1 = low.wy1 = low.gx1 = low.gy1 = 0xFFFFu;
    hipcpu::stale.assign((const unsigned char *)&low, (const unsigned char *)(&low + 1));
    if (head[1] == 3)
        hipcpu::memory_left = 2 << 20;
    owm_ctx *ctx = new owm_ctx;
    uint32_t *err = nullptr;
    int64_t after = 0, part = 0, groups = 0, mark = 0, kind = 0, repeats = 0;
    auto count_barriers = [&]() {
        (kind == 1 ? after : part) += kind ? hipcpu::barriers - mark : 0;
        mark = hipcpu::barriers;
        kind = 0;
    };
    hipcpu::before_launch = [&](const void *k, const void *arg) {
        if (k != (const void *)&k_flags_out)  // (whose first argument is no GridDev)
            err = ((const GridDev *)arg)->err;
        count_barriers();
        const void *const parts[4] = {(const void *)&k_grid_part<false, 10>, (const void *)&k_grid_part<false, 11>,
                                      (const void *)&k_grid_part<false, 12>, (const void *)&k_grid_part<true, 12>};
        for (const void *p : parts)
            if (k == p) {
                groups = ((const GridDev *)arg)->st_off[((const GridDev *)arg)->ntiles];
                kind = 2;
            }
        if (!kind && k != (const void *)&k_grid_prep && k != (const void *)&k_flags_out && *err)
            kind = 1;
        const bool heavy = k == (const void *)&k_grid_heavy<512, false>;
        if ((head[1] == 4 && k == (const void *)&k_grid_bin<512, false>) || (head[1] >= 4 && heavy))
            const_cast<GridDev *>((const GridDev *)arg)->list_cap = 600;
        if (head[1] == 2 && k == (const void *)&k_grid_bin<512, false>)
            for (uint32_t t = 0; t < T; ++t)
                const_cast<GridTile *>(((const GridDev *)arg)->tiles)[t].heavy_cap = 2;
    };
    if (head[1] == 1)
        hipcpu::before_wave = [&](const void *k, uint32_t, uint32_t w) {
            if (w == 4 && (k == (const void *)&k_grid_heavy<512, false> ||
                           k == (const void *)&k_grid_heavy<512, true>))
                *err |= GRID_ERR_POOL;
        };
    std::vector<uint32_t> ids(np + 1000000);
    std::vector<uint64_t> off(T + 1);
    bool taken = false;
    int64_t status = 0;
    uint64_t count = 0;
    for (int k = 0; k < calls; ++k) {
        if (mode == 0 || mode == 3) {
            std::vector<owm_tile> boxed;
            status = run_grid(ctx, x, y, z, tiles.data(), T, mode ? B_AUTO_GRAPH : 0, ids.data(), ids.size(),
                              off.data(), boxed, taken);
            count = off[T];
            if (mode)
                repeats += ctx->graphs.last_tree.repeats({'t', 'r', 'e', 'e'});
            continue;
        }
        owm_tree tree;
        std::vector<double2> xy(np);
        std::vector<PointZ> zi(np);
        std::vector<uint32_t> pos(np);
        tree.n = np;
        tree.P.box.resize(1);
        auto &b = tree.P.box[0];
        b = {INFINITY, -INFINITY, INFINITY, -INFINITY};
        for (uint32_t i = 0; i < np; ++i) {
            pos[i] = (uint32_t)np - 1 - i;
            xy[pos[i]] = make_double2(x[i], y[i]);
            zi[pos[i]] = PointZ{z[i], i, 0};
            b = {fmin(b[0], x[i]), fmax(b[1], x[i]), fmin(b[2], y[i]), fmax(b[3], y[i])};
        }
        tree.T.pts.xy = xy.data();
        tree.T.pts.zi = zi.data();
        tree.T.pos = pos.data();
        status = tree_grid(ctx, tree, tiles[0].params, mode == 2, ids.data(), ids.size(), &count, taken);
        off = {0, count};
    }
    if (status == 0 && !taken)
        count = 0;
    FILE *o = fopen(argv[2], "wb");
    count_barriers();
    const int64_t head_out[11] = {status, taken, err ? *err : 0, (int64_t)count, stray, after, part, groups,
                                  (int64_t)hipcpu::graph_launches, repeats, (int64_t)hipcpu::largest};
    fwrite(head_out, 8, 11, o);
    fwrite(off.data(), 8, T + 1, o);
    fwrite(ids.data(), 4, count, o);
    fclose(o);
    return 0;
}
