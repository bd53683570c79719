// Quadtree leaf statistics: the leaves of the reference's parallel_qtree
// (CPP-TBB-CPU/src/optim3_func.cpp:218-253) as owm_stats walks them
// (CPP-TBB-CPU/application/owm_stats.cpp, CPP-TBB-CPU/include/stats_func.hpp).
//
// The reference tree does not depend on insertion order: a node of depth
// 0..level is always split; below, under the maxNumber policy
// (insertPointMaxNum, :160-184) a node is split exactly when more than
// maxNumber points reach it, and under the minRadius policy (insertPoint,
// :103-123) when at least one point reaches it and radius * 0.5 > minRadius.
// So no pointer tree is built.  Every point gets a path key, its quadrants
// (quadrantIdx, :91-100, against the child centres of createQuadrants,
// :59-73) at depths 1..16, two bits a depth, and the keys are sorted by the
// quadrants of depths 1..S (S = 12, or 16 when the tree is expected to go
// deeper than 12).  Down to depth S a node's points are then one
// contiguous key range: depth by depth, each split ("open") node's range is
// cut into its four children's by binary searches on the keys, and each
// child is split (it gets an open-node index, a range and a centre) or a leaf
// (its (depth, points) pair is counted).  That work scales with the nodes,
// not the points.  Nodes still open at depth S go on point by point: each
// point in one holds its node and is routed to a child by its key's next
// quadrant (below depth 16 by its coordinates against the node's centre, the
// index of the point at each key position then coming from a second sort with
// values), the children's points are counted with atomics (runs of equal
// children within a wave add once) and classified as above.
#include "owm_kernels.h"

namespace owm {

constexpr int QS_TB = 256;

__global__ __launch_bounds__(QS_TB) void k_qs_path(const double *__restrict__ x,
                                                    const double *__restrict__ y, uint64_t n,
                                                    QsPath P, int sl, uint32_t *__restrict__ key)
{
    for (uint64_t i = (uint64_t)blockIdx.x * QS_TB + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * QS_TB) {
        const double px = x[i], py = y[i];
        double cx = P.cx, cy = P.cy;
        uint32_t k = 0;
#pragma unroll
        for (int l = 0; l < QS_KEY_LEVELS; ++l) {
            const bool qx = px >= cx, qy = py >= cy;
            k = (k << 2) | (qx ? 2u : 0u) | (qy ? 1u : 0u);
            cx += qx ? P.off[l] : -P.off[l];
            cy += qy ? P.off[l] : -P.off[l];
        }
        // depths 1..sl to bits 0..2sl-1, the deeper ones above
        key[i] = sl >= QS_KEY_LEVELS ? k : (k >> (2 * (QS_KEY_LEVELS - sl))) | (k << (2 * sl));
    }
}

__global__ void k_qs_root(QsDev D, double cx, double cy)
{
    D.nopen[0] = 1;
    D.cen[0][0] = make_double2(cx, cy);
    D.rng[0][0] = make_uint2(0u, (uint32_t)D.n);
}

// Leaves of one block: counts below QS_HB in LDS bins, larger ones listed.
__device__ __forceinline__ void qs_leaf(QsDev &D, uint32_t *s_hist, int d, uint32_t c)
{
    if (c < QS_HB) {
        atomicAdd(&s_hist[c], 1u);
    } else {
        const uint32_t o = atomicAdd(D.novf, 1u);
        if (o < D.ovf_cap)
            D.ovf[o] = make_uint2((uint32_t)d, c);
        else
            atomicOr(D.flags, 1u);
    }
}

__device__ __forceinline__ void qs_flush(QsDev &D, uint32_t *s_hist, int d)
{
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < QS_HB; k += QS_TB)
        if (s_hist[k])
            atomicAdd(&D.hist[(uint64_t)d * QS_HB + k], (unsigned long long)s_hist[k]);
}

__device__ __forceinline__ bool qs_split_rule(const QsDev &D, bool forced, bool radius_split,
                                              uint32_t c)
{
    return forced || (D.policy == 0 ? c > D.max_number : (c >= 1 && radius_split));
}

// The quadrant a path key gives at depth d (1..16), sl depths sorted.
__device__ __forceinline__ uint32_t qs_quadrant(uint32_t key, int d, int sl)
{
    return d <= sl ? (key >> (2 * (sl - d))) & 3u : (key >> (2 * sl + 2 * (QS_KEY_LEVELS - d))) & 3u;
}

// Depth d <= sort_levels: one thread per open depth-(d-1) node cuts its key
// range into its children's and classifies them; new open nodes get their
// indices from one atomic per block.
__global__ __launch_bounds__(QS_TB) void k_qs_split(QsDev D, int d, float rd, double off)
{
    __shared__ uint32_t s_hist[QS_HB];
    __shared__ uint32_t s_scan[QS_TB / 64];
    __shared__ uint32_t s_base;
    const uint32_t nprev = min(D.nopen[d - 1], D.open_cap);
    if (blockIdx.x * QS_TB >= nprev)
        return;
    for (uint32_t k = threadIdx.x; k < QS_HB; k += QS_TB)
        s_hist[k] = 0;
    const uint2 *pr = D.rng[(d - 1) & 1];
    const double2 *pc = D.cen[(d - 1) & 1];
    uint2 *nr = D.rng[d & 1];
    double2 *nc = D.cen[d & 1];
    const bool forced = d <= (int)D.level;
    const bool radius_split = (double)rd * 0.5 > (double)D.min_radius;
    const int sh = 2 * (D.sort_levels - d);
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (uint32_t base = blockIdx.x * QS_TB; base < nprev; base += gridDim.x * QS_TB) {
        const uint32_t o = base + threadIdx.x;
        uint32_t b[5] = {0, 0, 0, 0, 0};
        uint32_t nopen = 0;
        bool op[4] = {false, false, false, false};
        if (o < nprev) {
            const uint2 r = pr[o];
            b[0] = r.x;
            b[4] = r.y;
            // keys in [r.x, r.y) share the depth-(d-1) prefix; their depth-d
            // quadrant (key >> sh) & 3 ascends: b[q] = first with quadrant >= q
            for (uint32_t q = 1; q < 4; ++q) {
                uint32_t lo = b[q - 1], hi = r.y;
                while (lo < hi) {
                    const uint32_t mid = lo + (hi - lo) / 2;
                    if (((D.key[mid] >> sh) & 3u) < q)
                        lo = mid + 1;
                    else
                        hi = mid;
                }
                b[q] = lo;
            }
            for (int q = 0; q < 4; ++q) {
                op[q] = qs_split_rule(D, forced, radius_split, b[q + 1] - b[q]);
                nopen += op[q] ? 1u : 0u;
            }
        }
        // block-wide exclusive scan of the open children
        uint32_t incl = nopen;
#pragma unroll
        for (int k = 1; k < 64; k <<= 1) {
            const uint32_t v = __shfl_up(incl, k, 64);
            if (lane >= (uint32_t)k)
                incl += v;
        }
        __syncthreads();  // s_scan / s_base of the previous round are consumed
        if (lane == 63)
            s_scan[wv] = incl;
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t t = 0;
            for (int w = 0; w < QS_TB / 64; ++w) {
                const uint32_t v = s_scan[w];
                s_scan[w] = t;
                t += v;
            }
            s_base = t ? atomicAdd(&D.nopen[d], t) : 0u;
        }
        __syncthreads();
        uint32_t idx = s_base + s_scan[wv] + incl - nopen;
        if (o < nprev) {
            const double2 p = pc[o];
            for (int q = 0; q < 4; ++q) {
                if (!op[q]) {
                    qs_leaf(D, s_hist, d, b[q + 1] - b[q]);
                    continue;
                }
                if (idx < D.open_cap) {
                    nr[idx] = make_uint2(b[q], b[q + 1]);
                    nc[idx] = make_double2(p.x + ((q & 2) ? off : -off), p.y + ((q & 1) ? off : -off));
                } else {
                    atomicOr(D.flags, 2u);
                }
                ++idx;
            }
        }
    }
    qs_flush(D, s_hist, d);
}

// Depth sort_levels still has open nodes: every point of one holds its
// index (st was filled with OWM_NONE), and remap is the identity on them.
__global__ __launch_bounds__(QS_TB) void k_qs_deep_start(QsDev D)
{
    const uint32_t nopen = min(D.nopen[D.sort_levels], D.open_cap);
    const uint2 *r = D.rng[D.sort_levels & 1];
    for (uint32_t o = blockIdx.x * QS_TB + threadIdx.x; o < nopen; o += gridDim.x * QS_TB) {
        D.remap[o] = o;
        for (uint32_t i = r[o].x; i < r[o].y; ++i)
            D.st[i] = o;
    }
}

// Depth d > sort_levels: each point of an open depth-(d-1) node moves to
// child slot 4 * node + quadrant; points whose node became a leaf are marked
// settled.  Points are in key order; below depth 16, perm gives each one's
// index.
__global__ __launch_bounds__(QS_TB) void k_qs_route(QsDev D, int d)
{
    const uint32_t nprev = min(D.nopen[d - 1], D.open_cap);
    if (nprev == 0)
        return;
    const double2 *cen = D.cen[(d - 1) & 1];
    const uint32_t lane = threadIdx.x & 63;
    for (uint64_t base = (uint64_t)blockIdx.x * QS_TB; base < D.n;
         base += (uint64_t)gridDim.x * QS_TB) {
        const uint64_t i = base + threadIdx.x;
        uint32_t child = OWM_NONE;
        if (i < D.n) {
            const uint32_t s = D.st[i];
            if (s != OWM_NONE) {
                const uint32_t node = D.remap[s];
                if (node == OWM_NONE) {
                    D.st[i] = OWM_NONE;
                } else {
                    uint32_t q;
                    if (D.key && d <= QS_KEY_LEVELS) {
                        q = qs_quadrant(D.key[i], d, D.sort_levels);
                    } else {
                        const uint64_t pi = D.perm ? D.perm[i] : i;
                        const double2 c = cen[node];
                        q = (D.x[pi] >= c.x ? 2u : 0u) | (D.y[pi] >= c.y ? 1u : 0u);
                    }
                    child = 4u * node + q;
                    D.st[i] = child;
                }
            }
        }
        // a run of lanes with the same child adds its length once
        const uint32_t prev = __shfl_up(child, 1, 64);
        const bool starts = lane == 0 || prev != child;
        const uint64_t bnd = __ballot(starts);
        if (starts && child != OWM_NONE) {
            const uint64_t above = lane == 63 ? 0ull : (bnd & (~0ull << (lane + 1)));
            const uint32_t next = above ? (uint32_t)__builtin_ctzll(above) : 64u;
            atomicAdd(&D.cnt[child], next - lane);
        }
    }
}

// Depth d: every child slot of the open depth-(d-1) nodes is split or a leaf.
__global__ __launch_bounds__(QS_TB) void k_qs_classify(QsDev D, int d, float rd, double off)
{
    __shared__ uint32_t s_hist[QS_HB];
    const uint64_t nslots = 4ull * min(D.nopen[d - 1], D.open_cap);
    if ((uint64_t)blockIdx.x * QS_TB >= nslots)
        return;
    for (uint32_t k = threadIdx.x; k < QS_HB; k += QS_TB)
        s_hist[k] = 0;
    __syncthreads();
    const double2 *pc = D.cen[(d - 1) & 1];
    double2 *nc = D.cen[d & 1];
    const bool forced = d <= (int)D.level;
    const bool radius_split = (double)rd * 0.5 > (double)D.min_radius;
    const uint32_t lane = threadIdx.x & 63;
    for (uint64_t base = (uint64_t)blockIdx.x * QS_TB; base < nslots;
         base += (uint64_t)gridDim.x * QS_TB) {
        const uint64_t j = base + threadIdx.x;
        const bool valid = j < nslots;
        uint32_t c = 0;
        bool open = false;
        if (valid) {
            c = D.cnt[j];
            D.cnt[j] = 0;
            open = qs_split_rule(D, forced, radius_split, c);
        }
        const uint64_t m = __ballot(valid && open);
        uint32_t first = 0;
        if (m) {
            if (lane == 0)
                first = atomicAdd(&D.nopen[d], (uint32_t)__popcll(m));
            first = __shfl(first, 0, 64);
        }
        if (!valid)
            continue;
        if (open) {
            const uint32_t idx = first + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
            if (idx < D.open_cap) {
                D.remap[j] = idx;
                const double2 p = pc[j >> 2];
                const uint32_t q = (uint32_t)(j & 3);
                nc[idx] = make_double2(p.x + ((q & 2) ? off : -off), p.y + ((q & 1) ? off : -off));
            } else {
                D.remap[j] = OWM_NONE;
                atomicOr(D.flags, 2u);
            }
        } else {
            D.remap[j] = OWM_NONE;
            qs_leaf(D, s_hist, d, c);
        }
    }
    qs_flush(D, s_hist, d);
}

void launch_qs_root(hipStream_t s, const QsDev &D, double cx, double cy)
{
    hipLaunchKernelGGL(k_qs_root, dim3(1), dim3(1), 0, s, D, cx, cy);
}

void launch_qs_path(hipStream_t s, const double *x, const double *y, uint64_t n, const QsPath &P,
                    int sort_levels, uint32_t *key)
{
    if (n == 0)
        return;
    uint64_t b = (n + QS_TB - 1) / QS_TB;
    b = b > 16384 ? 16384 : b;
    hipLaunchKernelGGL(k_qs_path, dim3((unsigned)b), dim3(QS_TB), 0, s, x, y, n, P, sort_levels, key);
}

void launch_qs_split(hipStream_t s, const QsDev &D, int d, float rd, double off)
{
    uint64_t b = ((uint64_t)D.open_cap + QS_TB - 1) / QS_TB;
    b = b < 1 ? 1 : (b > 4096 ? 4096 : b);
    hipLaunchKernelGGL(k_qs_split, dim3((unsigned)b), dim3(QS_TB), 0, s, D, d, rd, off);
}

void launch_qs_deep_start(hipStream_t s, const QsDev &D)
{
    launch_fill_u32(s, D.st, D.n, OWM_NONE);
    uint64_t b = ((uint64_t)D.open_cap + QS_TB - 1) / QS_TB;
    b = b < 1 ? 1 : (b > 4096 ? 4096 : b);
    hipLaunchKernelGGL(k_qs_deep_start, dim3((unsigned)b), dim3(QS_TB), 0, s, D);
}

void launch_qs_level(hipStream_t s, const QsDev &D, int d, float rd, double off)
{
    uint64_t rb = (D.n + QS_TB - 1) / QS_TB;
    rb = rb < 1 ? 1 : (rb > 16384 ? 16384 : rb);
    hipLaunchKernelGGL(k_qs_route, dim3((unsigned)rb), dim3(QS_TB), 0, s, D, d);
    // slots of the open depth-(d-1) nodes: at most 4 * open_cap
    uint64_t cb = (4ull * D.open_cap + QS_TB - 1) / QS_TB;
    cb = cb < 1 ? 1 : (cb > 2048 ? 2048 : cb);
    hipLaunchKernelGGL(k_qs_classify, dim3((unsigned)cb), dim3(QS_TB), 0, s, D, d, rd, off);
}

// ------------------------------------------------- without sorting ----
//
// Whether a node is split depends on its own point count alone (a split node's
// ancestors hold at least its points, and are forced or as large in radius), so
// the counts of all depths give every leaf: a node is a leaf when its parent is
// split and it is not.  k_qs_part groups each sort tile's points by depth-5 node
// (16 B a point read, 4 written), k_qs_bins counts a node's points per depth-12
// cell in LDS and sums the counts upwards, depth by depth; k_qs_out does the
// depths above and leaves the classes in host memory.  20M points, 24 bytes each:
// 68 + 99 + 20 us, against 833 us for path keys (20 B), their histogram (4 B),
// three sort passes (8 B each) and binary searches per node.  The partition runs
// at 5.9 TB/s; the bins are bound by latency (two workgroups of 64 KB of counts
// to a CU, each a chain of run starts, records and twelve barriers).

constexpr int QP_NT = 512, QP_K = QF_PTS / QP_NT;
constexpr uint32_t QF_BIN_MASK = QF_BINS - 1u, QF_SLOT_MASK = QF_PTS - 1u;

__device__ __forceinline__ bool qf_rule(const QsFast &F, int d, uint32_t c)
{
    return d <= (int)F.D.level || (F.D.policy == 0 ? c > F.D.max_number
                                                   : (c >= 1u && ((F.radius_split >> d) & 1u)));
}

// Cell of a coordinate along one axis at depth QF_DEPTH.  The centres that
// quadrantIdx compares with down to that depth are c + k * side up to 12 roundings
// (side = the depth-12 cell's, a power-of-two fraction of the float root radius),
// so away from them the cell is the estimate's floor; false near one, and for
// NaN.
__device__ __forceinline__ bool qf_cell(double v, double c, double inv, double tol, uint32_t &cell)
{
    constexpr double half = (double)(1 << (QF_DEPTH - 1));
    const double f = (v - c) * inv, i = floor(f), d = f - i;
    cell = (uint32_t)(int)fmin(fmax(i + half, 0.0), 2.0 * half - 1.0);
    return d > tol && d < 1.0 - tol;
}

__device__ __forceinline__ uint32_t qf_path(const QsPath &P, double x, double y)
{
    double cx = P.cx, cy = P.cy;
    uint32_t k = 0;
#pragma unroll 1
    for (int l = 0; l < QF_DEPTH; ++l) {
        const bool qx = x >= cx, qy = y >= cy;
        k = (k << 2) | (qx ? 2u : 0u) | (qy ? 1u : 0u);
        cx += qx ? P.off[l] : -P.off[l];
        cy += qy ? P.off[l] : -P.off[l];
    }
    return k;
}

__global__ __launch_bounds__(QP_NT) void k_qs_part(QsFast F)
{
    extern __shared__ uint4 s_qp[];
    uint32_t *sKey = (uint32_t *)s_qp;  // [QF_PTS]
    __shared__ uint32_t hist[QF_BUCKETS], s_w[QP_NT / 64];
    const uint32_t tid = threadIdx.x, u = blockIdx.x;
    const uint64_t base = (uint64_t)u * QF_PTS;
    const uint32_t cnt = (uint32_t)min((unsigned long long)QF_PTS, (unsigned long long)(F.D.n - base));
    for (uint32_t b = tid; b < QF_BUCKETS; b += QP_NT)
        hist[b] = 0;
    uint32_t slow = 0;  // bit k: the thread's k-th point is near a centre
#pragma unroll 1
    for (int k0 = 0; k0 < QP_K; k0 += 8) {
        double x[8], y[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const uint64_t i = base + min(tid + (k0 + k) * QP_NT, cnt - 1u);
            x[k] = F.D.x[i];
            y[k] = F.D.y[i];
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            uint32_t ix, iy;
            const bool okx = qf_cell(x[k], F.P.cx, F.inv, F.tol, ix);
            const bool oky = qf_cell(y[k], F.P.cy, F.inv, F.tol, iy);
            slow |= (okx && oky ? 0u : 1u) << (k0 + k);
            sKey[tid + (k0 + k) * QP_NT] = spread16(ix) << 1 | spread16(iy);
        }
    }
#pragma unroll 1
    for (; slow; slow &= slow - 1u) {
        const uint32_t slot = tid + (uint32_t)__builtin_ctz(slow) * QP_NT;
        if (slot < cnt)
            sKey[slot] = qf_path(F.P, F.D.x[base + slot], F.D.y[base + slot]);
    }
    __syncthreads();
    uint32_t key[QP_K];
#pragma unroll
    for (int k = 0; k < QP_K; ++k) {
        key[k] = sKey[tid + k * QP_NT];
        if (tid + k * QP_NT < cnt)
            atomicAdd(&hist[key[k] >> QF_BIN_BITS], 1u);
    }
    __syncthreads();
    constexpr int PER = QF_BUCKETS / QP_NT;
    uint32_t h[PER], sum = 0, total;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        h[j] = hist[tid * PER + j];
        sum += h[j];
    }
    uint32_t run = owm_block_scan<QP_NT>(sum, s_w, total);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        hist[tid * PER + j] = run;
        run += h[j];
    }
    __syncthreads();
    uint16_t *tab = F.tab + (uint64_t)u * (QF_BUCKETS + 1);
    for (uint32_t b = tid; b < QF_BUCKETS; b += QP_NT)
        tab[b] = (uint16_t)hist[b];
    if (tid == 0)
        tab[QF_BUCKETS] = (uint16_t)cnt;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < QP_K; ++k) {
        const uint32_t slot = tid + k * QP_NT;
        if (slot < cnt)
            sKey[atomicAdd(&hist[key[k] >> QF_BIN_BITS], 1u)] =
                (key[k] & QF_BIN_MASK) << QF_SLOT_BITS | slot;
    }
    __syncthreads();
    uint4 *out = (uint4 *)(F.rec + base);
    for (uint32_t i = tid; i < (cnt + 3) / 4; i += QP_NT)
        out[i] = s_qp[i];
}

// Leaves of `count` nodes of depth d below their parents, four consecutive
// counts at a time: the parents' counts come back in pc (node tid + j * NT), and
// whether this thread met a split one.
template <int NT, int MAXP>
__device__ __forceinline__ bool qf_depth(const QsFast &F, int d, const uint32_t *cnt, uint32_t parents,
                                         uint32_t *s_hist, uint32_t *s_open, uint32_t (&pc)[MAXP])
{
    uint32_t open = 0;
#pragma unroll
    for (int j = 0; j < MAXP; ++j) {
        const uint32_t p = threadIdx.x + j * NT;
        pc[j] = 0;
        if (p >= parents)
            continue;
        const uint4 c = reinterpret_cast<const uint4 *>(cnt)[p];
        pc[j] = c.x + c.y + c.z + c.w;
        if (!qf_rule(F, d - 1, pc[j]))
            continue;
        const uint32_t v[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (qf_rule(F, d, v[q])) {
                ++open;
            } else if (v[q] < QS_HB) {
                atomicAdd(&s_hist[v[q]], 1u);
            } else {
                const uint32_t o = atomicAdd(F.D.novf, 1u);
                if (o < F.D.ovf_cap)
                    F.D.ovf[o] = make_uint2((uint32_t)d, v[q]);
                else
                    atomicOr(F.D.flags, 1u);
            }
        }
    }
    if (open)
        atomicAdd(s_open, open);
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < QS_HB; k += NT)
        if (s_hist[k]) {
            atomicAdd(&F.D.hist[(uint64_t)d * QS_HB + k], (unsigned long long)s_hist[k]);
            s_hist[k] = 0;
        }
    if (threadIdx.x == 0 && *s_open) {
        atomicAdd(&F.D.nopen[d], *s_open);
        *s_open = 0;
    }
    __syncthreads();
    return open != 0;
}

// Two workgroups to a CU by their LDS: 1024 threads each fill its wave slots and
// keep twice the loads of 512 in flight (20M points with clusters 121 -> 101 us,
// 99 with the next chunk's run starts loaded ahead; 60M uniform points, all
// launches: 418 -> 397 us).
constexpr int QB_NT = 1024;

// A bucket's run in sort tile s: its start, and above it its points.
__device__ __forceinline__ uint32_t qf_run(const QsFast &F, uint32_t bucket, uint32_t s)
{
    if (s >= F.nst)
        return 0;
    const uint16_t *row = F.tab + (uint64_t)s * (QF_BUCKETS + 1) + bucket;
    return (uint32_t)row[0] | (uint32_t)(row[1] - row[0]) << 16;
}

// Every run of a bucket, 16 lanes a run and four runs a group in flight:
// f(record, sort tile).  v: the run in sort tile threadIdx.x.
template <class Fn>
__device__ __forceinline__ void qf_runs(const QsFast &F, uint32_t bucket, uint32_t v, uint32_t *s_run,
                                        Fn f)
{
    const uint32_t tid = threadIdx.x, grp = tid >> 4, gl = tid & 15u;
    constexpr uint32_t G = QB_NT / 16;
    for (uint32_t s0 = 0; s0 < F.nst; s0 += QB_NT) {
        __syncthreads();
        s_run[tid] = v;
        __syncthreads();
        v = qf_run(F, bucket, s0 + QB_NT + tid);
        const uint32_t here = min((uint32_t)QB_NT, F.nst - s0);
        for (uint32_t r0 = grp; r0 < here; r0 += 4 * G) {
            uint32_t rec[4][2], len[4];
            const uint32_t *p[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t r = r0 + k * G, w = r < here ? s_run[r] : 0u;
                len[k] = w >> 16;
                p[k] = F.rec + (uint64_t)(s0 + r) * QF_PTS + (w & 0xFFFFu);
                if (gl < len[k])
                    rec[k][0] = p[k][gl];
                if (gl + 16 < len[k])
                    rec[k][1] = p[k][gl + 16];
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (gl < len[k])
                    f(rec[k][0], s0 + r0 + k * G);
                if (gl + 16 < len[k])
                    f(rec[k][1], s0 + r0 + k * G);
                for (uint32_t i = gl + 32; i < len[k]; i += 16)
                    f(p[k][i], s0 + r0 + k * G);
            }
        }
    }
    __syncthreads();
}

__global__ __launch_bounds__(QB_NT, 8) void k_qs_bins(QsFast F)
{
    extern __shared__ uint4 s_qb[];
    uint32_t *bins = (uint32_t *)s_qb;  // [QF_BINS]
    __shared__ uint32_t s_hist[QS_HB], s_run[QB_NT], s_w[QB_NT / 64];
    __shared__ uint32_t s_open, s_pts, s_nodes, s_ids, s_node;
    const uint32_t tid = threadIdx.x;
    // neighbouring buckets, whose runs share cache lines, on one XCD
    const uint32_t bucket = (blockIdx.x & 7u) * (QF_BUCKETS / 8) + (blockIdx.x >> 3);
    const uint32_t run0 = qf_run(F, bucket, tid);
    uint32_t sum = run0 >> 16, total;
    for (uint32_t s = tid + QB_NT; s < F.nst; s += QB_NT)
        sum += qf_run(F, bucket, s) >> 16;
    for (uint32_t b = tid; b < QF_BINS / 4; b += QB_NT)
        s_qb[b] = make_uint4(0, 0, 0, 0);
    for (uint32_t k = tid; k < QS_HB; k += QB_NT)
        s_hist[k] = 0;
    if (tid == 0)
        s_open = s_pts = s_nodes = 0;
    owm_block_scan<QB_NT>(sum, s_w, total);
    if (tid == 0)
        F.tot[bucket] = total;
    if (total > F.bucket_cap) {  // one workgroup would hold the call up
        if (tid == 0)
            atomicOr(F.D.flags, QF_SKEW);
        return;
    }
    qf_runs(F, bucket, run0, s_run, [&](uint32_t r, uint32_t) { atomicAdd(&bins[r >> QF_SLOT_BITS], 1u); });
    uint32_t pc[QF_BINS / 4 / QB_NT];
    const bool deep = qf_depth<QB_NT>(F, QF_DEPTH, bins, QF_BINS / 4, s_hist, &s_open, pc);
    // cells still open: their points are listed by cell for k_qs_deep
    if (__syncthreads_or(deep)) {
        for (uint32_t b = tid; b < QF_BINS; b += QB_NT)
            if (qf_rule(F, QF_DEPTH, bins[b])) {
                if (bins[b] > QF_NODE_PTS)
                    atomicOr(F.D.flags, QF_DEEP);
                atomicAdd(&s_pts, bins[b]);
                atomicAdd(&s_nodes, 1u);
            }
        __syncthreads();
        if (tid == 0) {
            s_ids = atomicAdd(F.used, s_pts);
            s_node = atomicAdd(F.used + 16, s_nodes);
            if (s_ids + s_pts > F.ids_cap || s_node + s_nodes > F.node_cap) {
                atomicOr(F.D.flags, QF_DEEP);
                s_ids = OWM_NONE;
            }
            s_pts = s_nodes = 0;
        }
        __syncthreads();
        if (s_ids != OWM_NONE) {
            for (uint32_t b = tid; b < QF_BINS; b += QB_NT) {
                const uint32_t c = bins[b];
                bins[b] = OWM_NONE;
                if (qf_rule(F, QF_DEPTH, c)) {
                    const uint32_t at = s_ids + atomicAdd(&s_pts, c);
                    bins[b] = at;
                    F.node[s_node + atomicAdd(&s_nodes, 1u)] =
                        make_uint4(bucket << QF_BIN_BITS | b, at, c, 0u);
                }
            }
            __syncthreads();
            qf_runs(F, bucket, qf_run(F, bucket, tid), s_run, [&](uint32_t r, uint32_t st) {
                const uint32_t b = r >> QF_SLOT_BITS;
                if (bins[b] != OWM_NONE)
                    F.ids[atomicAdd(&bins[b], 1u)] = st * QF_PTS + (r & QF_SLOT_MASK);
            });
        }
    }
    __syncthreads();
    uint32_t n = QF_BINS / 4;
    for (int d = QF_DEPTH - 1; d > QF_TOP; --d, n /= 4) {
#pragma unroll
        for (int j = 0; j < (int)(QF_BINS / 4 / QB_NT); ++j)
            if (tid + j * QB_NT < n)
                bins[tid + j * QB_NT] = pc[j];
        __syncthreads();
        qf_depth<QB_NT>(F, d, bins, n / 4, s_hist, &s_open, pc);
    }
}

// One workgroup per node open at depth QF_DEPTH (maxNumber policy, at most
// QF_NODE_PTS points): depth by depth, its points routed to children, counted
// and classified in LDS.
__global__ __launch_bounds__(256) void k_qs_deep(QsFast F)
{
    constexpr uint32_t NO = (QF_NODE_PTS + 1) / 2;  // open nodes hold at least two points
    __shared__ double px[QF_NODE_PTS], py[QF_NODE_PTS];
    __shared__ double2 cen[2][NO];
    __shared__ uint32_t st[QF_NODE_PTS], cnt[4 * NO], remap[4 * NO], s_n;
    const uint32_t tid = threadIdx.x;
    if (*F.D.flags & (QF_DEEP | QF_SKEW))
        return;  // the lists are not whole
    const uint32_t nodes = min(F.used[16], F.node_cap);
    for (uint32_t i = blockIdx.x; i < nodes; i += gridDim.x) {
        const uint4 nd = F.node[i];
        __syncthreads();
        for (uint32_t k = tid; k < nd.z; k += 256) {
            const uint32_t id = F.ids[nd.y + k];
            px[k] = F.D.x[id];
            py[k] = F.D.y[id];
            st[k] = 0;
        }
        if (tid == 0) {
            double cx = F.P.cx, cy = F.P.cy;
            for (int l = 0; l < QF_DEPTH; ++l) {
                const uint32_t q = nd.x >> (2 * (QF_DEPTH - 1 - l));
                cx += q & 2u ? F.P.off[l] : -F.P.off[l];
                cy += q & 1u ? F.P.off[l] : -F.P.off[l];
            }
            cen[0][0] = make_double2(cx, cy);
        }
        float r = F.r0;  // radius of the parents' depth
        for (int l = 0; l < QF_DEPTH; ++l)
            r = (float)((double)r * 0.5);
        uint32_t open = 1;
        for (int d = QF_DEPTH + 1; open && d <= QS_MAX_DEPTH; ++d) {
            const double off = (double)(r * 0.5f);
            r = (float)((double)r * 0.5);
            const double2 *pc = cen[(d - QF_DEPTH - 1) & 1];
            double2 *nc = cen[(d - QF_DEPTH) & 1];
            for (uint32_t k = tid; k < 4 * open; k += 256)
                cnt[k] = 0;
            if (tid == 0)
                s_n = 0;
            __syncthreads();
            for (uint32_t k = tid; k < nd.z; k += 256)
                if (st[k] != OWM_NONE) {
                    const double2 c = pc[st[k]];
                    const uint32_t to = 4u * st[k] + (px[k] >= c.x ? 2u : 0u) + (py[k] >= c.y ? 1u : 0u);
                    st[k] = to;
                    atomicAdd(&cnt[to], 1u);
                }
            __syncthreads();
            for (uint32_t k = tid; k < 4 * open; k += 256) {
                remap[k] = OWM_NONE;
                if (cnt[k] > F.D.max_number) {
                    const uint32_t o = atomicAdd(&s_n, 1u);
                    const double2 p = pc[k >> 2];
                    remap[k] = o;
                    nc[o] = make_double2(p.x + (k & 2u ? off : -off), p.y + (k & 1u ? off : -off));
                } else {
                    atomicAdd(&F.D.hist[(uint64_t)d * QS_HB + cnt[k]], 1ull);
                }
            }
            __syncthreads();
            for (uint32_t k = tid; k < nd.z; k += 256)
                if (st[k] != OWM_NONE)
                    st[k] = remap[st[k]];
            open = s_n;
            __syncthreads();
            if (tid == 0 && open)
                atomicAdd(&F.D.nopen[d], open);
        }
    }
}

// Depths 1..QF_TOP from the buckets' totals, then every class to host memory, in
// ascending (depth, points).
__global__ __launch_bounds__(1024) void k_qs_out(QsFast F)
{
    __shared__ __align__(16) uint32_t cnt[QF_BUCKETS];
    __shared__ uint32_t s_hist[QS_HB], s_open, s_w[16];
    const uint32_t tid = threadIdx.x;
    cnt[tid] = F.tot[tid];
    s_hist[tid] = 0;
    if (tid == 0)
        s_open = 0;
    __syncthreads();
    uint32_t pc[1];
    for (int d = QF_TOP; d > 0; --d) {
        qf_depth<1024>(F, d, cnt, 1u << (2 * (d - 1)), s_hist, &s_open, pc);
        if (tid < 1u << (2 * (d - 1)))
            cnt[tid] = pc[0];
        __syncthreads();
    }
    if (tid == 0)
        F.D.nopen[0] = 1;
    __threadfence();
    __syncthreads();
    // a wave per depth: classes of it, then their places
    __shared__ uint32_t s_no[QS_MAX_DEPTH + 1], s_at[QS_MAX_DEPTH + 2];
    if (tid <= QS_MAX_DEPTH) {
        const uint32_t v = __hip_atomic_load(F.D.nopen + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_no[tid] = v;
        F.host[4 + tid] = v;
    }
    __syncthreads();
    const uint32_t lane = tid & 63, wv = tid >> 6;
    for (int write = 0; write < 2; ++write) {
        for (uint32_t d = wv; d <= QS_MAX_DEPTH; d += 16) {
            uint32_t at = write ? s_at[d] : 0u;
            if (d && s_no[d - 1]) {
                unsigned long long v[QS_HB / 64];
#pragma unroll
                for (int k = 0; k < (int)(QS_HB / 64); ++k)
                    v[k] = __hip_atomic_load(F.D.hist + (uint64_t)d * QS_HB + k * 64 + lane,
                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                for (int k = 0; k < (int)(QS_HB / 64); ++k) {
                    const unsigned long long m = __ballot(v[k] != 0);
                    const uint32_t o = at + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
                    if (write && v[k] && o < QF_OUT)
                        reinterpret_cast<uint4 *>(F.host + 128)[o] =
                            make_uint4(d, k * 64 + lane, (uint32_t)v[k], (uint32_t)(v[k] >> 32));
                    at += (uint32_t)__popcll(m);
                }
            }
            if (!write && lane == 0)
                s_at[d + 1] = at;
        }
        __syncthreads();
        if (!write && tid == 0) {
            s_at[0] = 0;
            for (uint32_t d = 1; d <= QS_MAX_DEPTH + 1; ++d)
                s_at[d] += s_at[d - 1];
        }
        __syncthreads();
    }
    if (tid == 0) {
        F.host[0] = s_at[QS_MAX_DEPTH + 1];
        F.host[1] = *F.D.novf;
        F.host[2] = *F.D.flags;
    }
}

hipError_t qs_kernels_init()
{
    hipError_t e = hipFuncSetAttribute((const void *)k_qs_part,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, QF_PTS * 4);
    if (e == hipSuccess)
        e = hipFuncSetAttribute((const void *)k_qs_bins, hipFuncAttributeMaxDynamicSharedMemorySize,
                                QF_BINS * 4);
    return e;
}

void launch_qs_fast(hipStream_t s, const QsFast &F)
{
    hipLaunchKernelGGL(k_qs_part, dim3(F.nst), dim3(QP_NT), QF_PTS * 4, s, F);
    hipLaunchKernelGGL(k_qs_bins, dim3(QF_BUCKETS), dim3(QB_NT), QF_BINS * 4, s, F);
    if (F.D.policy == 0)
        hipLaunchKernelGGL(k_qs_deep, dim3(1024), dim3(256), 0, s, F);
    hipLaunchKernelGGL(k_qs_out, dim3(1), dim3(1024), 0, s, F);
}

}  // namespace owm
