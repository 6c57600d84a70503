// Single-source shortest paths as repeated (min,+) SpMSpV.
//
// Semantics: sssp() (sssp.cuh:27-115) with spmspvSssp() (spmspvSssp.cuh:91-291):
// dist[src] = 0, dist[v] = min over paths of the FP32 weight sums, unreached
// = 1.70141e+38 (sssp.cuh:48-49).  The reference multiplies with unit weights
// after the first round (sssp.cuh:83,91) and stops after a fixed depth; here
// every round uses the real weights and the loop runs to the fixed point, so
// the result equals the CPU Dijkstra of testSssp.cpp:33-115.
//
// One kernel per round: the frontier holds the vertices whose distance went
// down in the previous round; each expanded edge relaxes its head with an
// atomic min on the distance bits (non-negative floats order like their bit
// patterns), and the thread whose relaxation lowered a vertex first in this
// round appends it to the next frontier (the atomic OR that sets its bit in
// the next frontier's bitmap).
// With integer-valued weights every sum is exact, so the fixed point does not
// depend on the relaxation order.
#include <cmath>

#include "common.hpp"
#include "device.hpp"
#include "frontier.hpp"
#include "levels.hpp"
#include "timing.hpp"

namespace apspie {

namespace {

constexpr float kInf = APSPIE_SSSP_INF;

template <int TILE>
__global__ void k_sssp_seed(const int32_t *rowptr, int32_t src, int32_t *dist, FrontierBufs f0,
                            uint64_t *ctl) {
    const int32_t rs = rowptr[src];
    const int32_t d = rowptr[src + 1] - rs;
    if (threadIdx.x == 0) {
        dist[src] = dev::fbits(0.0f);
        ctl[0] = d > 0 ? ((uint64_t(1) << 32) | uint64_t(d)) : 0;
        ctl[1] = 0;
        ctl[2] = 0;
        for (int i = 4; i < 12; ++i) ctl[i] = 0;
        f0.v[0] = src;
        f0.start[0] = rs;
        f0.off[0] = 0;
    }
    for (int32_t t = threadIdx.x; (int64_t)t * TILE < d; t += blockDim.x) f0.tfirst[t] = 0;
}

// -------------------------------------------------------- pull rounds
// Direction-optimising Bellman-Ford for a CSR equal to its transpose (values
// included): a round whose frontier holds more than nnz / sssp_pull_div edges
// is pulled instead of pushed -- every vertex takes the minimum of
// dist[u] + w(v, u) over its neighbours u in the frontier (a bitmap), which
// is the same set of relaxations as pushing the frontier, with far fewer
// atomics.  Rows of at most kLight entries are scanned by one lane (8
// vertices per thread, 8 loads in flight) and written by that lane alone.
// Longer rows are walked in tiles of kHvTile entries over a list of all such
// vertices built once per graph: each thread takes kHvPer consecutive
// entries (at most two rows, since every long row has more than kHvPer
// entries), the minimum per row is reduced in LDS and applied with one atomic
// min per tile and row.  The next frontier's bitmap doubles as the claim: the
// thread whose atomic OR sets a vertex's bit appends it to the next queue.
constexpr int kDoBlock = 1024;
constexpr int kDoTile = 2048;  // tiles of the pushed queue
constexpr int32_t kLight = 32;
constexpr int kDoPer = 8;
constexpr int kDoIlp = 8;
constexpr int kHvPer = 8;
constexpr int kHvTile = kDoBlock * kHvPer;
constexpr int kHvEnt = kHvTile / (kLight + 1) + 3;  // rows meeting one tile, with slack
static_assert(kHvEnt < kDoBlock, "one claim per thread");
static_assert(kHvPer <= kLight, "a thread's entries span at most two rows");

__device__ __forceinline__ bool claim_bit(uint32_t *bits, int32_t v) {
    const uint32_t bit = 1u << (v & 31);
    return !(dev::atomic_or_dev(bits + (v >> 5), bit) & bit);
}

// A relaxation that beats the distance it read applies its atomic min without
// waiting for the result: if a racing thread of the same round lowered v
// further, v still improved in this round and belongs to the next queue, so
// the claim (the bitmap OR) decides the append alone.
struct SsspPushOp {
    static constexpr bool kStreamColumns = true;  // columns and weights stream past the L2
    const float *w;
    int32_t *dist;  // float bits
    uint32_t *fb_next;
    __device__ __forceinline__ bool probe(int32_t u, int32_t e, int32_t v, int32_t &nd) const {
        nd = dev::fbits(dev::bitsf(dist[u]) + __builtin_nontemporal_load(w + e));
        return nd < dist[v];
    }
    __device__ __forceinline__ uint32_t claim(int32_t v, int32_t nd) const {
        __hip_atomic_fetch_min(dist + v, nd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return dev::atomic_or_dev(fb_next + (v >> 5), 1u << (v & 31));
    }
    __device__ __forceinline__ bool appends(int32_t) const { return true; }
    __device__ __forceinline__ bool won(int32_t v, uint32_t old) const {
        return !((old >> (v & 31)) & 1u);
    }
};

struct HeavyLds {
    int32_t off[kHvEnt + 1], start[kHvEnt], v[kHvEnt], best[kHvEnt];
    uint64_t scan[kDoBlock / 64 + 1];
    uint64_t base;
};

union DoLds {
    ExpandLds<kDoBlock, kDoTile, true> ex;
    HeavyLds hv;
};
struct PushLds {
    ExpandLds<kDoBlock, kDoTile, true> ex;
};

struct HeavyOp {
    const int32_t *rowptr;
    __device__ __forceinline__ bool keep(int32_t v) const {
        return rowptr[v + 1] - rowptr[v] > kLight;
    }
};

__global__ void k_do_seed(const int32_t *rowptr, int32_t src, int32_t *dist, uint32_t *fb0,
                          FrontierBufs f0, uint64_t *ctl) {
    const int32_t rs = rowptr[src];
    const int32_t d = rowptr[src + 1] - rs;
    if (threadIdx.x == 0) {
        dist[src] = dev::fbits(0.0f);
        fb0[src >> 5] = 1u << (src & 31);
        ctl[0] = d > 0 ? ((uint64_t(1) << 32) | uint64_t(d)) : 0;
        f0.v[0] = src;
        f0.start[0] = rs;
        f0.off[0] = 0;
    }
    for (int32_t t = threadIdx.x; (int64_t)t * kDoTile < d; t += blockDim.x) f0.tfirst[t] = 0;
}

// two 1024-thread blocks per CU resident: at most 64 VGPRs.  Rounds of a call
// that never pulls (PULL false, the default) are a kernel of their own, which
// the pull branch's registers and LDS do not weigh on.
template <bool PULL>
__global__ __launch_bounds__(kDoBlock) __attribute__((amdgpu_waves_per_eu(8))) void
k_sssp_do_round(const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col,
                const float *__restrict__ w, int32_t nnz, int32_t m, int32_t *dist,
                const uint32_t *__restrict__ fb_cur, uint32_t *fb_next, uint32_t *fb_clear,
                FrontierBufs cur, FrontierBufs nxt, FrontierBufs heavy, uint64_t heavy_cnt,
                int32_t pull_div, uint64_t *ctl, int32_t r, Progress *prog) {
    __shared__ std::conditional_t<PULL, DoLds, PushLds> lds;
    const uint64_t cc = ctl[r % 3];
    const int32_t F = (int32_t)cnt_entries(cc), E = (int32_t)cnt_edges(cc);
    const bool pull = PULL && (int64_t)E * pull_div > (int64_t)nnz;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        ctl[(r + 2) % 3] = 0;  // the counter of round r + 1's output
        if (F > 0) {
            ctl[4] += (uint64_t)E;
            ctl[5] += (uint64_t)F;
            ctl[6] += 1;
            ctl[7] += pull ? (uint64_t)nnz : (uint64_t)E;  // CSR entries read
        }
    }
    if (blockIdx.x == 0) {
        if (F > 0) report_level(prog, r);
        else report_done(prog, ctl);
    }
    if (F == 0) return;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m / 32 + 1;
         i += (int64_t)gridDim.x * blockDim.x)
        fb_clear[i] = 0;
    uint64_t *cnt_next = ctl + (r + 1) % 3;
    if (!pull) {
        SsspPushOp op{w, dist, fb_next};
        expand_tiles<kDoBlock, kDoTile, true, true, true>(lds.ex, op, rowptr, col, nnz, cur, F,
                                                          E, nxt, cnt_next);
        return;
    }
    if constexpr (PULL) {
    const int lane = dev::lane_id();
    // short rows: one lane per vertex
    for (int64_t pbase = (int64_t)blockIdx.x * kDoBlock * kDoPer; pbase < m;
         pbase += (int64_t)gridDim.x * kDoBlock * kDoPer) {
        int32_t crs[kDoPer], cd[kDoPer], best[kDoPer], d0[kDoPer];
        uint32_t pend = 0;
#pragma unroll
        for (int k = 0; k < kDoPer; ++k) {
            const int64_t v = pbase + (int64_t)k * kDoBlock + threadIdx.x;
            const bool in = v < m;
            crs[k] = in ? rowptr[v] : 0;
            cd[k] = in ? rowptr[v + 1] - crs[k] : 0;
            d0[k] = in ? dist[v] : 0;
            best[k] = d0[k];
            if (cd[k] > 0 && cd[k] <= kLight) pend |= 1u << k;
        }
        // each lane walks its short rows one after another, kDoIlp loads in flight
        {
            int32_t e = 0, lim = 0, kk = -1, bk = 0;  // (e + kDoIlp can pass 2^31)
            for (;;) {
                if (e >= lim) {
                    if (kk >= 0) {
#pragma unroll
                        for (int k = 0; k < kDoPer; ++k)
                            if (k == kk) best[k] = bk;
                    }
                    if (!pend) break;
                    kk = __ffs(pend) - 1;
                    pend &= pend - 1;
#pragma unroll
                    for (int k = 0; k < kDoPer; ++k)
                        if (k == kk) {
                            e = crs[k];
                            lim = crs[k] + cd[k];
                            bk = best[k];
                        }
                }
                int32_t u[kDoIlp];
#pragma unroll
                for (int q = 0; q < kDoIlp; ++q) u[q] = q < lim - e ? col[e + q] : -1;
                bool f[kDoIlp];
#pragma unroll
                for (int q = 0; q < kDoIlp; ++q)
                    f[q] = u[q] >= 0 && ((fb_cur[u[q] >> 5] >> (u[q] & 31)) & 1u);
#pragma unroll
                for (int q = 0; q < kDoIlp; ++q)
                    if (f[q]) bk = min(bk, dev::fbits(dev::bitsf(dist[u[q]]) + w[e + q]));
                e += min(kDoIlp, lim - e);
            }
        }
        int32_t pc[kDoPer], prs[kDoPer], pcd[kDoPer];
#pragma unroll
        for (int k = 0; k < kDoPer; ++k) {
            const int32_t v = (int32_t)(pbase + (int64_t)k * kDoBlock + threadIdx.x);
            const bool imp = cd[k] > 0 && cd[k] <= kLight && best[k] < d0[k];
            pc[k] = v;
            prs[k] = imp ? crs[k] : 0;
            pcd[k] = imp ? cd[k] : 0;
            if (imp) dist[v] = best[k];
            const uint64_t bm = __ballot(imp);
            const int64_t wb = (pbase + (int64_t)k * kDoBlock + (threadIdx.x & ~63)) >> 5;
            if (lane == 0 && (uint32_t)bm) dev::atomic_or_dev(fb_next + wb, (uint32_t)bm);
            if (lane == 32 && (uint32_t)(bm >> 32))
                dev::atomic_or_dev(fb_next + wb + 1, (uint32_t)(bm >> 32));
        }
        produce<kDoBlock, kDoPer, kDoTile, true>(pc, prs, pcd, nxt, cnt_next, lds.hv.scan,
                                                 &lds.hv.base);
    }
    // long rows: tiles over the long-row list
    const int32_t HF = (int32_t)cnt_entries(heavy_cnt), HE = (int32_t)cnt_edges(heavy_cnt);
    if (HF == 0) return;
    HeavyLds &L = lds.hv;
    const int32_t ntiles = (int32_t)(((int64_t)HE + kHvTile - 1) / kHvTile);
    for (int32_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const int32_t i0 = min(max(heavy.tfirst[t], 0), HF - 1);
        const int32_t i1 = (t + 1 < ntiles) ? min(max(heavy.tfirst[t + 1], i0), HF - 1) : HF - 1;
        const int32_t nv = min(i1 - i0 + 1, kHvEnt);
        // off[nv]: where the row after the tile's last one starts (or HE)
        for (int32_t j = threadIdx.x; j <= nv; j += kDoBlock) {
            L.off[j] = i0 + j < HF ? heavy.off[i0 + j] : HE;
            if (j < nv) {
                L.start[j] = heavy.start[i0 + j];
                L.v[j] = heavy.v[i0 + j];
                L.best[j] = 0x7fffffff;
            }
        }
        __syncthreads();
        const uint32_t x0 = t * kHvTile + threadIdx.x * kHvPer;  // (x0 + k can pass 2^31)
        if (x0 < (uint32_t)HE) {
            const int j = dev::upper_bound_m1(L.off, 0, nv, (int32_t)x0);
            const uint32_t split = L.off[j + 1];  // first entry of row j + 1
            int32_t idx[kHvPer], u[kHvPer];
#pragma unroll
            for (int k = 0; k < kHvPer; ++k) {
                const uint32_t x = x0 + k;
                const int jj = x >= split ? j + 1 : j;
                idx[k] = -1;
                if (x < (uint32_t)HE && jj < nv) idx[k] = L.start[jj] + (int32_t)(x - L.off[jj]);
                if ((uint32_t)idx[k] >= (uint32_t)nnz) idx[k] = -1;  // guard only
                u[k] = idx[k] >= 0 ? col[idx[k]] : -1;
            }
            bool f[kHvPer];
#pragma unroll
            for (int k = 0; k < kHvPer; ++k)
                f[k] = u[k] >= 0 && ((fb_cur[u[k] >> 5] >> (u[k] & 31)) & 1u);
            int32_t b0 = 0x7fffffff, b1 = 0x7fffffff;
#pragma unroll
            for (int k = 0; k < kHvPer; ++k)
                if (f[k]) {
                    const int32_t c = dev::fbits(dev::bitsf(dist[u[k]]) + w[idx[k]]);
                    if (x0 + k >= split) b1 = min(b1, c);
                    else b0 = min(b0, c);
                }
            if (b0 != 0x7fffffff) atomicMin(&L.best[j], b0);
            if (b1 != 0x7fffffff) atomicMin(&L.best[j + 1], b1);
        }
        __syncthreads();
        int32_t hc[1] = {0}, hrs[1] = {0}, hcd[1] = {0};
        if (threadIdx.x < nv && L.best[threadIdx.x] != 0x7fffffff) {
            const int32_t j = threadIdx.x, v = L.v[j], b = L.best[j];
            if (b < dev::atomic_min_dev(dist + v, b) && claim_bit(fb_next, v)) {
                hc[0] = v;
                hrs[0] = L.start[j];
                hcd[0] = L.off[j + 1] - L.off[j];
            }
        }
        produce<kDoBlock, 1, kDoTile, true>(hc, hrs, hcd, nxt, cnt_next, L.scan, &L.base);
        __syncthreads();  // the tile's LDS is refilled next
    }
    }
}

// The long-row list of a graph (rows longer than kLight, with tile owners
// every kHvTile entries), built once and kept with the graph.
void graph_prepare_heavy(Ctx *c, Graph *g) {
    std::lock_guard<std::mutex> lock(g->derived_mu);
    if (g->heavy_mem || g->m == 0) return;
    const int64_t ent = g->nnz / (kLight + 1) + 2, tiles = g->nnz / kHvTile + 2;
    const size_t bytes = sizeof(int32_t) * (3 * ent + tiles) + 64;
    // owned by the graph (freed with it), like its other derived arrays
    APSPIE_HIP(device_malloc(c, (void **)&g->heavy_mem, bytes));
    int32_t *p = (int32_t *)g->heavy_mem;
    g->heavy_v = p;
    g->heavy_start = p + ent;
    g->heavy_off = p + 2 * ent;
    g->heavy_tfirst = p + 3 * ent;
    uint64_t *cnt = (uint64_t *)scratch(c, "sssp_heavy_cnt", 64);
    fill_i32(c, (int32_t *)cnt, 0, 2);
    FrontierBufs hb{g->heavy_v, g->heavy_start, g->heavy_off, g->heavy_tfirst};
    const int grid = fill_grid(c, kDoBlock, 2);
    k_build<kDoBlock, 8, kHvTile, true><<<grid, kDoBlock, 0, c->stream>>>(
        HeavyOp{g->rowptr}, g->rowptr, nullptr, g->m, nullptr, hb, cnt);
    APSPIE_LAUNCH_CHECK();
    APSPIE_HIP(hipMemcpyAsync(&g->heavy_cnt, cnt, 8, hipMemcpyDeviceToHost, c->stream));
    sync(c);
}

void sssp_do(Ctx *c, const Graph *g0, int32_t source, float *dist_out, int32_t pull_div) {
    Graph *g = const_cast<Graph *>(g0);
    if (pull_div > 0) graph_prepare_heavy(c, g);  // only pulled rounds walk the long-row list
    FrontierSet fs = frontier_alloc(c, "sssp", g->m, g->nnz, kDoTile, true);
    int32_t *dist = (int32_t *)dist_out;
    const int64_t words = g->m / 32 + 1;
    uint32_t *fb = (uint32_t *)scratch(c, "sssp_fb", sizeof(uint32_t) * 3 * words);
    fill_i32(c, dist, __builtin_bit_cast(int32_t, kInf), g->m);
    fill_i32(c, (int32_t *)fb, 0, 3 * words);
    fill_i32(c, (int32_t *)fs.ctl, 0, 2 * kCtlWords);
    k_do_seed<<<1, 256, 0, c->stream>>>(g->rowptr, source, dist, fb, fs.f[0], fs.ctl);
    APSPIE_LAUNCH_CHECK();
    const FrontierBufs heavy{g->heavy_v, g->heavy_start, g->heavy_off, g->heavy_tfirst};
    const int grid = fill_grid(
        c, kDoBlock, (int)std::max<int64_t>(1, opt(c, "bfs_blocks_per_cu", 8) * 256 / kDoBlock));
    KernelTimer kt(c);
    LevelFeed feed(c, levels_ahead(c));
    const auto round = pull_div > 0 ? k_sssp_do_round<true> : k_sssp_do_round<false>;
    int r = 0;
    kt.begin();
    for (; feed.more(r); ++r) {
        APSPIE_CHECK(r <= 4 * (int64_t)g->m + 256, APSPIE_ERR_DEVICE, "SSSP did not converge");
        round<<<grid, kDoBlock, 0, c->stream>>>(
            g->rowptr, g->col, g->val, (int32_t)g->nnz, g->m, dist, fb + (r % 3) * words,
            fb + ((r + 1) % 3) * words, fb + ((r + 2) % 3) * words, fs.f[r & 1],
            fs.f[(r + 1) & 1], heavy, g->heavy_cnt, pull_div, fs.ctl, r, feed.device());
        APSPIE_LAUNCH_CHECK();
    }
    kt.end(r);
    const uint64_t *h = feed.finish();
    c->stats.edges_traversed = (int64_t)h[4];
    c->stats.vertices_reached = (int64_t)h[5];
    c->stats.iterations = (int32_t)h[6];
    c->stats.edges_checked = (int64_t)h[7];
    kt.collect();
}

// ---------------------------------------------------------------- near-far
// Near-far rounds (Davidson et al.'s two-pile form of delta-stepping): a
// relaxation that lowers dist[v] below the threshold T puts v in the next
// frontier as above; one that leaves it at or above T only marks v pending.
// When a round finds the frontier empty it is a split round instead: T grows
// by delta and a sweep over all vertices moves the pending ones now below T
// into the frontier.  A pending vertex whose distance is already below the
// old T was lowered again by a near relaxation, which queued it with that
// distance: the sweep drops it (so near relaxations never clear the mark,
// and a far relaxation that lost the race to a near one costs nothing).  Vertices are expanded fewer times (mostly once, near
// their final distance); the fixed point is the same.  Relaxations and
// claims are those of the Bellman-Ford rounds above (a non-returning atomic
// min, the next bitmap's OR as the claim); a split's sweep meets every vertex
// once and appends without a claim.
//
// Light / heavy mode (delta-stepping's split of the edges, Meyer and
// Sanders): each row holds its light entries (value below delta) first, in
// a copy of the CSR kept with the graph.  A vertex claimed for the frontier
// expands only its light entries and is marked; the next split adds the
// marked vertices' heavy entries to the frontier (and clears the marks)
// while it moves the pending vertices, each with its light and its heavy
// entries.  A vertex is re-expanded with every improvement in its bucket,
// but its heavy entries, whose relaxations land at or above T whenever the
// step is delta, only once per bucket, with its distance at the bucket's
// end (R-MAT-22, width 64: 273M -> 165M expanded entries per source).  The
// fixed point is the same: every vertex whose distance drops is marked or
// moved, and a split sweeps every mark before the rounds can end.
//
// ctl words (every word a round reads was written by the previous round, and
// no word a round reads is written in that round): [0..2] frontier counter
// ring, [4..7] stats, [10 + (r & 1)] the split step of round r (float bits),
// [12 + (r & 1)] T of round r (float bits), [14 + (r & 1)]
// 1 if round r - 1 was a split, and, in the spread slots, the pending-vertex
// count left by the split of round r ([16 + 16 i + r % 3]) and the smallest
// distance among them ([16 + 16 i + 3 + r % 3], float bits, ~0 if none).
//
// The threshold of a split is T + step, at least the next float above T (T +
// step rounds to T once T exceeds step * 2^24); the step starts at delta.  A
// split that follows a split that expanded nothing doubles the step and
// jumps at least to just above the smallest pending distance the earlier
// sweep left: with weights much larger than delta, T would otherwise climb in
// maxdist / delta empty splits.  Any threshold above T gives the same fixed
// point; the jump and the doubling only bound the rounds (every second
// consecutive split moves a vertex, and sparse distances widen the step).
constexpr int kNfBlock = 1024;
constexpr int kNfPer = 8;  // vertices per thread per sweep pass

struct SsspNearOp {
    static constexpr bool kStreamColumns = true;  // columns and weights stream past the L2
    const float *w;
    int32_t *dist;  // float bits
    uint32_t *fb_next;
    uint8_t *pend;
    int32_t tbits;  // threshold T (float bits; distances are non-negative)
    const int32_t *rend;  // end of the row part a claimed vertex expands next
    uint32_t *hb;         // light / heavy mode: bit per vertex whose heavy entries are due
    __device__ __forceinline__ int32_t row_end(int32_t v) const { return rend[v]; }
    __device__ __forceinline__ bool probe(int32_t u, int32_t e, int32_t v, int32_t &nd) const {
        nd = dev::fbits(dev::bitsf(dist[u]) + __builtin_nontemporal_load(w + e));
        return nd < dist[v];
    }
    __device__ __forceinline__ uint32_t claim(int32_t v, int32_t nd) const {
        __hip_atomic_fetch_min(dist + v, nd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (nd >= tbits) {  // far: expanded by a later split round
            pend[v] = 1;
            return 0;
        }
        return dev::atomic_or_dev(fb_next + (v >> 5), 1u << (v & 31));
    }
    __device__ __forceinline__ bool appends(int32_t nd) const { return nd < tbits; }
    __device__ __forceinline__ bool won(int32_t v, uint32_t old) const {
        if ((old >> (v & 31)) & 1u) return false;
        // its light entries come next; the heavy ones once the frontier empties
        if (hb) __hip_atomic_fetch_or(hb + (v >> 5), 1u << (v & 31), __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
        return true;
    }
};

// two 1024-thread blocks per CU resident: at most 64 VGPRs
template <int TILE>
__global__ __launch_bounds__(kNfBlock) __attribute__((amdgpu_waves_per_eu(8))) void
k_sssp_nf_round(const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col,
                const float *w, int32_t nnz, int32_t m, int32_t *dist, uint32_t *fb_next,
                uint32_t *fb_clear, uint8_t *pend, FrontierBufs cur,
                FrontierBufs nxt, uint64_t *ctl, int32_t r, const int32_t *rend,
                uint32_t *hb, Progress *prog) {
    __shared__ ExpandLds<kNfBlock, TILE, true> lds;
    __shared__ uint64_t s_part[kNfBlock / 64];
    __shared__ uint32_t s_min[kNfBlock / 64];
    const uint64_t cc = ctl[r % 3];
    const int32_t F = (int32_t)cnt_entries(cc), E = (int32_t)cnt_edges(cc);
    const int32_t tbits = (int32_t)ctl[12 + (r & 1)];
    const bool split_last = ctl[14 + (r & 1)] != 0;
    const bool split = F == 0;
    // left by the previous round's split (only a split round asks)
    const uint64_t left_before = split ? nf_left(ctl, r + 2) : 0;
    const bool done = split && split_last && left_before == 0;
    const uint64_t min_before = split ? nf_min_left(ctl, r + 2) : ~0ull;
    const bool jump = split && !done && split_last && min_before != ~0ull;
    const float step = nf_next_step(dev::bitsf((int32_t)ctl[10 + (r & 1)]), jump);
    const int32_t tnext =
        split && !done ? nf_next_threshold(tbits, step, split_last, min_before) : tbits;
    // (no word read above is written by a block of this round)
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        ctl[(r + 2) % 3] = 0;
        ctl[10 + ((r + 1) & 1)] = (uint64_t)(uint32_t)dev::fbits(step);
        ctl[12 + ((r + 1) & 1)] = (uint64_t)(uint32_t)tnext;
        ctl[14 + ((r + 1) & 1)] = split ? 1 : 0;
        nf_reset(ctl, r + 1);
        if (F > 0) {
            ctl[4] += (uint64_t)E;
            ctl[5] += (uint64_t)F;
            ctl[6] += 1;
            ctl[7] += (uint64_t)E;  // CSR entries read
        } else if (!done) {
            ctl[6] += 1;  // split rounds count as rounds
        }
    }
    // finished: the last round was a split that left nothing pending and
    // found nothing below the new threshold
    if (blockIdx.x == 0) {
        if (!done) report_level(prog, r);
        else report_done(prog, ctl);
    }
    if (done) return;
    // the bitmap round r + 1 claims into (round r claims into another)
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m / 32 + 1;
         i += (int64_t)gridDim.x * blockDim.x)
        fb_clear[i] = 0;
    if (F > 0) {
        SsspNearOp op{w, dist, fb_next, pend, tbits, rend, hb};
        expand_tiles<kNfBlock, TILE, true, true, true>(lds, op, rowptr, col, nnz, cur, F, E, nxt,
                                                       ctl + ((r + 1) % 3));
        return;
    }
    // split: move the pending vertices below the new threshold into the
    // frontier, and in light / heavy mode add the heavy entries of the
    // vertices marked since the last split.  A moved vertex brings its light
    // and its heavy entries as one frontier entry, its whole row: with one for
    // each part a split could append 2 m of them, and the frontier holds m + 1
    // (2^20 vertices joined to a hub at one weight, light and heavy entries
    // each: 2,097,150).  The 32 vertices of a mark word sit in 32
    // consecutive lanes, and the word's first lane clears it after the wave
    // has read it (nothing marks during a split).
    uint64_t left = 0;
    uint32_t min_left = ~0u;  // smallest distance left pending (bits)
    const int64_t width = (int64_t)gridDim.x * kNfBlock;
    const int per = (int)min<int64_t>(kNfPer, (m + width - 1) / width);
    for (int64_t pbase = (int64_t)blockIdx.x * kNfBlock * per; pbase < m; pbase += width * per) {
        int32_t cv[kNfPer], crs[kNfPer], cd[kNfPer];
        bool take[kNfPer], drop[kNfPer], marked[kNfPer];
#pragma unroll
        for (int k = 0; k < kNfPer; ++k) {
            const int64_t v = pbase + (int64_t)k * kNfBlock + threadIdx.x;
            cv[k] = (int32_t)v;
            crs[k] = cd[k] = 0;
            take[k] = drop[k] = marked[k] = false;
            if (k >= per) continue;
            if (v < m && pend[v]) {
                const int32_t dv = dist[v];
                if (dv < tbits) drop[k] = true;  // lowered below T since: already expanded
                else if (dv < tnext) take[k] = true;
                else {
                    ++left;
                    min_left = min(min_left, (uint32_t)dv);
                }
            }
            if (hb && v < m) {
                const uint32_t word = hb[v >> 5];
                marked[k] = (word >> (v & 31)) & 1u;
                if ((v & 31) == 0 && word) hb[v >> 5] = 0;
            }
        }
#pragma unroll
        for (int k = 0; k < kNfPer; ++k) {
            if (take[k] || drop[k]) pend[cv[k]] = 0;
            // the sweep meets each vertex once: no claim needed
            if (take[k] || marked[k]) {
                crs[k] = take[k] ? rowptr[cv[k]] : rend[cv[k]];
                cd[k] = rowptr[cv[k] + 1] - crs[k];
            }
        }
        produce<kNfBlock, kNfPer, TILE, true>(cv, crs, cd, nxt, ctl + ((r + 1) % 3), lds.scan,
                                              &lds.base);
    }
    const uint64_t ws = dev::wave_sum_u64(left);
    const uint32_t wm = dev::wave_min_u32(min_left);
    if (dev::lane_id() == 0) {
        s_part[threadIdx.x / 64] = ws;
        s_min[threadIdx.x / 64] = wm;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t t = 0;
        uint32_t mn = ~0u;
        for (int q = 0; q < kNfBlock / 64; ++q) {
            t += s_part[q];
            mn = min(mn, s_min[q]);
        }
        nf_report(ctl, r, t, mn);
    }
}

// Rows split by value for the light / heavy mode: the light entries (value
// below delta) first and the heavy ones after them, each part in CSR order
// (ballot ranks), and where the light part ends.  kLfLanes lanes take a row of
// up to kLfShort entries at once, all its columns and values in flight; the
// wave then takes its longer rows one by one, counting before it writes; and
// rows above kLfWave go to a list for whole blocks, 8192 entries a step.  (One
// wave walked a hub's 200,000 entries twice, 64 at a time: R-MAT-22 6.1 -> 1.8
// ms, R-MAT-20 2.25 -> 0.49.)
constexpr int kLfBlock = 256;
constexpr int kLfLanes = 16, kLfPer = 4, kLfShort = kLfLanes * kLfPer;
constexpr int32_t kLfStep = 64 * kLfPer, kLfWave = 2048;
__global__ __launch_bounds__(kLfBlock) void k_light_first(const int32_t *__restrict__ rowptr,
                                                          const int32_t *__restrict__ col,
                                                          const float *__restrict__ val,
                                                          int32_t m, float delta, int32_t *lcol,
                                                          float *lval, int32_t *lend,
                                                          int32_t *hubs, uint32_t *nhubs) {
    constexpr int kRows = 64 / kLfLanes;
    const int lane = dev::lane_id(), sub = lane % kLfLanes;
    const uint64_t below = (1ull << lane) - 1;
    const uint64_t group = ((1ull << kLfLanes) - 1) << (lane - sub);
    const int64_t step = (int64_t)gridDim.x * (kLfBlock / 64) * kRows;
    for (int64_t v0 = (blockIdx.x * (int64_t)(kLfBlock / 64) + threadIdx.x / 64) * kRows; v0 < m;
         v0 += step) {
        const int64_t v = v0 + lane / kLfLanes;
        // (unsigned: a step past a row's end can pass 2^31)
        const uint32_t rs = v < m ? rowptr[v] : 0, re = v < m ? rowptr[v + 1] : 0;
        const bool mine = re - rs <= kLfShort;
        float x[kLfPer];
        int32_t c[kLfPer];
#pragma unroll
        for (int k = 0; k < kLfPer; ++k) {
            const uint32_t e = rs + k * kLfLanes + sub;
            const bool in = mine && e < re;
            x[k] = in ? val[e] : 0.0f;
            c[k] = in ? col[e] : 0;
        }
        uint64_t bl[kLfPer];
        uint32_t nl = 0;
#pragma unroll
        for (int k = 0; k < kLfPer; ++k) {
            const bool in = mine && rs + k * kLfLanes + sub < re;
            bl[k] = __ballot(in && x[k] < delta) & group;
            nl += __popcll(bl[k]);
        }
        uint32_t lpos = rs, hpos = rs + nl;
#pragma unroll
        for (int k = 0; k < kLfPer; ++k) {
            const bool in = mine && rs + k * kLfLanes + sub < re;
            const bool light = in && x[k] < delta;
            const uint64_t bh = __ballot(in && !light) & group;
            if (in) {
                const uint32_t p = light ? lpos + __popcll(bl[k] & below) : hpos + __popcll(bh & below);
                lcol[p] = c[k];
                lval[p] = x[k];
            }
            lpos += __popcll(bl[k]);
            hpos += __popcll(bh);
        }
        if (mine && sub == 0 && v < m) lend[v] = (int32_t)(rs + nl);
        if (re - rs > kLfWave && sub == 0) hubs[dev::atomic_add_dev(nhubs, 1u)] = (int32_t)v;
        uint64_t longm = __ballot(!mine && re - rs <= kLfWave && sub == 0);
        while (longm) {
            const int from = __ffsll((unsigned long long)longm) - 1;
            longm &= longm - 1;
            const uint32_t ls = __shfl(rs, from, 64), le = __shfl(re, from, 64);
            // kLfStep entries a step, their loads in flight; a row of one
            // step is counted from the registers it is written from
            uint32_t cnt = 0;
            if (le - ls > kLfStep) {
                for (uint32_t e0 = ls; e0 < le; e0 += kLfStep)
#pragma unroll
                    for (int k = 0; k < kLfPer; ++k) {
                        const uint32_t e = e0 + k * 64 + lane;
                        cnt += e < le && val[e] < delta ? 1u : 0u;
                    }
                cnt = (uint32_t)dev::wave_sum_u64(cnt);
            }
            uint32_t lp = ls, hp = ls + cnt;
            for (uint32_t e0 = ls; e0 < le; e0 += kLfStep) {
                float y[kLfPer];
                int32_t d[kLfPer];
                uint64_t ml[kLfPer], mh[kLfPer];
#pragma unroll
                for (int k = 0; k < kLfPer; ++k) {
                    const uint32_t e = e0 + k * 64 + lane;
                    y[k] = e < le ? val[e] : 0.0f;
                    d[k] = e < le ? col[e] : 0;
                }
                uint32_t step = 0;
#pragma unroll
                for (int k = 0; k < kLfPer; ++k) {
                    const bool in = e0 + k * 64 + lane < le, light = y[k] < delta;
                    ml[k] = __ballot(in && light);
                    mh[k] = __ballot(in && !light);
                    step += __popcll(ml[k]);
                }
                if (le - ls <= kLfStep) {
                    cnt = step;
                    hp = ls + cnt;
                }
#pragma unroll
                for (int k = 0; k < kLfPer; ++k) {
                    if (e0 + k * 64 + lane < le) {
                        const uint32_t p = (ml[k] >> lane) & 1u ? lp + __popcll(ml[k] & below)
                                                               : hp + __popcll(mh[k] & below);
                        lcol[p] = d[k];
                        lval[p] = y[k];
                    }
                    lp += __popcll(ml[k]);
                    hp += __popcll(mh[k]);
                }
            }
            if (lane == from) lend[v] = (int32_t)(ls + cnt);
        }
    }
}

constexpr int kLfHubBlock = 1024, kLfHubPer = 8;
__global__ __launch_bounds__(kLfHubBlock) void k_light_first_hubs(
    const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col,
    const float *__restrict__ val, float delta, int32_t *lcol, float *lval, int32_t *lend,
    const int32_t *hubs, const uint32_t *nhubs) {
    constexpr int kStep = kLfHubBlock * kLfHubPer;
    __shared__ uint64_t s_scan[kLfHubBlock / 64];
    const int lane = dev::lane_id();
    const uint64_t below = (1ull << lane) - 1;
    const uint32_t n = *nhubs;
    for (uint32_t q = blockIdx.x; q < n; q += gridDim.x) {
        const int32_t v = hubs[q];
        const uint32_t rs = rowptr[v], re = rowptr[v + 1];
        // a wave takes kLfHubPer * 64 consecutive entries of a step
        const uint32_t first = rs + (threadIdx.x & ~63) * kLfHubPer + lane;
        uint32_t cnt = 0;
        for (uint32_t e0 = 0; first - lane + e0 < re; e0 += kStep)
#pragma unroll
            for (int k = 0; k < kLfHubPer; ++k) {
                const uint32_t e = first + e0 + k * 64;
                cnt += e < re && val[e] < delta ? 1u : 0u;
            }
        dev::Pair32 tot;
        (void)dev::block_exclusive_add_pair<kLfHubBlock>(cnt, 0u, s_scan, tot);
        const uint32_t nl = tot.a;
        if (threadIdx.x == 0) lend[v] = (int32_t)(rs + nl);
        uint32_t lp = rs, hp = rs + nl;
        for (uint32_t e0 = 0; rs + e0 < re; e0 += kStep) {
            float x[kLfHubPer];
            int32_t c[kLfHubPer];
            uint64_t ml[kLfHubPer], mh[kLfHubPer];
            uint32_t wl = 0, wh = 0;
#pragma unroll
            for (int k = 0; k < kLfHubPer; ++k) {
                const uint32_t e = first + e0 + k * 64;
                x[k] = e < re ? val[e] : 0.0f;
                c[k] = e < re ? col[e] : 0;
            }
#pragma unroll
            for (int k = 0; k < kLfHubPer; ++k) {
                const bool in = first + e0 + k * 64 < re, light = x[k] < delta;
                ml[k] = __ballot(in && light);
                mh[k] = __ballot(in && !light);
                wl += __popcll(ml[k]);
                wh += __popcll(mh[k]);
            }
            __syncthreads();  // s_scan's last readers
            const dev::Pair32 ex = dev::block_exclusive_add_pair<kLfHubBlock>(
                lane == 0 ? wl : 0u, lane == 0 ? wh : 0u, s_scan, tot);
            uint32_t l = lp + dev::wave_read_lane(ex.a, 0);
            uint32_t h = hp + dev::wave_read_lane(ex.b, 0);
#pragma unroll
            for (int k = 0; k < kLfHubPer; ++k) {
                if (first + e0 + k * 64 < re) {
                    const uint32_t p = (ml[k] >> lane) & 1u ? l + __popcll(ml[k] & below)
                                                           : h + __popcll(mh[k] & below);
                    lcol[p] = c[k];
                    lval[p] = x[k];
                }
                l += __popcll(ml[k]);
                h += __popcll(mh[k]);
            }
            lp += tot.a;
            hp += tot.b;
        }
        __syncthreads();  // s_scan is written by the next row
    }
}

// The light-first copy of a graph's rows for width delta, built on first
// use and kept with the graph until it is destroyed: none is freed while the
// graph lives, since a call on another context may still be launching
// rounds over the copy it took (of this width or another).
Graph::LightFirst graph_light_first(Ctx *c, Graph *g, float delta) {
    std::lock_guard<std::mutex> lock(g->derived_mu);
    for (const Graph::LightFirst &x : g->lf)
        if (x.delta == delta) return x;
    const int64_t E = std::max<int64_t>(g->nnz, 1);
    const size_t ecol = ((size_t)E * 4 + 255) / 256 * 256;
    const size_t bytes = 2 * ecol + sizeof(int32_t) * ((size_t)g->m + 1);
    void *mem = nullptr;
    // owned by the graph (freed with it), like its other derived arrays
    if (device_malloc(c, &mem, bytes) != hipSuccess) {
        (void)hipGetLastError();
        throw Error{APSPIE_ERR_OOM, "no room for the light-first rows"};
    }
    int32_t *lcol = (int32_t *)mem;
    float *lval = (float *)((char *)mem + ecol);
    int32_t *lend = (int32_t *)((char *)mem + 2 * ecol);
    try {
        if (g->m > 0) {
            // every group of rows its own wave: a few dependent loads each
            const int grid = (int)std::min<int64_t>(
                ceil_div(g->m, kLfBlock / kLfLanes), 1 << 24);
            uint32_t *nhubs = (uint32_t *)scratch(
                c, "sssp_hubs", sizeof(int32_t) * ((size_t)(g->nnz / kLfWave) + 2));
            fill_i32(c, (int32_t *)nhubs, 0, 1);
            k_light_first<<<grid, kLfBlock, 0, c->stream>>>(
                g->rowptr, g->col, g->val, g->m, delta, lcol, lval, lend, (int32_t *)nhubs + 1,
                nhubs);
            k_light_first_hubs<<<fill_grid(c, kLfHubBlock, 2), kLfHubBlock, 0, c->stream>>>(
                g->rowptr, g->col, g->val, delta, lcol, lval, lend, (int32_t *)nhubs + 1, nhubs);
            APSPIE_LAUNCH_CHECK();
        }
        sync(c);
    } catch (...) {
        (void)hipFree(mem);
        throw;
    }
    g->lf.push_back(Graph::LightFirst{delta, mem, lcol, lend, lval});
    return g->lf.back();
}

template <int TILE>
void sssp_near_far(Ctx *c, const Graph *g, int32_t source, float *dist_out, float delta) {
    FrontierSet fs = frontier_alloc(c, "sssp", g->m, g->nnz, TILE, true);
    int32_t *dist = (int32_t *)dist_out;
    const int64_t words = g->m / 32 + 1;
    uint32_t *fb = (uint32_t *)scratch(c, "sssp_fb", sizeof(uint32_t) * 3 * words);
    uint8_t *pend = (uint8_t *)scratch(c, "sssp_pend", (size_t)g->m + 4);
    // light / heavy mode (option sssp_light_heavy, on by default) when the
    // weights fall on both sides of delta: a claimed vertex expands its light
    // entries (value below delta), and its heavy ones once per bucket, at
    // the next split, with its distance by then -- a heavy relaxation lands
    // at or above the threshold whenever the step is delta, so re-expanding
    // it with every improvement only repeats far marks
    float lo = 0.0f, hi = 0.0f;
    const bool lh = opt(c, "sssp_light_heavy", 1) != 0 &&
                    graph_weight_range(c, const_cast<Graph *>(g), &lo, &hi) && lo < delta &&
                    hi >= delta;
    const int32_t *col = g->col, *rend = g->rowptr + 1;
    const float *val = g->val;
    uint32_t *hb = nullptr;
    if (lh) {
        const Graph::LightFirst lf = graph_light_first(c, const_cast<Graph *>(g), delta);
        col = lf.col;
        val = lf.val;
        rend = lf.end;
        hb = (uint32_t *)scratch(c, "sssp_hb", sizeof(uint32_t) * words);
        fill_i32(c, (int32_t *)hb, 0, words);
    }
    fill_i32(c, dist, __builtin_bit_cast(int32_t, kInf), g->m);
    fill_i32(c, (int32_t *)fb, 0, 3 * words);
    fill_i32(c, (int32_t *)pend, 0, ceil_div(g->m + 4, 4));
    fill_i32(c, (int32_t *)fs.ctl, 0, 2 * kCtlWords);
    k_sssp_seed<TILE><<<1, 256, 0, c->stream>>>(g->rowptr, source, dist, fs.f[0], fs.ctl);
    fill_i32(c, (int32_t *)(fs.ctl + 12), __builtin_bit_cast(int32_t, delta), 1);  // T of round 0
    fill_i32(c, (int32_t *)(fs.ctl + 10), __builtin_bit_cast(int32_t, delta), 1);  // its step
    APSPIE_LAUNCH_CHECK();
    const int grid = fill_grid(
        c, kNfBlock, (int)std::max<int64_t>(1, opt(c, "bfs_blocks_per_cu", 8) * 256 / kNfBlock));
    KernelTimer kt(c);
    LevelFeed feed(c, levels_ahead(c));
    int r = 0;
    kt.begin();
    for (; feed.more(r); ++r) {
        APSPIE_CHECK(r <= 8 * (int64_t)g->m + 1024, APSPIE_ERR_DEVICE, "SSSP did not converge");
        k_sssp_nf_round<TILE><<<grid, kNfBlock, 0, c->stream>>>(
            g->rowptr, col, val, (int32_t)g->nnz, g->m, dist, fb + ((r + 1) % 3) * words,
            fb + ((r + 2) % 3) * words, pend, fs.f[r & 1], fs.f[(r + 1) & 1], fs.ctl, r, rend,
            hb, feed.device());
        APSPIE_LAUNCH_CHECK();
    }
    kt.end(r);
    const uint64_t *h = feed.finish();
    c->stats.edges_traversed = (int64_t)h[4];
    c->stats.vertices_reached = (int64_t)h[5];
    c->stats.iterations = (int32_t)h[6];
    c->stats.edges_checked = (int64_t)h[7];
    kt.collect();
}

}  // namespace

// The near-far split width a graph's weights suggest: ten times the largest
// weight over the mean row length, rounded to the nearest power of two of at
// least 16 -- 64 on R-MAT-22 at weights 1..255 (mean row 30; 48-64 measured
// best, 8 % under Bellman-Ford) and 512 on 2D lattices (mean row 3.6; 1.35x
// and 2.5x under Bellman-Ford at 2048^2 and 4096^2).  No upper cap: the width
// follows the weights' scale (2^32 at weights up to 1e10 on R-MAT), so the
// number of splits does not grow with the weights.  0 when the weights are
// not positive or lie within a factor of two of each other (a vertex then
// settles in the round that first reaches it).
double sssp_weight_delta(Ctx *c, Graph *g) {
    float lo = 0.0f, hi = 0.0f;
    if (g->m == 0 || !graph_weight_range(c, g, &lo, &hi) || !(lo > 0.0f) || !(hi >= 2.0f * lo))
        return 0;
    const double want = 10.0 * hi / std::max(1.0, (double)g->nnz / g->m);
    double d = 16;
    while (d < 0x1p100 && d * 1.4142135623730951 < want) d *= 2;
    return d;
}

// The width used when sssp_delta is left at -1.
//
// Sparse rows (the weights' width above every weight, so that no entry is
// heavy), kNfFrom vertices or more (fewer: Bellman-Ford rounds, 0): a wide
// bucket, for the rounds' fixed cost (about 8 us) weighs more than the
// re-expansions it adds, as long as the paths are long.  On graphs with short
// paths four times the width is all of them, Bellman-Ford rounds in effect: no
// loss against those below kNfWide vertices, but from there on the width itself
// is better.  Long paths are told from short ones by the longest row: 8 entries
// at most on lattices with a few far edges, 16 and more on random graphs of a
// mean row of 3.  Weights 1..255, ms per source, Bellman-Ford / 256 / 512 / 1024 /
// 2048 / 4096.  Lattices (width 512): 900^2 2.03 / 2.87 / 2.17 / 1.85 / 1.64 /
// 1.67, 1024^2 2.16 / 3.05 / 2.36 / 1.98 / 1.85 / 1.81, 1774^2 4.52 / 3.77 / 3.02 /
// 2.70 / 2.57 / 2.88, 2048^2 6.14 / 4.14 / 3.34 / 2.98 / 3.01 / 3.18, 2896^2 11.7 /
// 5.42 / 4.51 / 4.17 / 4.36 / 4.59.  Random edges, mean row 4 (width 512), 2^20
// vertices 0.79 / 0.80 / 0.70 / 0.68 / 0.83 / 0.84, 2^22 2.31 / 1.51 / 1.46 / 1.45 /
// 2.38 / 2.37; mean row 8 (256), 2^20 1.27 / 0.86 / 0.88 / 1.32 / 1.31 / 1.32, 2^22
// 4.43 / 1.86 / 1.85 / 4.43 / 4.47 / 4.46; mean row 12 (256), 2^22 6.02 / 3.37 /
// 4.17 / 6.03 / 6.07 / 6.09.  Smaller lattices, Bellman-Ford / 2048: 512^2 1.14 /
// 1.30, 724^2 1.43 / 1.51.
//
// Longer rows (light / heavy rounds): 1.42 * largest weight / sqrt(mean row),
// narrower on large graphs by (2^20 / m)^0.4, from kNfFrom vertices on too.
// The light-first copy makes a graph's first call longer and every later one
// shorter, ms with Bellman-Ford and with light / heavy rounds, first call /
// later ones: 786432 vertices at edge factor 16 1.10 / 1.05 and 1.29 / 0.82,
// 900000 1.36 / 1.31 and 1.39 / 0.97, at edge factor 8 0.99 / 0.93 and 1.12 /
// 0.82, 2^20 at edge factor 16 1.49 / 1.44 and 1.74 / 1.04.  (Below, less is
// gained a call: 2^18 0.67 against 0.52.)  R-MAT, edge factor 16, later calls,
// Bellman-Ford / 32 / 48 / 64 / 96: 2^17 0.45 / 0.52 / 0.46 / 0.44 / 0.44, 2^18
// 0.67 / 0.67 / 0.52 / 0.55 / 0.57, 2^20 1.39 / 1.15 / 1.08 / 1.07 / 1.12, 2^22
// 4.44 / 2.67 / 2.76 / 2.93 / 3.23; edge factor 8: 2^20 1.09 / 0.99 / 0.87 / 0.92 /
// 0.78, 2^22 2.95 / 1.99 / 1.94 / 2.00 / 2.19.
constexpr int32_t kNfFrom = 3 << 18, kNfWide = 1 << 22, kLongPathRow = 8;
double sssp_auto_delta(Ctx *c, Graph *g) {
    if (g->m < kNfFrom) return 0;
    const double d = sssp_weight_delta(c, g);
    float lo = 0.0f, hi = 0.0f;
    if (!(d > 0) || !graph_weight_range(c, g, &lo, &hi)) return 0;
    if (d > hi) {
        if (g->m < kNfWide) return 4 * d;
        return graph_max_degree(c, g) <= kLongPathRow ? 2 * d : d;
    }
    if (opt(c, "sssp_light_heavy", 1) == 0) return g->m >= (1 << 22) ? d : 0;
    const double w = 1.42 * hi / std::sqrt(std::max(1.0, (double)g->nnz / g->m)) *
                     std::min(1.0, std::pow((double)(1 << 20) / g->m, 0.4));
    return w > lo && w <= hi ? w : d;
}

// The batched SSSP width when batch_sssp_delta is left at -1: the weights'
// width where it is at least 256 (sparse rows, long paths: 512 on the
// lattices, marginally ahead of 256 at 128 and 512 sources), Bellman-Ford
// rounds otherwise (R-MAT, width 64: with many sources in flight the splits
// cost more than the re-expansions they save -- 32 / 128 sources of R-MAT-22
// measured 2.64 / 2.09 ms per query without splits, 2.68 / 2.24 at width
// 256, 4.57 / 3.05 at 64).
double sssp_batch_auto_delta(Ctx *c, Graph *g) {
    const double d = sssp_weight_delta(c, g);
    return d >= 256 ? d : 0;
}

void sssp_run(Ctx *c, const Graph *g, int32_t source, float *dist) {
    const double asked = (double)opt(c, "sssp_delta", -1);
    const double delta = asked < 0 ? sssp_auto_delta(c, const_cast<Graph *>(g)) : asked;
    if (delta > 0) {
        try {
            switch (opt(c, "bfs_tile", 2048)) {
            case 1024: sssp_near_far<1024>(c, g, source, dist, (float)delta); return;
            case 4096: sssp_near_far<4096>(c, g, source, dist, (float)delta); return;
            default: sssp_near_far<2048>(c, g, source, dist, (float)delta); return;
            }
        } catch (const Error &e) {
            // near-far rounds need a byte per vertex more than Bellman-Ford rounds,
            // and maybe the light-first rows: a default that does not fit gives way
            if (asked >= 0 || (e.status != APSPIE_ERR_OOM && e.status != APSPIE_ERR_BUDGET)) throw;
        }
        for (const char *name : {"sssp_pend", "sssp_hb", "sssp_hubs"}) scratch_drop(c, name);
    }
    // pulled rounds read w(v, u) for the edge u -> v: symmetric values only
    int32_t pull_div = (int32_t)opt(c, "sssp_pull_div", 0);
    if (pull_div > 0 && !graph_is_symmetric_weighted(c, const_cast<Graph *>(g))) pull_div = 0;
    sssp_do(c, g, source, dist, pull_div);
}

}  // namespace apspie
