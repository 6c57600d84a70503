// The SpMSpV primitive y = A^T x under a semiring.
//
// Reference: sparse mXv (mXv.cuh:249-389) and its per-algorithm copies
// (spmspvBfs.cuh:174-222, spmspvSssp.cuh:172-241, spmspvMis.cuh:245-293):
//   1. frontier column gather: start/degree of every x entry (IntervalGather)
//   2. exclusive scan of column lengths (mgpu::Scan)
//   3. load-balanced edge expansion: per expanded edge (key = column,
//      value = x_u (x) a_uv) (IntervalGather / IntervalExpand / elementMult)
//      with the mask filter applied at expansion (bfs.cuh:16-30)
//   4a. SORT path: stable key-value radix sort on the low ceil(log2 n) bits
//       (cub::DeviceRadixSort::SortPairs) then segmented reduce by key
//       (mgpu::ReduceByKey).  Each run is folded by the thread that owns its
//       head, in sorted (= expansion) order, so results are bit-identical to
//       a sequential fold in (x order, CSR order) even for non-integer data.
//   4b. ATOMIC path: atomic semiring-add into a dense row, then an
//       order-preserving compaction of the touched entries.  Exact for
//       integer-valued data and for the idempotent semirings (or/min/max);
//       (+) on non-integer values depends on the atomic order.
// Output: sorted unique indices and their values.
//
// A call is short, so what it costs are launches and host round trips: four
// kernels (fill, gather + scan, expansion, finish) that read the expanded
// edge count from device memory and choose the path themselves, and one
// round trip for the result's size, where a kernel per stage and a round trip
// per scan took 13 launches and 3 round trips (R-MAT-18, 1 % of the rows:
// 150 -> 66 us; 20 entries of R-MAT-20: 145 -> 50 us).  Only a sort of more
// than kSmallSort products is launched by the host after that round trip
// (18,608 products: 190 -> 147 us).
#include <cmath>

#include "common.hpp"
#include "device.hpp"
#include "frontier.hpp"
#include "primitives.hpp"

namespace apspie {

namespace {

constexpr int kBlock = 256;
constexpr int kTile = 2048;  // expanded edges per partition

__device__ __forceinline__ float sr_mul(int sr, float x, float a) {
    switch (sr) {
    case APSPIE_SR_PLUS_TIMES: return x * a;
    case APSPIE_SR_BOOL: return 1.0f;
    case APSPIE_SR_MIN_PLUS: return x + a;
    default: return x;  // max-priority: the source's value
    }
}

__device__ __forceinline__ float sr_add(int sr, float a, float b) {
    switch (sr) {
    case APSPIE_SR_PLUS_TIMES: return a + b;
    case APSPIE_SR_BOOL: return 1.0f;
    case APSPIE_SR_MIN_PLUS: return b < a ? b : a;
    default: return b > a ? b : a;
    }
}

// Device control words of a call, then the status words of the chained tiles.
struct SpvCtl {
    uint64_t entries;  // frontier entries with a non-empty row
    uint64_t edges;    // their expanded edges
    uint64_t count;    // entries of y
    uint32_t ticket[2];
};

// Which path a call takes, by the same rule on the host and in the kernels:
// `sort_max` < 0 forces the atomic path, `all_sort` the sort path.
struct SpvPath {
    int64_t sort_max;
    int32_t all_sort;
    int64_t cap_edges;  // the tile partition's room
    __host__ __device__ bool sorts(uint64_t edges, int32_t n) const {
        return all_sort || ((int64_t)edges <= sort_max && (int64_t)edges * 8 < n);
    }
};

// the dense row at the semiring's identity, the touched bits and the control
// words at zero
__global__ void k_spv_init(float *yd, float ident, int64_t n, uint32_t *touched, int64_t words,
                           uint64_t *ctl, int64_t nctl) {
    const int64_t gid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = gid; i < n; i += stride) yd[i] = ident;
    for (int64_t i = gid; i < words; i += stride) touched[i] = 0;
    for (int64_t i = gid; i < nctl; i += stride) ctl[i] = 0;
}

// Stages 1 and 2: row start and length of every x entry, entries with empty
// rows dropped, offsets in x order by chained tiles (one chain for the slots,
// one for the edges), and the tile partition of the edges.  Entry j's v is
// its position in x.
constexpr int kGatherItems = 8;
constexpr int kGatherTile = kBlock * kGatherItems;
__global__ __launch_bounds__(kBlock) void k_spv_gather(const int32_t *rowptr,
                                                       const int32_t *x_ind, int64_t nx,
                                                       FrontierBufs f, SpvCtl *ctl,
                                                       uint64_t *st_cnt, uint64_t *st_edge,
                                                       int64_t cap_edges) {
    __shared__ uint64_t s_scan[kBlock / 64 + 1];
    __shared__ uint64_t s_prefix[2];
    __shared__ uint32_t s_tile;
    if (threadIdx.x == 0) s_tile = dev::atomic_add_dev(&ctl->ticket[0], 1u);
    __syncthreads();
    const int64_t tile = s_tile;
    const int64_t base = tile * kGatherTile + (int64_t)threadIdx.x * kGatherItems;
    int32_t u[kGatherItems], start[kGatherItems], deg[kGatherItems];
#pragma unroll
    for (int k = 0; k < kGatherItems; ++k) u[k] = base + k < nx ? x_ind[base + k] : -1;
#pragma unroll
    for (int k = 0; k < kGatherItems; ++k) {
        start[k] = u[k] >= 0 ? rowptr[u[k]] : 0;
        deg[k] = u[k] >= 0 ? rowptr[u[k] + 1] - start[k] : 0;
    }
    uint64_t c = 0, d = 0;
#pragma unroll
    for (int k = 0; k < kGatherItems; ++k) {
        c += deg[k] > 0 ? 1 : 0;
        d += (uint64_t)deg[k];
    }
    uint64_t tc, td;
    const uint64_t ec = dev::block_exclusive_add64<kBlock>(c, s_scan, tc);
    const uint64_t ed = dev::block_exclusive_add64<kBlock>(d, s_scan, td);
    const int w = threadIdx.x / 64;
    if (w < 2) {
        const uint64_t p = dev::chain_tiles(w ? st_edge : st_cnt, tile, w ? td : tc);
        if (dev::lane_id() == 0) {
            s_prefix[w] = p;
            if (tile == (nx + kGatherTile - 1) / kGatherTile - 1) {
                if (w) ctl->edges = p + td;
                else ctl->entries = p + tc;
            }
        }
    }
    __syncthreads();
    int64_t slot = (int64_t)(s_prefix[0] + ec), o = (int64_t)(s_prefix[1] + ed);
#pragma unroll
    for (int k = 0; k < kGatherItems; ++k) {
        if (deg[k] <= 0) continue;
        // repeated x entries can pass the partition's room: the call is then
        // run again with more
        if (o + deg[k] <= cap_edges) {
            f.v[slot] = (int32_t)(base + k);
            f.start[slot] = start[k];
            f.off[slot] = (int32_t)o;
            for (int64_t t = (o + kTile - 1) / kTile; t * kTile < o + deg[k]; ++t)
                f.tfirst[t] = (int32_t)slot;
        }
        ++slot;
        o += deg[k];
    }
}

// Stages 3 and 4b: every expanded edge accumulates into the dense row.
struct SpvAtomicOp {
    int sr;
    const float *aval, *x_val;
    const int32_t *mask;
    float *yd;
    uint32_t *touched;
    __device__ __forceinline__ bool edge(int32_t i, int32_t e, int32_t v) const {
        const float prod = sr_mul(sr, x_val ? x_val[i] : 1.0f, aval ? aval[e] : 1.0f);
        if (mask && mask[v] != 0) return false;
        float *p = yd + v;
        switch (sr) {
        case APSPIE_SR_PLUS_TIMES: atomicAdd(p, prod); break;
        case APSPIE_SR_BOOL: *p = 1.0f; break;
        case APSPIE_SR_MIN_PLUS: {
            float cur = *p;
            while (prod < cur) {
                const float seen = __int_as_float(
                    atomicCAS((int *)p, __float_as_int(cur), __float_as_int(prod)));
                if (seen == cur) break;
                cur = seen;
            }
            break;
        }
        default: {
            float cur = *p;
            while (prod > cur) {
                const float seen = __int_as_float(
                    atomicCAS((int *)p, __float_as_int(cur), __float_as_int(prod)));
                if (seen == cur) break;
                cur = seen;
            }
            break;
        }
        }
        const uint32_t bit = 1u << (v & 31);
        if (!(touched[v >> 5] & bit))  // possibly stale: at worst a second atomic
            __hip_atomic_fetch_or(touched + (v >> 5), bit, __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT);
        return false;
    }
};

__global__ __launch_bounds__(kBlock) void k_spv_expand(SpvAtomicOp op, const int32_t *col,
                                                       int32_t nnz, int32_t n, FrontierBufs f,
                                                       const SpvCtl *ctl, SpvPath path) {
    const uint64_t E = ctl->edges;
    if (E == 0 || E > (uint64_t)path.cap_edges || path.sorts(E, n)) return;
    expand_tiles<kBlock, kTile, true, false, false>(op, nullptr, col, nnz, f,
                                                    (int32_t)ctl->entries, (int32_t)E, f, nullptr);
}

// Where the products of the sort path come from.
struct SpvProducts {
    int sr;
    const int32_t *col;
    const float *aval, *x_val;
    const int32_t *mask;
    int32_t nnz, n;
    // product of edge e of entry j (its x position i, row start and offset);
    // a masked output's key is past the end
    __device__ __forceinline__ void get(int32_t i, int32_t idx, uint32_t &key, float &val) const {
        key = (uint32_t)n;
        val = 0.0f;
        if ((uint32_t)idx >= (uint32_t)nnz) return;  // guard only
        const int32_t v = col[idx];
        val = sr_mul(sr, x_val ? x_val[i] : 1.0f, aval ? aval[idx] : 1.0f);
        key = mask && mask[v] != 0 ? (uint32_t)n : (uint32_t)v;
    }
};

// Up to kSmallSort products sorted and folded by one block in LDS: a thread
// holds kSmallItems of them in registers between the digit passes.
constexpr int kSmallItems = 16;
constexpr int kSmallSort = kBlock * kSmallItems;
struct SmallLds {
    uint32_t key[kSmallSort];
    float val[kSmallSort];
    uint32_t cnt[kBlock / 64][256];
    uint64_t scan[kBlock / 64 + 1];
};

__device__ __forceinline__ void small_sort(SmallLds &L, const SpvProducts &p,
                                           const FrontierBufs &f, int32_t F, int32_t E, int bits,
                                           int32_t *y_ind, float *y_val, SpvCtl *ctl) {
    constexpr int NW = kBlock / 64;
    const int w = threadIdx.x / 64, lane = dev::lane_id();
    const int32_t base = w * (64 * kSmallItems) + lane;  // item k is product base + 64 k
    int32_t *s_off = reinterpret_cast<int32_t *>(L.val);
    for (int32_t j = threadIdx.x; j < F; j += kBlock) s_off[j] = f.off[j];
    __syncthreads();
    uint32_t key[kSmallItems];
    float val[kSmallItems];
#pragma unroll
    for (int k = 0; k < kSmallItems; ++k) {
        const int32_t e = base + 64 * k;
        key[k] = 0xffffffffu;
        val[k] = 0.0f;
        if (e < E) {
            const int j = dev::upper_bound_m1(s_off, 0, F, e);
            p.get(f.v[j], f.start[j] + (e - s_off[j]), key[k], val[k]);
        }
    }
    for (int shift = 0; shift < bits; shift += 8) {
        __syncthreads();
        for (int i = threadIdx.x; i < NW * 256; i += kBlock) (&L.cnt[0][0])[i] = 0;
        __syncthreads();
        uint32_t pos[kSmallItems];
#pragma unroll
        for (int k = 0; k < kSmallItems; ++k) {
            // the items past E keep the largest digit and so the last places
            const uint32_t d = (key[k] >> shift) & 255u;
            uint64_t peers = ~0ull;
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                const uint64_t bm = __ballot((d >> b) & 1u);
                peers &= ((d >> b) & 1u) ? bm : ~bm;
            }
            const int below = __popcll(peers & dev::lanemask_lt());
            const uint32_t seen = L.cnt[w][d];
            pos[k] = seen + below;
            dev::wave_sync();
            if (below == 0) L.cnt[w][d] = seen + __popcll(peers);
            dev::wave_sync();
        }
        __syncthreads();
        uint32_t c[NW], tot = 0;
#pragma unroll
        for (int q = 0; q < NW; ++q) {
            c[q] = tot;
            tot += L.cnt[q][threadIdx.x];
        }
        dev::Pair32 all;
        const uint32_t excl = dev::block_exclusive_add_pair<kBlock>(tot, 0u, L.scan, all).a;
#pragma unroll
        for (int q = 0; q < NW; ++q) L.cnt[q][threadIdx.x] = excl + c[q];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kSmallItems; ++k) {
            const uint32_t to = pos[k] + L.cnt[w][(key[k] >> shift) & 255u];
            L.key[to] = key[k];
            L.val[to] = val[k];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kSmallItems; ++k) {
            key[k] = L.key[base + 64 * k];
            val[k] = L.val[base + 64 * k];
        }
    }
    // run heads, in order; each folds its run
    uint64_t heads[kSmallItems];
    uint32_t c = 0;
#pragma unroll
    for (int k = 0; k < kSmallItems; ++k) {
        const int32_t e = base + 64 * k;
        heads[k] = __ballot(e < E && key[k] < (uint32_t)p.n && (e == 0 || L.key[e - 1] != key[k]));
        c += __popcll(heads[k]);
    }
    __syncthreads();
    dev::Pair32 all;
    uint32_t run = dev::block_exclusive_add_pair<kBlock>(lane == 0 ? c : 0u, 0u, L.scan, all).a;
    run = dev::wave_read_lane(run, 0);
#pragma unroll
    for (int k = 0; k < kSmallItems; ++k) {
        if ((heads[k] >> lane) & 1u) {
            const int32_t e = base + 64 * k;
            float acc = val[k];
            for (int32_t q = e + 1; q < E && L.key[q] == key[k]; ++q)
                acc = sr_add(p.sr, acc, L.val[q]);
            const uint32_t at = run + __popcll(heads[k] & dev::lanemask_lt());
            y_ind[at] = (int32_t)key[k];
            y_val[at] = acc;
        }
        run += __popcll(heads[k]);
    }
    if (threadIdx.x == 0) ctl->count = all.a;
}

// The last kernel of a call: the touched entries of the dense row in order
// (chained tiles of 256 bitmap words; a wave writes 64 outputs at a time from
// two words), or a small sort by block 0.
__global__ __launch_bounds__(kBlock) void k_spv_finish(SpvProducts p, FrontierBufs f,
                                                       SpvPath path, int bits, const float *yd,
                                                       const uint32_t *touched, int32_t *y_ind,
                                                       float *y_val, SpvCtl *ctl,
                                                       uint64_t *status) {
    __shared__ SmallLds lds;
    __shared__ uint64_t s_prefix;
    __shared__ uint32_t s_tile;
    const uint64_t E = ctl->edges;
    if (E == 0 || E > (uint64_t)path.cap_edges) return;
    if (path.sorts(E, p.n)) {
        if (blockIdx.x == 0 && E <= kSmallSort)
            small_sort(lds, p, f, (int32_t)ctl->entries, (int32_t)E, bits, y_ind, y_val, ctl);
        return;
    }
    if (!touched) return;  // no dense row
    if (threadIdx.x == 0) s_tile = dev::atomic_add_dev(&ctl->ticket[1], 1u);
    __syncthreads();
    const int64_t tile = s_tile, words = (p.n + 31) / 32;
    const int64_t wi = tile * kBlock + threadIdx.x;
    const int lane = dev::lane_id();
    const uint32_t bitsw = wi < words ? touched[wi] : 0u;
    dev::Pair32 all;
    const uint32_t excl =
        dev::block_exclusive_add_pair<kBlock>(__popc(bitsw), 0u, lds.scan, all).a;
    if (threadIdx.x < 64) {
        const uint64_t prefix = dev::chain_tiles(status, tile, all.a);
        if (threadIdx.x == 0) {
            s_prefix = prefix;
            if (tile == (words + kBlock - 1) / kBlock - 1) ctl->count = prefix + all.a;
        }
    }
    __syncthreads();
    const uint32_t mine = (uint32_t)s_prefix + excl;
    const int64_t w0 = tile * kBlock + (threadIdx.x & ~63);
    for (int q = 0; q < 64; q += 2) {
        const int from = q + (lane >> 5);
        const uint32_t b = __shfl(bitsw, from, 64), at = __shfl(mine, from, 64);
        if ((b >> (lane & 31)) & 1u) {
            const int64_t v = (w0 + from) * 32 + (lane & 31);
            const uint32_t to = at + __popc(b & ((1u << (lane & 31)) - 1u));
            y_ind[to] = (int32_t)v;
            y_val[to] = yd[v];
        }
    }
}

// The sort path's larger calls: all products in expansion order ...
__global__ __launch_bounds__(kBlock) void k_spv_pairs(SpvProducts p, FrontierBufs f, int64_t F,
                                                      int64_t E, uint32_t *keys, float *vals) {
    __shared__ int32_t s_off[kTile + 1];
    const int64_t ntiles = (E + kTile - 1) / kTile;
    for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const int32_t i0 = t == 0 ? 0 : f.tfirst[t];
        const int32_t i1 = t + 1 < ntiles ? f.tfirst[t + 1] : (int32_t)(F - 1);
        const int32_t nv = min(i1 - i0 + 1, kTile + 1);
        for (int32_t j = threadIdx.x; j < nv; j += kBlock) s_off[j] = f.off[i0 + j];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kTile / kBlock; ++k) {
            const int64_t e = t * kTile + k * kBlock + threadIdx.x;
            if (e < E) {
                const int j = dev::upper_bound_m1(s_off, 0, nv, (int32_t)e);
                uint32_t key;
                float val;
                p.get(f.v[i0 + j], f.start[i0 + j] + (int32_t)(e - s_off[j]), key, val);
                keys[e] = key;
                vals[e] = val;
            }
        }
        __syncthreads();
    }
}

// ... and the fold of their sorted runs, the heads numbered by chained tiles
__global__ __launch_bounds__(kBlock) void k_spv_fold(int sr, const uint32_t *keys,
                                                     const float *vals, int64_t E, uint32_t n,
                                                     int32_t *y_ind, float *y_val, SpvCtl *ctl,
                                                     uint64_t *status) {
    constexpr int ITEMS = 8;
    __shared__ uint64_t s_scan[kBlock / 64];
    __shared__ uint64_t s_prefix;
    __shared__ uint32_t s_tile;
    if (threadIdx.x == 0) s_tile = dev::atomic_add_dev(&ctl->ticket[1], 1u);
    __syncthreads();
    const int64_t tile = s_tile;
    const int lane = dev::lane_id();
    const int64_t base = tile * (kBlock * ITEMS) + (threadIdx.x & ~63) * ITEMS + lane;
    uint32_t key[ITEMS];
    uint64_t heads[ITEMS];
    uint32_t c = 0;
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const int64_t e = base + 64 * k;
        key[k] = e < E ? keys[e] : n;
        heads[k] = __ballot(key[k] < n && (e == 0 || keys[e - 1] != key[k]));
        c += __popcll(heads[k]);
    }
    dev::Pair32 all;
    uint32_t mine = dev::block_exclusive_add_pair<kBlock>(lane == 0 ? c : 0u, 0u, s_scan, all).a;
    mine = dev::wave_read_lane(mine, 0);
    if (threadIdx.x < 64) {
        const uint64_t prefix = dev::chain_tiles(status, tile, all.a);
        if (threadIdx.x == 0) {
            s_prefix = prefix;
            if (tile == (E + kBlock * ITEMS - 1) / (kBlock * ITEMS) - 1)
                ctl->count = prefix + all.a;
        }
    }
    __syncthreads();
    int64_t run = (int64_t)s_prefix + mine;
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        if ((heads[k] >> lane) & 1u) {
            int64_t e = base + 64 * k;
            float acc = vals[e];
            for (++e; e < E && keys[e] == key[k]; ++e) acc = sr_add(sr, acc, vals[e]);
            const int64_t at = run + __popcll(heads[k] & dev::lanemask_lt());
            y_ind[at] = (int32_t)key[k];
            y_val[at] = acc;
        }
        run += __popcll(heads[k]);
    }
}

__global__ void k_fill_f32(float *p, float v, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

__global__ void k_gather_dense(const int32_t *idx, int64_t k, const float *ydense, float *y_val) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < k;
         i += (int64_t)gridDim.x * blockDim.x)
        y_val[i] = ydense[idx[i]];
}

// the dense mXv's frontier: entries above 0.5 (the reference's bitify)
__global__ void k_above_half(const float *x, int64_t n, int32_t *flag) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        flag[i] = x[i] > 0.5f ? 1 : 0;
}

__global__ void k_scatter_dense(const int32_t *idx, const float *val, int64_t k, float *y) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < k;
         i += (int64_t)gridDim.x * blockDim.x)
        y[idx[i]] = val[i];
}

float host_identity(int sr) {
    switch (sr) {
    case APSPIE_SR_MIN_PLUS: return INFINITY;
    case APSPIE_SR_MAX_FIRST: return -INFINITY;
    default: return 0.0f;
    }
}

size_t dense_bytes(const Graph *g) { return sizeof(float) * (size_t)g->n; }

// One call, with the atomic path's dense row at hand (dense) or got when the edge
// count asks for it, after a round trip.
int64_t spmspv_call(Ctx *c, const Graph *g, int sr, int64_t nx, const int32_t *x_ind,
                    const float *x_val, const int32_t *mask, int32_t *y_ind, float *y_val,
                    SpvPath sp, bool dense) {
    const int64_t n = g->n, words = n / 32 + 1;
    const int64_t gtiles = ceil_div(nx, kGatherTile), ftiles = ceil_div((n + 31) / 32, kBlock);
    FrontierBufs f;
    f.v = (int32_t *)scratch(c, "spv_v", sizeof(int32_t) * nx);
    f.start = (int32_t *)scratch(c, "spv_start", sizeof(int32_t) * nx);
    f.off = (int32_t *)scratch(c, "spv_off", sizeof(int32_t) * nx);
    float *yd = nullptr;
    uint32_t *touched = nullptr;
    auto dense_row = [&] {
        yd = (float *)scratch(c, "spv_dense", dense_bytes(g));
        touched = (uint32_t *)scratch(c, "spv_touched", sizeof(uint32_t) * words);
    };
    if (dense) dense_row();
    const int64_t nctl = sizeof(SpvCtl) / 8 + 2 * gtiles + std::max<int64_t>(ftiles, 1);
    SpvCtl *ctl = (SpvCtl *)scratch(c, "spv_ctl", sizeof(uint64_t) * nctl);
    uint64_t *st = (uint64_t *)(ctl + 1), *st_fin = st + 2 * gtiles;
    const SpvProducts prod{sr, g->col, g->val, x_val, mask, (int32_t)g->nnz, g->n};
    const int bits = bits_for(g->n);  // keys <= n
    const uint64_t *h = (const uint64_t *)c->pinned;
    // distinct x entries expand at most nnz edges; repeated ones may need
    // another run with a larger tile partition
    sp.cap_edges = g->nnz;
    for (;;) {
        f.tfirst = (int32_t *)scratch(c, "spv_tfirst",
                                      sizeof(int32_t) * (sp.cap_edges / kTile + 2));
        const int64_t work = std::max(dense ? n : 0, nctl);
        k_spv_init<<<(int)std::min<int64_t>(ceil_div(work, kBlock), 4 * c->cus), kBlock, 0,
                     c->stream>>>(yd, host_identity(sr), dense ? n : 0, touched,
                                  dense ? words : 0, (uint64_t *)ctl, nctl);
        k_spv_gather<<<(int)gtiles, kBlock, 0, c->stream>>>(g->rowptr, x_ind, nx, f, ctl, st,
                                                            st + gtiles, sp.cap_edges);
        if (dense)
            k_spv_expand<<<4 * c->cus, kBlock, 0, c->stream>>>(
                SpvAtomicOp{sr, g->val, x_val, mask, yd, touched}, g->col, (int32_t)g->nnz, g->n,
                f, ctl, sp);
        k_spv_finish<<<(int)(dense ? std::max<int64_t>(ftiles, 1) : 1), kBlock, 0, c->stream>>>(
            prod, f, sp, bits, yd, touched, y_ind, y_val, ctl, st_fin);
        APSPIE_LAUNCH_CHECK();
        APSPIE_HIP(hipMemcpyAsync(c->pinned, ctl, 3 * sizeof(uint64_t), hipMemcpyDeviceToHost,
                                  c->stream));
        // the call's timing ends with this round trip when it is the last
        APSPIE_HIP(hipEventRecord(c->ev1, c->stream));
        APSPIE_HIP(hipEventSynchronize(c->ev1));
        c->stats.host_syncs++;
        const bool fits = (int64_t)h[1] <= sp.cap_edges;
        const bool have = dense || h[1] == 0 || sp.sorts(h[1], g->n);
        if (fits && have) break;
        APSPIE_CHECK(h[1] < INT32_MAX, APSPIE_ERR_OVERFLOW,
                     "the frontier expands more than 2^31 edges");
        sp.cap_edges = std::max(sp.cap_edges, (int64_t)h[1]);
        if (!have) {
            dense_row();
            dense = true;
        }
    }
    const int64_t F = (int64_t)h[0], E = (int64_t)h[1];
    c->stats.edges_traversed = E;
    c->stats.vertices_reached = nx;
    c->stats.iterations = 1;
    if (!sp.sorts(E, g->n) || E <= kSmallSort) {
        c->ev1_recorded = true;
        return (int64_t)h[2];
    }
    // 4a over more products than one block sorts
    const int64_t rtiles = ceil_div(E, kBlock * 8);
    uint32_t *ka = (uint32_t *)scratch(c, "spv_keys", sizeof(uint32_t) * E);
    uint32_t *kb = (uint32_t *)scratch(c, "spv_keys2", sizeof(uint32_t) * E);
    float *va = (float *)scratch(c, "spv_vals", sizeof(float) * E);
    float *vb = (float *)scratch(c, "spv_vals2", sizeof(float) * E);
    uint64_t *st_fold = (uint64_t *)scratch(c, "spv_fold", sizeof(uint64_t) * rtiles);
    k_spv_pairs<<<(int)std::min<int64_t>(ceil_div(E, kTile), 4 * c->cus), kBlock, 0,
                  c->stream>>>(prod, f, F, E, ka, va);
    if (radix_sort(c, ka, (uint32_t *)va, kb, (uint32_t *)vb, E, 0, bits)) {
        std::swap(ka, kb);
        std::swap(va, vb);
    }
    fill_i32(c, (int32_t *)st_fold, 0, 2 * rtiles);
    fill_i32(c, (int32_t *)ctl->ticket, 0, 2);
    k_spv_fold<<<(int)rtiles, kBlock, 0, c->stream>>>(sr, ka, va, E, (uint32_t)g->n, y_ind, y_val,
                                                      ctl, st_fold);
    APSPIE_LAUNCH_CHECK();
    APSPIE_HIP(hipMemcpyAsync(c->pinned, ctl, 3 * sizeof(uint64_t), hipMemcpyDeviceToHost,
                              c->stream));
    APSPIE_HIP(hipEventRecord(c->ev1, c->stream));
    APSPIE_HIP(hipEventSynchronize(c->ev1));
    c->ev1_recorded = true;
    return (int64_t)h[2];
}

}  // namespace

int64_t spmspv_run(Ctx *c, const Graph *g, int sr, int64_t nx, const int32_t *x_ind,
                   const float *x_val, const int32_t *mask, int32_t *y_ind, float *y_val,
                   int path) {
    if (nx == 0 || g->nnz == 0) {
        c->stats.iterations = 1;
        return 0;
    }
    if (path == APSPIE_PATH_AUTO) path = (int)opt(c, "spmspv_path", 0);
    SpvPath sp{opt(c, "spmspv_sort_max", 1 << 16), 0, 0};
    if (path == APSPIE_PATH_SORT) sp.all_sort = 1;
    else if (path != APSPIE_PATH_AUTO) sp.sort_max = -1;
    auto call = [&](bool dense) {
        return spmspv_call(c, g, sr, nx, x_ind, x_val, mask, y_ind, y_val, sp, dense);
    };
    if (path != APSPIE_PATH_AUTO) return call(!sp.all_sort);
    // A call that may turn out to sort takes the dense row beforehand only where
    // its memory is nobody else's loss: the context has it already, or has neither
    // a budget nor an arena and the device is not full.
    if ((c->budget > 0 || c->arena) && scratch_held(c, "spv_dense") < dense_bytes(g))
        return call(false);
    try {
        return call(true);
    } catch (const Error &e) {
        if (e.status != APSPIE_ERR_OOM && e.status != APSPIE_ERR_BUDGET) throw;
    }
    scratch_drop(c, "spv_dense");
    scratch_drop(c, "spv_touched");
    return call(false);
}

// Dense mXv (mXv.cuh:110-247): the entries of x above 0.5 (bitify,
// mXv.cuh:50-55) compacted in index order (Scan + streamCompact, :142-147)
// with their values, expanded and reduced by the SpMSpV stages above, y
// zeroed (preprocessFlag, :185) and the sums scattered (scatterFloat, :205).
// Returns the sum of the frontier rows' lengths (`total`, :229); with no
// frontier y is left as it was and 0 is returned (:143-145).
int64_t mxv_dense_run(Ctx *c, const Graph *g, const float *x, float *y, int path) {
    const int grid = fill_grid(c, kBlock, 4);
    int32_t *flag = (int32_t *)scratch(c, "mxd_flag", sizeof(int32_t) * std::max(g->m, 1));
    int32_t *xi = (int32_t *)scratch(c, "mxd_xi", sizeof(int32_t) * std::max(g->m, 1));
    k_above_half<<<grid, kBlock, 0, c->stream>>>(x, g->m, flag);
    APSPIE_LAUNCH_CHECK();
    const int64_t nx = compact_flags(c, flag, g->m, xi);
    if (nx == 0) {
        c->stats.iterations = 1;
        return 0;
    }
    float *xv = (float *)scratch(c, "mxd_xv", sizeof(float) * nx);
    k_gather_dense<<<grid, kBlock, 0, c->stream>>>(xi, nx, x, xv);
    int32_t *yi = (int32_t *)scratch(c, "mxd_yi", sizeof(int32_t) * std::max(g->n, 1));
    float *yv = (float *)scratch(c, "mxd_yv", sizeof(float) * std::max(g->n, 1));
    APSPIE_LAUNCH_CHECK();
    const int64_t k = spmspv_run(c, g, APSPIE_SR_PLUS_TIMES, nx, xi, xv, nullptr, yi, yv, path);
    c->ev1_recorded = false;  // more work follows
    const int64_t total = c->stats.edges_traversed;
    c->stats.vertices_reached = nx;
    k_fill_f32<<<grid, kBlock, 0, c->stream>>>(y, 0.0f, g->n);
    if (k > 0) k_scatter_dense<<<grid, kBlock, 0, c->stream>>>(yi, yv, k, y);
    APSPIE_LAUNCH_CHECK();
    return total;
}

}  // namespace apspie
