// Scan, radix sort and compaction for gfx950 (see primitives.hpp).
#include "common.hpp"
#include "device.hpp"
#include "primitives.hpp"

namespace apspie {

namespace {

constexpr int kB = 256;          // threads per block
constexpr int kItems = 8;        // items per thread
constexpr int kTileN = kB * kItems;

// ------------------------------------------------------------------- scan
// Single-pass scan with decoupled look-back (dev::chain_tiles).  Tiles take
// ids from a ticket counter in launch order.
// elements per thread: 16, or 4 for up to kScanSmall elements, which then
// spread over four times the blocks (and one look-back window holds them all)
constexpr int kScanItems = 16, kScanItemsSmall = 4;
constexpr int64_t kScanSmall = 64 * kB * kScanItemsSmall;

template <int ITEMS>
__global__ __launch_bounds__(kB) void k_scan(const int32_t *in, int32_t *out, int64_t n,
                                             uint64_t *status, uint32_t *ticket,
                                             int64_t *total_dev) {
    constexpr int TILE = kB * ITEMS;
    __shared__ uint64_t s_scan[kB / 64 + 1];
    __shared__ uint64_t s_prefix;
    __shared__ uint32_t s_tile;
    if (threadIdx.x == 0) s_tile = dev::atomic_add_dev(ticket, 1u);
    __syncthreads();
    const int64_t tile = s_tile;
    const int64_t base = tile * TILE + (int64_t)threadIdx.x * ITEMS;
    // 16-byte accesses where the caller's arrays allow them and the tile is whole
    const bool wide = (((uintptr_t)in | (uintptr_t)out) & 15) == 0 &&
                      (tile + 1) * TILE <= n;
    int32_t v[ITEMS];
    uint64_t sum = 0;
    if (wide) {
#pragma unroll
        for (int k = 0; k < ITEMS / 4; ++k) {
            const int4 x = reinterpret_cast<const int4 *>(in + base)[k];
            v[4 * k] = x.x;
            v[4 * k + 1] = x.y;
            v[4 * k + 2] = x.z;
            v[4 * k + 3] = x.w;
        }
    } else {
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) v[k] = base + k < n ? in[base + k] : 0;
    }
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) sum += (uint64_t)(int64_t)v[k];
    uint64_t agg;
    const uint64_t excl = dev::block_exclusive_add64<kB>(sum, s_scan, agg);
    if (threadIdx.x < 64) {
        const uint64_t prefix = dev::chain_tiles(status, tile, agg);
        if (threadIdx.x == 0) {
            s_prefix = prefix;
            const int64_t ntiles = (n + TILE - 1) / TILE;
            if (tile == ntiles - 1 && total_dev) *total_dev = (int64_t)(prefix + agg);
        }
    }
    __syncthreads();
    int64_t run = (int64_t)(s_prefix + excl);
    if (wide) {
#pragma unroll
        for (int k = 0; k < ITEMS / 4; ++k) {
            int4 x;
            x.x = (int32_t)run;
            run += v[4 * k];
            x.y = (int32_t)run;
            run += v[4 * k + 1];
            x.z = (int32_t)run;
            run += v[4 * k + 2];
            x.w = (int32_t)run;
            run += v[4 * k + 3];
            reinterpret_cast<int4 *>(out + base)[k] = x;
        }
        return;
    }
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        if (base + k < n) out[base + k] = (int32_t)run;
        run += v[k];
    }
}

__global__ void k_zero_u64(uint64_t *p, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = 0;
}

// ------------------------------------------------------------- radix sort
// LSD passes over digits of at most 8 bits, on 32- or 64-bit keys.  Pass =
// per-tile digit histogram -> exclusive scan of the digit-major count table ->
// stable scatter.  A wave owns 512 consecutive elements of a tile and visits
// them in input order, 64 at a time; a lane's rank among equal digits comes
// from one ballot per digit bit and the wave's own digit counters in LDS (no
// barrier), and the waves' counters are chained once per tile.  The tile is
// then put in digit order in LDS, so that the stores of a digit's run are
// consecutive: written from input order, each element was a store into a
// line of its own, 569 us a pass for 33M pairs of 32 bits; now 33M pairs of 64
// and 32 bits take 177 us (4.5 TB/s, what a plain copy reaches) and their
// histogram 75 us (3.6 TB/s).
constexpr int kRsBlock = 512;
constexpr int kRsItems = 8;
constexpr int kRsTile = kRsBlock * kRsItems;
constexpr int kRsDigits = 256;

// Consecutive tiles on one XCD (blocks go round the 8 XCDs): their runs of a
// digit are neighbours in the output, and the partly written lines between
// them meet in one L2.
__device__ __forceinline__ int64_t xcd_tile(int64_t b, int64_t ntiles) {
    const int64_t q = ntiles / 8, r = ntiles % 8, x = b % 8;
    return x * q + min(x, r) + b / 8;
}

template <class K>
__global__ __launch_bounds__(kRsBlock) void k_rs_hist(const K *keys, int64_t n, int shift,
                                                      uint32_t mask, int32_t *counts,
                                                      int64_t ntiles) {
    __shared__ int32_t s_h[kRsDigits];
    const int64_t tile = xcd_tile(blockIdx.x, ntiles);
    if (threadIdx.x < kRsDigits) s_h[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = tile * kRsTile;
#pragma unroll
    for (int k = 0; k < kRsItems; ++k) {
        const int64_t i = base + k * kRsBlock + threadIdx.x;
        if (i < n) atomicAdd(&s_h[(uint32_t)(keys[i] >> shift) & mask], 1);
    }
    __syncthreads();
    if (threadIdx.x <= mask) counts[(int64_t)threadIdx.x * ntiles + tile] = s_h[threadIdx.x];
}

// offsets: the scanned count table, null when there is one tile
template <class K, bool HAS_VAL>
__global__ __launch_bounds__(kRsBlock) void k_rs_scatter(const K *keys, const uint32_t *vals,
                                                         K *okeys, uint32_t *ovals, int64_t n,
                                                         int shift, uint32_t mask,
                                                         const int32_t *offsets,
                                                         int64_t ntiles) {
    constexpr int NW = kRsBlock / 64;
    __shared__ K s_key[kRsTile];  // then the values
    __shared__ uint32_t s_cnt[NW][kRsDigits];
    __shared__ int32_t s_goff[kRsDigits];
    __shared__ uint64_t s_scan[NW];
    const int w = threadIdx.x / 64, lane = dev::lane_id();
    const int64_t tile = xcd_tile(blockIdx.x, ntiles);
    for (int i = threadIdx.x; i < NW * kRsDigits; i += kRsBlock) (&s_cnt[0][0])[i] = 0;
    const int64_t base = tile * kRsTile + w * (64 * kRsItems) + lane;
    K key[kRsItems];
    uint32_t val[HAS_VAL ? kRsItems : 1], pos[kRsItems];
#pragma unroll
    for (int k = 0; k < kRsItems; ++k) {
        const int64_t i = base + k * 64;
        key[k] = i < n ? keys[i] : 0;
        if (HAS_VAL) val[k] = i < n ? vals[i] : 0;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kRsItems; ++k) {
        const bool valid = base + k * 64 < n;
        const uint32_t d = (uint32_t)(key[k] >> shift) & mask;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const uint64_t bm = __ballot((d >> b) & 1u);
            peers &= ((d >> b) & 1u) ? bm : ~bm;
        }
        const int below = __popcll(peers & dev::lanemask_lt());
        const uint32_t seen = s_cnt[w][d];
        pos[k] = seen + below;
        dev::wave_sync();
        if (valid && below == 0) s_cnt[w][d] = seen + __popcll(peers);
        dev::wave_sync();
    }
    __syncthreads();
    // digit d: its waves' counts chained, then the digits
    uint32_t tot = 0, c[NW];
    if (threadIdx.x < kRsDigits) {
#pragma unroll
        for (int q = 0; q < NW; ++q) {
            c[q] = tot;
            tot += s_cnt[q][threadIdx.x];
        }
    }
    dev::Pair32 all;
    const uint32_t excl = dev::block_exclusive_add_pair<kRsBlock>(tot, 0u, s_scan, all).a;
    if (threadIdx.x < kRsDigits) {
#pragma unroll
        for (int q = 0; q < NW; ++q) s_cnt[q][threadIdx.x] = excl + c[q];
        s_goff[threadIdx.x] = offsets && threadIdx.x <= mask
                                  ? offsets[(int64_t)threadIdx.x * ntiles + tile] - (int32_t)excl
                                  : 0;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kRsItems; ++k) {
        if (base + k * 64 >= n) continue;
        pos[k] += s_cnt[w][(uint32_t)(key[k] >> shift) & mask];
        s_key[pos[k]] = key[k];
    }
    __syncthreads();
    const int32_t cnt = (int32_t)min<int64_t>(kRsTile, n - tile * kRsTile);
    int32_t to[kRsItems];
#pragma unroll
    for (int k = 0; k < kRsItems; ++k) {
        const int32_t i = k * kRsBlock + threadIdx.x;
        to[k] = -1;
        if (i < cnt) {
            const K x = s_key[i];
            const int32_t g = s_goff[(uint32_t)(x >> shift) & mask] + i;
            if ((uint64_t)g < (uint64_t)n) {  // always true for a consistent count table
                okeys[g] = x;
                to[k] = g;
            }
        }
    }
    if (HAS_VAL) {
        uint32_t *s_val = reinterpret_cast<uint32_t *>(s_key);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kRsItems; ++k)
            if (base + k * 64 < n) s_val[pos[k]] = val[k];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kRsItems; ++k)
            if (to[k] >= 0) ovals[to[k]] = s_val[k * kRsBlock + threadIdx.x];
    }
}

// ------------------------------------------------------------- compaction
__global__ __launch_bounds__(kB) void k_flag_count(const int32_t *flag, int64_t n,
                                                   int32_t *block_counts) {
    __shared__ int32_t s[kB / 64];
    const int64_t base = (int64_t)blockIdx.x * kTileN;
    int32_t c = 0;
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
        const int64_t i = base + k * kB + threadIdx.x;
        c += (i < n && flag[i] != 0) ? 1 : 0;
    }
    const uint32_t wc = (uint32_t)dev::wave_sum_u64((uint64_t)c);
    if (dev::lane_id() == 0) s[threadIdx.x / 64] = (int32_t)wc;
    __syncthreads();
    if (threadIdx.x == 0) {
        int32_t t = 0;
        for (int q = 0; q < kB / 64; ++q) t += s[q];
        block_counts[blockIdx.x] = t;
    }
}

__global__ __launch_bounds__(kB) void k_flag_write(const int32_t *flag, int64_t n,
                                                   const int32_t *block_offsets, int32_t *out) {
    constexpr int NW = kB / 64;
    __shared__ int32_t s_wc[NW];
    __shared__ int32_t s_run;
    if (threadIdx.x == 0) s_run = block_offsets[blockIdx.x];
    const int w = threadIdx.x / 64;
    const int64_t base = (int64_t)blockIdx.x * kTileN;
    for (int k = 0; k < kItems; ++k) {
        const int64_t i = base + k * kB + threadIdx.x;
        const bool f = i < n && flag[i] != 0;
        const uint64_t bm = __ballot(f);
        if (dev::lane_id() == 0) s_wc[w] = __popcll(bm);
        __syncthreads();
        if (f) {
            int pos = s_run + __popcll(bm & dev::lanemask_lt());
            for (int q = 0; q < w; ++q) pos += s_wc[q];
            if (pos < n) out[pos] = (int32_t)i;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            int t = 0;
            for (int q = 0; q < NW; ++q) t += s_wc[q];
            s_run += t;
        }
        __syncthreads();
    }
}

}  // namespace

void scan_exclusive_i32_async(Ctx *c, const int32_t *in, int32_t *out, int64_t n,
                              int64_t *total_dev) {
    if (n <= 0) {
        k_zero_u64<<<1, 64, 0, c->stream>>>((uint64_t *)total_dev, 1);
        APSPIE_LAUNCH_CHECK();
        return;
    }
    const bool small = n <= kScanSmall;
    const int64_t ntiles = ceil_div(n, kB * (small ? kScanItemsSmall : kScanItems));
    uint64_t *status = (uint64_t *)scratch(c, "scan_status", sizeof(uint64_t) * (ntiles + 1));
    uint32_t *ticket = (uint32_t *)(status + ntiles);
    k_zero_u64<<<(int)std::min<int64_t>(ceil_div(ntiles + 1, 256), 1024), 256, 0, c->stream>>>(
        status, ntiles + 1);
    const auto scan = small ? k_scan<kScanItemsSmall> : k_scan<kScanItems>;
    scan<<<(int)ntiles, kB, 0, c->stream>>>(in, out, n, status, ticket, total_dev);
    APSPIE_LAUNCH_CHECK();
}

int64_t scan_exclusive_i32(Ctx *c, const int32_t *in, int32_t *out, int64_t n) {
    int64_t *tot = (int64_t *)scratch(c, "scan_total", sizeof(int64_t));
    scan_exclusive_i32_async(c, in, out, n, tot);
    int64_t h = 0;
    APSPIE_HIP(hipMemcpyAsync(&h, tot, sizeof h, hipMemcpyDeviceToHost, c->stream));
    sync(c);
    return h;
}

int64_t scan_exclusive_dev(Ctx *c, const int32_t *in, int32_t *out, int64_t n) {
    return scan_exclusive_i32(c, in, out, n);
}

template <class K>
bool radix_sort(Ctx *c, K *ka, uint32_t *va, K *kb, uint32_t *vb, int64_t n, int lo, int bits) {
    if (n <= 1) return false;
    APSPIE_CHECK(n < INT32_MAX, APSPIE_ERR_UNSUPPORTED, "sort size must fit int32");
    const int64_t ntiles = ceil_div(n, kRsTile);
    // as many passes as 8-bit digits need, the bits dealt evenly over them
    const int passes = (bits + 7) / 8, width = (bits + passes - 1) / passes;
    int32_t *counts = nullptr, *offs = nullptr;
    int64_t *tot = nullptr;
    if (ntiles > 1) {  // one tile orders itself
        counts = (int32_t *)scratch(c, "rs_counts", sizeof(int32_t) * kRsDigits * ntiles);
        offs = (int32_t *)scratch(c, "rs_offs", sizeof(int32_t) * kRsDigits * ntiles);
        tot = (int64_t *)scratch(c, "rs_total", sizeof(int64_t));
    }
    for (int p = 0; p < passes; ++p) {
        const int w = std::min(width, bits - p * width);
        const int shift = lo + p * width;
        const uint32_t mask = (1u << w) - 1;
        if (ntiles > 1) {
            k_rs_hist<K><<<(int)ntiles, kRsBlock, 0, c->stream>>>(ka, n, shift, mask, counts,
                                                                  ntiles);
            scan_exclusive_i32_async(c, counts, offs, (int64_t)(mask + 1) * ntiles, tot);
        }
        if (va)
            k_rs_scatter<K, true><<<(int)ntiles, kRsBlock, 0, c->stream>>>(
                ka, va, kb, vb, n, shift, mask, offs, ntiles);
        else
            k_rs_scatter<K, false><<<(int)ntiles, kRsBlock, 0, c->stream>>>(
                ka, nullptr, kb, nullptr, n, shift, mask, offs, ntiles);
        APSPIE_LAUNCH_CHECK();
        std::swap(ka, kb);
        std::swap(va, vb);
    }
    return passes & 1;
}

template bool radix_sort<uint32_t>(Ctx *, uint32_t *, uint32_t *, uint32_t *, uint32_t *, int64_t,
                                   int, int);
template bool radix_sort<uint64_t>(Ctx *, uint64_t *, uint32_t *, uint64_t *, uint32_t *, int64_t,
                                   int, int);

void radix_sort_pairs(Ctx *c, uint32_t *keys, uint32_t *vals, int64_t n, int bits) {
    if (n <= 1) return;
    APSPIE_CHECK(n < INT32_MAX, APSPIE_ERR_UNSUPPORTED, "sort size must fit int32");
    uint32_t *k2 = (uint32_t *)scratch(c, "rs_k2", sizeof(uint32_t) * n);
    uint32_t *v2 = vals ? (uint32_t *)scratch(c, "rs_v2", sizeof(uint32_t) * n) : nullptr;
    if (!radix_sort(c, keys, vals, k2, v2, n, 0, bits)) return;
    APSPIE_HIP(hipMemcpyAsync(keys, k2, sizeof(uint32_t) * n, hipMemcpyDeviceToDevice, c->stream));
    if (vals)
        APSPIE_HIP(hipMemcpyAsync(vals, v2, sizeof(uint32_t) * n, hipMemcpyDeviceToDevice,
                                  c->stream));
}

// The entry point sorts whole bytes: `bits` rounded up to a multiple of 8.
void sort_pairs_dev(Ctx *c, uint32_t *keys, uint32_t *vals, int64_t n, int bits) {
    radix_sort_pairs(c, keys, vals, n, (bits + 7) / 8 * 8);
}

int64_t compact_flags(Ctx *c, const int32_t *flag, int64_t n, int32_t *idx_out) {
    if (n <= 0) return 0;
    const int64_t nb = ceil_div(n, kTileN);
    int32_t *bc = (int32_t *)scratch(c, "cf_counts", sizeof(int32_t) * nb);
    int32_t *bo = (int32_t *)scratch(c, "cf_offs", sizeof(int32_t) * nb);
    k_flag_count<<<(int)nb, kB, 0, c->stream>>>(flag, n, bc);
    const int64_t total = scan_exclusive_i32(c, bc, bo, nb);
    k_flag_write<<<(int)nb, kB, 0, c->stream>>>(flag, n, bo, idx_out);
    APSPIE_LAUNCH_CHECK();
    return total;
}

}  // namespace apspie
