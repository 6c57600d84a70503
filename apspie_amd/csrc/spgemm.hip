// General sparse product C = A * B over (+, x) by row-wise accumulation.
//
// Reference: the hash SpGEMM spgemm() (spgemm.cuh:131-342) with its insert
// kernels (spgemmKernel.cuh:179-343): open-addressing tables keyed by output
// coordinates, atomic value accumulation, a sort to order the output.  The
// reference tiles C in 2D over global-memory tables and drops products after
// 25 probes; here each output row gets its own accumulator sized from the
// row, so nothing is ever dropped:
//   0. p[i] = sum_{k in A_i} |B_k|, the products of row i, and
//      u[i] = min(p[i], n): no row has more distinct outputs
//   1. rows binned by u: 16 lanes of a wave, a product each, in registers
//      (p <= 16); wave + LDS table of up to 512 slots (u <= 256); block +
//      8192-slot LDS table (u <= 4096, only for n > 16384); longer rows with
//      n <= 32768 a dense LDS accumulator (value per column + a column bitmap,
//      no hashing and no sort); longer rows of wider matrices a table in
//      global memory
//   2. symbolic pass: distinct columns per row
//   3. exclusive scan -> C row offsets
//   4. numeric pass: accumulate, then write the row in column order (the
//      dense accumulator is in order already; a block table on a matrix of
//      at most 32768 columns writes each entry at its rank among the row's
//      columns, from a column bitmap; other tables compact their used slots
//      and sort only those)
// The block tiers walk a row's products load-balanced: an exclusive scan of
// |B_k| over a chunk of A_i's entries, then a wave takes 512 consecutive
// products, lane by lane.  Values are exact for integer-valued inputs; float
// (+) order otherwise follows the atomic order.
#include <algorithm>
#include <type_traits>
#include <utility>

#include "common.hpp"
#include "device.hpp"
#include "primitives.hpp"

namespace apspie {

namespace {

constexpr int kBlock = 256;
constexpr int kBig = 1024;          // threads of the dense and global tiers
constexpr int kWaveUb = 256, kWaveTable = 512;
constexpr int kBlockUb = 4096, kBlockTable = 8192;
constexpr int kDenseFrom = 64;      // products of the shortest dense rows (up to kDenseN / 2 columns)
constexpr int kDenseN = 32768;      // dense accumulator: value + bit per column
constexpr int kChunk = 1024;        // entries of A_i staged per enumeration chunk
constexpr int kRun = 8;             // products per lane whose loads are in flight together
constexpr int kTinyUb = 16;         // products of a row held by 16 lanes
constexpr int kBinPer = 8;          // rows per thread of the binning
constexpr int64_t kHeavy = 32768;   // dense rows with more products are taken first
// words of the control block (16 uint32, zero before a call): rows per bin,
// the global bin's largest u, tiny rows, the dense kernels' row tickets
enum { kCtlBin = 0, kCtlMaxU = 4, kCtlTiny = 5, kCtlTicket = 6 };
constexpr int32_t kEmpty = 0x7fffffff;  // sorts after every column id

// p[i] = products of row i.  16 lanes per row: a wave per row left 60 of its
// lanes idle on rows of four entries.  Rows of more than kBoundRow entries take
// the whole wave, with several loads in flight (R-MAT-14, a hub of 3,665
// entries: 57 -> 22 us; 512^2 lattice 70 -> 14).
constexpr int kBoundRow = 128;
__global__ __launch_bounds__(kBlock) void k_row_bound(const int32_t *__restrict__ arp,
                                                      const int32_t *__restrict__ acol,
                                                      const int32_t *__restrict__ brp, int32_t m,
                                                      int64_t *__restrict__ prods) {
    const int j = threadIdx.x & 15;
    const int64_t step = (int64_t)gridDim.x * (kBlock / 16);
    const int64_t i0 = (int64_t)blockIdx.x * (kBlock / 16) + threadIdx.x / 64 * 4;
    for (int64_t w = i0; w < m; w += step) {  // the wave's first row
        const int64_t i = w + (threadIdx.x / 16 & 3);
        // (unsigned: a step past a row's end can pass 2^31)
        const uint32_t b = i < m ? arp[i] : 0, e1 = i < m ? arp[i + 1] : 0;
        const bool is_long = e1 - b > kBoundRow;
        uint64_t s = 0;
        if (!is_long)
            for (uint32_t e = b + j; e < e1; e += 16) {
                const int32_t k = acol[e];
                s += (uint64_t)(brp[k + 1] - brp[k]);
            }
#pragma unroll
        for (int d = 8; d >= 1; d >>= 1) s += __shfl_xor(s, d, 16);
        if (j == 0 && i < m && !is_long) prods[i] = (int64_t)s;
        for (uint64_t todo = __ballot(is_long && j == 0); todo; todo &= todo - 1) {
            const int src = __ffsll((unsigned long long)todo) - 1;
            const uint32_t lb = __shfl(b, src, 64), le = __shfl(e1, src, 64);
            uint64_t t = 0;
#pragma unroll 8
            for (uint32_t e = lb + dev::lane_id(); e < le; e += 64) {
                const int32_t k = acol[e];
                t += (uint64_t)(brp[k + 1] - brp[k]);
            }
            t = dev::wave_sum_u64(t);
            if (dev::lane_id() == 0) prods[w + src / 16] = (int64_t)t;
        }
    }
}

// bins: 0 wave, 1 block-LDS, 2 dense, 3 block-global, or with the dense tier
// its rows of more than kHeavy products; 4 tiny rows, which share the last
// bin's slots from their other end (a row is in one bin).  A block takes
// kBinPer rows per thread and reserves its slots with one atomic per bin: one
// per wave and bin took 50 us at 2^18 rows.
__global__ __launch_bounds__(kBlock) void k_bin_rows(const int64_t *prods, const int32_t *arp,
                                                     int32_t m, int32_t n, int32_t wave_ub,
                                                     int32_t block_ub, bool dense_ok,
                                                     int32_t *lists, uint32_t *ctl,
                                                     int32_t *row_nnz) {
    __shared__ uint32_t s_cnt[5], s_base[5], s_max;
    // fewer rows per thread where they would not fill the grid
    const int64_t all = (int64_t)gridDim.x * kBlock;
    const int per = (int)min<int64_t>(kBinPer, (m + all - 1) / all);
    const int64_t width = (int64_t)kBlock * per;
    for (int64_t r0 = blockIdx.x * width; r0 < m; r0 += gridDim.x * width) {
        if (threadIdx.x < 5) s_cnt[threadIdx.x] = 0;
        if (threadIdx.x == 5) s_max = 0;
        __syncthreads();
        int bin[kBinPer];
        uint32_t slot[kBinPer];
#pragma unroll
        for (int k = 0; k < kBinPer; ++k) {
            const int64_t r = r0 + k * kBlock + threadIdx.x;
            const int64_t p = k < per && r < m ? prods[r] : 0, u = min<int64_t>(p, n);
            bin[k] = p == 0 ? -1
                     : p <= kTinyUb && p <= wave_ub && arp[r + 1] - arp[r] <= 16 ? 4
                     : u <= wave_ub ? 0
                     : u <= block_ub ? 1
                     : dense_ok && p <= kHeavy ? 2 : 3;
            if (k < per && r < m && p == 0) row_nnz[r] = 0;
            slot[k] = 0;
#pragma unroll
            for (int b = 0; b < 5; ++b) {
                const uint64_t mask = __ballot(bin[k] == b);
                if (!mask) continue;
                const int leader = __ffsll((unsigned long long)mask) - 1;
                uint32_t at = 0;
                if (dev::lane_id() == leader) at = atomicAdd(&s_cnt[b], (uint32_t)__popcll(mask));
                at = __shfl(at, leader, 64);
                if (bin[k] == b) slot[k] = at + __popcll(mask & dev::lanemask_lt());
            }
            if (bin[k] == 3) atomicMax(&s_max, (uint32_t)u);
        }
        __syncthreads();
        if (threadIdx.x < 5 && s_cnt[threadIdx.x])
            s_base[threadIdx.x] = dev::atomic_add_dev(
                ctl + (threadIdx.x < 4 ? kCtlBin + threadIdx.x : kCtlTiny), s_cnt[threadIdx.x]);
        if (threadIdx.x == 5 && s_max) atomicMax(ctl + kCtlMaxU, s_max);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kBinPer; ++k)
            if (bin[k] >= 0) {
                const int64_t at = (int64_t)s_base[bin[k]] + slot[k];
                lists[bin[k] == 4 ? 4 * (int64_t)m - 1 - at : bin[k] * (int64_t)m + at] =
                    (int32_t)(r0 + k * kBlock + threadIdx.x);
            }
        __syncthreads();  // s_cnt is reset by the next pass
    }
}

// f(lanes behind, value of the lane that far behind in the 16, cyclically)
// for 15 .. 1 lanes behind: the 16 lanes after this one, in their order
template <class F, int... R>
__device__ __forceinline__ void rotate16(std::integer_sequence<int, R...>, F &&f) {
    (f(std::integral_constant<int, 15 - R>{}), ...);
}
template <int R>
__device__ __forceinline__ int32_t ror16(int32_t x) {  // row_ror:R
    return __builtin_amdgcn_update_dpp(0, x, 0x120 + R, 0xf, 0xf, false);
}

// Tiny rows (at most 16 products from at most 16 entries): 16 lanes per row, a
// product per lane, everything in registers.  The first lane of a column owns
// it: its place in the row is the number of smaller owned columns, its value
// the sum of the column's products in the order of A_i's entries; the lanes
// meet by DPP rotations.  A wave per row with a sorted 512-slot table took
// 3.3 ms for the 2^18 rows of a 512^2 lattice.
template <bool NUMERIC>
__global__ __launch_bounds__(kBlock) void k_rows_tiny(const int32_t *last, const uint32_t *cnt,
                                                      const int32_t *__restrict__ arp,
                                                      const int32_t *__restrict__ acol,
                                                      const float *__restrict__ aval,
                                                      const int32_t *__restrict__ brp,
                                                      const int32_t *__restrict__ bcol,
                                                      const float *__restrict__ bval,
                                                      int32_t *row_nnz, const int32_t *crp,
                                                      int32_t *ccol, float *cval) {
    constexpr int NG = kBlock / 16;
    const int j = threadIdx.x & 15;
    const int64_t n = cnt[0];
    for (int64_t i = (int64_t)blockIdx.x * NG + threadIdx.x / 16; i < n;
         i += (int64_t)gridDim.x * NG) {
        const int32_t r = last[-i], a0 = arp[r], an = arp[r + 1] - a0;
        int32_t b0 = 0;
        uint32_t len = 0;
        float av = 1.0f;
        if (j < an) {
            const int32_t k = acol[a0 + j];
            b0 = brp[k];
            len = (uint32_t)(brp[k + 1] - b0);
            if (NUMERIC && aval) av = aval[a0 + j];
        }
        const int32_t inc = (int32_t)dev::row16_inclusive_add(len), pre = inc - (int32_t)len;
        const int32_t total = __shfl(inc, 15, 16);
        // the last entry that starts at or before product j (an empty one
        // starts where the next does)
        int t = 0;
#pragma unroll
        for (int d = 8; d >= 1; d >>= 1)
            if (__shfl(pre, t + d, 16) <= j) t += d;
        const int32_t e = __shfl(b0, t, 16) + j - __shfl(pre, t, 16);
        const float a = NUMERIC ? __shfl(av, t, 16) : 1.0f;
        int32_t key = kEmpty;
        float v = 0.0f;
        if (j < total) {
            key = bcol[e];
            if (NUMERIC) v = a * (bval ? bval[e] : 1.0f);
        }
        bool own = key != kEmpty;
        rotate16(std::make_integer_sequence<int, 15>{}, [&](auto R) {
            if (ror16<R.value>(key) == key && j >= R.value) own = false;
        });
        if (!NUMERIC) {
            const uint32_t owned = uint32_t(__ballot(own) >> (dev::lane_id() & 48)) & 0xffffu;
            if (j == 0) row_nnz[r] = __popc(owned);
            continue;
        }
        const int32_t mine = own ? key : kEmpty;
        int32_t rank = 0;
        float sum = 0.0f + v;
        rotate16(std::make_integer_sequence<int, 15>{}, [&](auto R) {
            rank += ror16<R.value>(mine) < key ? 1 : 0;
            const float w = __int_as_float(ror16<R.value>(__float_as_int(v)));
            if (ror16<R.value>(key) == key) sum += w;
        });
        if (own) {
            const int32_t at = crp[r] + rank;
            ccol[at] = key;
            cval[at] = sum;
        }
    }
}

// insert key; returns true if this call created the entry
__device__ __forceinline__ bool tab_insert(int32_t *keys, uint32_t mask, int32_t key,
                                           uint32_t *slot_out) {
    uint32_t h = dev::fib_slot((uint32_t)key, mask);
    for (;;) {
        const int32_t prev = atomicCAS(keys + h, kEmpty, key);
        if (prev == kEmpty || prev == key) {
            *slot_out = h;
            return prev == kEmpty;
        }
        h = (h + 1) & mask;
    }
}

// bitonic sort of (keys, vals) of power-of-two size `size` by `nthreads`
// cooperating threads (thread index tid); `barrier` orders the stages
template <class V, class Barrier>
__device__ __forceinline__ void bitonic(int32_t *keys, V *vals, uint32_t size, int tid,
                                        int nthreads, Barrier barrier) {
    for (uint32_t k = 2; k <= size; k <<= 1) {
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            for (uint32_t i = tid; i < size; i += nthreads) {
                const uint32_t p = i ^ j;
                if (p > i) {
                    const bool up = (i & k) == 0;
                    const int32_t a = keys[i], b = keys[p];
                    if ((a > b) == up) {
                        keys[i] = b;
                        keys[p] = a;
                        if (vals) {
                            const V t = vals[i];
                            vals[i] = vals[p];
                            vals[p] = t;
                        }
                    }
                }
            }
            barrier();
        }
    }
}

// Small rows: one wave per row, an LDS table of the power of two that holds
// twice the row's products.  64 entries of A_i are read at once and their
// products dealt to the lanes (entry by entry, a row of many short B rows was
// a chain of dependent loads); only the used slots are sorted.
template <bool NUMERIC>
__device__ __forceinline__ void wave_row(int32_t r, const int32_t *arp, const int32_t *acol,
                                         const float *aval, const int32_t *brp,
                                         const int32_t *bcol, const float *bval, uint32_t u,
                                         int32_t *keys, double *vals, int32_t *row_nnz,
                                         const int32_t *crp, int32_t *ccol, float *cval) {
    const int tid = dev::lane_id();
    uint32_t tsize = 64;
    while (tsize < 2 * u) tsize <<= 1;  // u <= kWaveUb: at most kWaveTable
    const uint32_t mask = tsize - 1;
    for (uint32_t s = tid; s < tsize; s += 64) {
        keys[s] = kEmpty;
        if (NUMERIC) vals[s] = 0.0;
    }
    dev::wave_sync();
    uint32_t created = 0;
    const uint32_t a1 = arp[r + 1];  // (a step past the row's end can pass 2^31)
    for (uint32_t e0 = arp[r]; e0 < a1; e0 += 64) {
        int32_t b0 = 0;
        uint32_t len = 0;
        float av = 1.0f;
        if (e0 + tid < a1) {
            const int32_t k = acol[e0 + tid];
            b0 = brp[k];
            len = (uint32_t)(brp[k + 1] - b0);
            if (NUMERIC && aval) av = aval[e0 + tid];
        }
        const uint32_t inc = dev::wave_inclusive_add(len);
        const int32_t pre = (int32_t)(inc - len), total = (int32_t)dev::wave_read_lane(inc, 63);
        for (int32_t x0 = 0; x0 < total; x0 += 64) {
            const int32_t x = min(x0 + tid, total - 1);
            int t = 0;
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1)
                if (__shfl(pre, t + d, 64) <= x) t += d;
            const int32_t f = __shfl(b0, t, 64) + x - __shfl(pre, t, 64);
            const float a = NUMERIC ? __shfl(av, t, 64) : 1.0f;
            if (x0 + tid < total) {
                uint32_t slot;
                created += tab_insert(keys, mask, bcol[f], &slot) ? 1u : 0u;
                if (NUMERIC) atomicAdd(vals + slot, double(a * (bval ? bval[f] : 1.0f)));
            }
        }
    }
    if (!NUMERIC) {
        const uint32_t n = dev::wave_read_lane(dev::wave_inclusive_add(created), 63);
        if (tid == 0) row_nnz[r] = (int32_t)n;
        dev::wave_sync();
        return;
    }
    dev::wave_sync();
    // used slots to the front (a slot's place never lies beyond those read)
    uint32_t nz = 0;
    for (uint32_t s0 = 0; s0 < tsize; s0 += 64) {
        const int32_t k = keys[s0 + tid];
        const double v = vals[s0 + tid];
        const uint64_t used = __ballot(k != kEmpty);
        dev::wave_sync();
        if (k != kEmpty) {
            const uint32_t at = nz + (uint32_t)__popcll(used & dev::lanemask_lt());
            keys[at] = k;
            vals[at] = v;
        }
        nz += (uint32_t)__popcll(used);
        dev::wave_sync();
    }
    uint32_t p = 1;
    while (p < nz) p <<= 1;
    for (uint32_t s = nz + tid; s < p; s += 64) keys[s] = kEmpty;
    dev::wave_sync();
    bitonic(keys, vals, p, tid, 64, [] { dev::wave_sync(); });
    const int32_t c0 = crp[r];
    for (uint32_t s = tid; s < nz; s += 64) {
        ccol[c0 + s] = keys[s];
        cval[c0 + s] = (float)vals[s];
    }
    dev::wave_sync();
}

template <bool NUMERIC>
__global__ __launch_bounds__(kBlock) void k_rows_wave(const int32_t *rows, const uint32_t *cnt,
                                                      const int32_t *arp, const int32_t *acol,
                                                      const float *aval, const int32_t *brp,
                                                      const int32_t *bcol, const float *bval,
                                                      const int64_t *prods, int32_t ncols,
                                                      int32_t *row_nnz, const int32_t *crp,
                                                      int32_t *ccol, float *cval) {
    constexpr int NW = kBlock / 64;
    __shared__ int32_t s_keys[NW][kWaveTable];
    __shared__ double s_vals[NUMERIC ? NW : 1][NUMERIC ? kWaveTable : 1];
    const int w = threadIdx.x / 64;
    const int32_t n = (int32_t)cnt[0];
    for (int32_t i = blockIdx.x * NW + w; i < n; i += gridDim.x * NW)
        wave_row<NUMERIC>(rows[i], arp, acol, aval, brp, bcol, bval,
                          (uint32_t)min<int64_t>(prods[rows[i]], ncols), s_keys[w],
                          NUMERIC ? s_vals[w] : nullptr, row_nnz, crp, ccol, cval);
}

// Largest j < cn with pre[j] <= x (pre[0] <= x, cn <= 1024), found by a whole
// wave with two reads per lane.
__device__ __forceinline__ int wave_find(const int32_t *pre, int cn, int32_t x) {
    static_assert(kChunk == 1024, "64 lanes, 16 entries each");
    const int lane = dev::lane_id();
    const int c = 16 * (__popcll(__ballot(16 * lane < cn && pre[min(16 * lane, cn)] <= x)) - 1);
    return c + __popcll(__ballot(lane < 16 && c + lane < cn && pre[min(c + lane, cn)] <= x)) - 1;
}

// A staged entry of A_i.
struct Entry {
    int32_t base;  // product x of the chunk is B's entry base + x
    float a;
};

// One wave's share of a chunk's W products: RUN slices of 64 consecutive ones
// from w0, a product per lane and slice, so that a long B row is read
// coalesced and its entry found once (R-MAT-14: 91 % of the products lie in B
// rows of 256 entries and more).  All loads of B go out before the first
// product is applied.
template <int RUN, class F>
__device__ __forceinline__ void wave_products(const int32_t *pre, const Entry *ent, int cn,
                                              uint32_t w0, uint32_t W,  // W < 2^31
                                              const int32_t *__restrict__ bcol,
                                              const float *__restrict__ bval, F &&f) {
    const int jl = __builtin_amdgcn_readfirstlane(wave_find(pre, cn, (int32_t)w0));
    const int jh = __builtin_amdgcn_readfirstlane(
        wave_find(pre, cn, (int32_t)(min(w0 + 64 * RUN, W) - 1)));
    int32_t x[RUN], key[RUN];
    int j[RUN];
    float a[RUN], b[RUN];
#pragma unroll
    for (int q = 0; q < RUN; ++q) {
        x[q] = (int32_t)min(w0 + q * 64 + dev::lane_id(), W - 1);
        j[q] = jl;
    }
    // the slices' searches side by side: a step is one LDS round trip for all
    for (int d = jh > jl ? 1 << (31 - __clz(jh - jl)) : 0; d > 0; d >>= 1) {
#pragma unroll
        for (int q = 0; q < RUN; ++q) {
            const int t = min(j[q] + d, jh);
            if (pre[t] <= x[q]) j[q] = t;
        }
    }
#pragma unroll
    for (int q = 0; q < RUN; ++q) {
        const Entry t = ent[j[q]];
        const int32_t e = t.base + x[q];
        key[q] = bcol[e];
        a[q] = t.a;
        b[q] = bval ? bval[e] : 1.0f;
    }
#pragma unroll
    for (int q = 0; q < RUN; ++q)
        if (w0 + q * 64 + dev::lane_id() < W) f(key[q], a[q] * b[q]);
}

// The products of row r, load-balanced over the block: f(col, value) per
// product.  pre / ent are LDS staging of kChunk entries of A_r; RUN products per
// lane have their loads in flight together.
template <int BLOCK, int RUN, class F>
__device__ __forceinline__ void for_products(int32_t r, const int32_t *arp, const int32_t *acol,
                                             const float *aval, const int32_t *brp,
                                             const int32_t *bcol, const float *bval,
                                             int32_t *pre, Entry *ent, uint64_t *s_scan,
                                             F &&f) {
    const int32_t ab = arp[r], an = arp[r + 1] - ab;
    for (uint32_t c0 = 0; c0 < (uint32_t)an; c0 += kChunk) {
        const int32_t cn = min(kChunk, an - (int32_t)c0);
        uint32_t carry = 0;
        for (int32_t x0 = 0; x0 < cn; x0 += BLOCK) {
            const int32_t x = x0 + threadIdx.x;
            uint32_t len = 0;
            int32_t b0 = 0;
            if (x < cn) {
                const int32_t k = acol[ab + c0 + x];
                b0 = brp[k];
                len = (uint32_t)(brp[k + 1] - b0);
            }
            if (x0 > 0) __syncthreads();  // s_scan is free again
            dev::Pair32 tot;
            const uint32_t ex =
                carry + dev::block_exclusive_add_pair<BLOCK>(len, 0u, s_scan, tot).a;
            if (x < cn) {
                pre[x] = (int32_t)ex;
                ent[x] = Entry{b0 - (int32_t)ex, aval ? aval[ab + c0 + x] : 1.0f};
            }
            carry += tot.a;
        }
        if (threadIdx.x == 0) pre[cn] = (int32_t)carry;
        __syncthreads();
        const uint32_t W = carry, wave = threadIdx.x / 64;
        // a chunk that does not give every wave half a run goes out in slices
        if (W >= BLOCK * RUN / 2) {
            for (uint32_t w0 = wave * 64 * RUN; w0 < W; w0 += BLOCK * RUN)
                wave_products<RUN>(pre, ent, cn, w0, W, bcol, bval, f);
        } else if (RUN > 4 && W >= BLOCK * 2) {
            for (uint32_t w0 = wave * 64 * 4; w0 < W; w0 += BLOCK * 4)
                wave_products<4>(pre, ent, cn, w0, W, bcol, bval, f);
        } else {
            for (uint32_t w0 = wave * 64; w0 < W; w0 += BLOCK)
                wave_products<1>(pre, ent, cn, w0, W, bcol, bval, f);
        }
        __syncthreads();  // pre / ent are refilled by the next chunk
    }
}

// Moves the used slots of a table to its front, in slot order, 256 slots at
// a time (a slot's destination never lies beyond the slots already read), and
// returns their number; slots [count, next power of two) are set empty.
template <int BLOCK>
__device__ __forceinline__ uint32_t compact_table(int32_t *keys, float *vals, uint32_t tsize,
                                                  uint32_t *s_scan, uint32_t *s_n) {
    if (threadIdx.x == 0) *s_n = 0;
    __syncthreads();
    for (uint32_t s0 = 0; s0 < tsize; s0 += BLOCK) {
        const uint32_t s = s0 + threadIdx.x;
        int32_t k = kEmpty;
        float v = 0.0f;
        if (s < tsize) {
            k = keys[s];
            if (vals) v = vals[s];
        }
        const uint32_t used = k != kEmpty ? 1u : 0u;
        uint32_t tot;
        const uint32_t ex = dev::block_exclusive_add32<BLOCK>(used, s_scan, tot);  // syncs
        const uint32_t base = *s_n;
        if (used) {
            keys[base + ex] = k;
            if (vals) vals[base + ex] = v;
        }
        __syncthreads();
        if (threadIdx.x == 0) *s_n = base + tot;
        __syncthreads();
    }
    const uint32_t n = *s_n;
    uint32_t p = 1;
    while (p < n) p <<= 1;
    for (uint32_t s = n + threadIdx.x; s < p; s += BLOCK) keys[s] = kEmpty;
    __syncthreads();
    return n;
}

// Longer rows: one block per row with an open-addressing table in LDS
// (TABLE > 0, 2u <= TABLE) or in the block's region of global memory.
template <bool NUMERIC, int BLOCK, int TABLE>
__global__ __launch_bounds__(BLOCK) void k_rows_table(const int32_t *rows, const uint32_t *cnt,
                                                      const int32_t *arp, const int32_t *acol,
                                                      const float *aval, const int32_t *brp,
                                                      const int32_t *bcol, const float *bval,
                                                      int32_t *row_nnz, const int32_t *crp,
                                                      int32_t *ccol, float *cval,
                                                      const int64_t *prods, int32_t *g_keys,
                                                      float *g_vals, int64_t g_cap,
                                                      int32_t ncols) {
    constexpr bool LDS = TABLE > 0;
    __shared__ int32_t s_keys[LDS ? TABLE : 1];
    __shared__ float s_vals[(LDS && NUMERIC) ? TABLE : 1];
    __shared__ int32_t pre[kChunk + 1];
    __shared__ Entry ent[kChunk];
    __shared__ uint32_t s_scan[BLOCK / 64 + 1];
    __shared__ uint64_t s_stage[BLOCK / 64];
    __shared__ uint32_t s_count;
    int32_t *keys = LDS ? s_keys : g_keys + (int64_t)blockIdx.x * g_cap;
    float *vals = NUMERIC ? (LDS ? s_vals : g_vals + (int64_t)blockIdx.x * g_cap) : nullptr;
    const int32_t nrows = (int32_t)cnt[0];
    for (int32_t i = blockIdx.x; i < nrows; i += gridDim.x) {
        const int32_t r = rows[i];
        uint32_t tsize = 1;  // at most TABLE where the tier's rows have u <= TABLE / 2
        while (tsize < 2 * (uint64_t)min<int64_t>(prods[r], ncols)) tsize <<= 1;
        const uint32_t mask = tsize - 1;
        for (uint32_t s = threadIdx.x; s < tsize; s += BLOCK) {
            keys[s] = kEmpty;
            if (NUMERIC) vals[s] = 0.0f;
        }
        if (threadIdx.x == 0) s_count = 0;
        __syncthreads();
        uint32_t created = 0;
        for_products<BLOCK, kRun>(r, arp, acol, aval, brp, bcol, bval, pre, ent, s_stage,
                            [&](int32_t col, float v) {
                                uint32_t slot;
                                created += tab_insert(keys, mask, col, &slot) ? 1u : 0u;
                                if (NUMERIC) atomicAdd(vals + slot, v);
                            });
        if (!NUMERIC) {
            if (created) atomicAdd(&s_count, created);
            __syncthreads();
            if (threadIdx.x == 0) row_nnz[r] = (int32_t)s_count;
            __syncthreads();
            continue;
        }
        if (LDS && ncols <= 32 * kChunk) {
            // order by rank instead of sorting: a bit per column (the chunk
            // staging arrays, free once the products are done), the words'
            // popcount prefix, and each entry's rank from its own word
            uint32_t *bits = (uint32_t *)pre, *wpre = (uint32_t *)ent;
            const int32_t nw = (ncols + 31) / 32;
            __syncthreads();  // every thread is past the last chunk
            for (int32_t q = threadIdx.x; q < nw; q += BLOCK) bits[q] = 0;
            __syncthreads();
            for (uint32_t t = threadIdx.x; t < tsize; t += BLOCK) {
                const int32_t k = keys[t];
                if (k != kEmpty) atomicOr(bits + (k >> 5), 1u << (k & 31));
            }
            __syncthreads();
            uint32_t carry = 0;
            for (int32_t q0 = 0; q0 < nw; q0 += BLOCK) {
                const int32_t q = q0 + threadIdx.x;
                uint32_t tot;
                const uint32_t ex = dev::block_exclusive_add32<BLOCK>(
                    q < nw ? (uint32_t)__popc(bits[q]) : 0u, s_scan, tot);
                if (q < nw) wpre[q] = carry + ex;
                carry += tot;
            }
            __syncthreads();
            const int32_t c0 = crp[r];
            for (uint32_t t = threadIdx.x; t < tsize; t += BLOCK) {
                const int32_t k = keys[t];
                if (k == kEmpty) continue;
                const uint32_t below = bits[k >> 5] & ((1u << (k & 31)) - 1u);
                const int32_t pos = (int32_t)(wpre[k >> 5] + (uint32_t)__popc(below));
                ccol[c0 + pos] = k;
                cval[c0 + pos] = vals[t];
            }
            __syncthreads();
            continue;
        }
        const uint32_t nz = compact_table<BLOCK>(keys, vals, tsize, s_scan, &s_count);
        uint32_t p = 1;
        while (p < nz) p <<= 1;
        bitonic(keys, vals, p, threadIdx.x, BLOCK, [] { __syncthreads(); });
        const int32_t c0 = crp[r];
        for (uint32_t s = threadIdx.x; s < nz; s += BLOCK) {
            ccol[c0 + s] = keys[s];
            cval[c0 + s] = vals[s];
        }
        __syncthreads();
    }
}

// Rows of matrices with at most DN columns: a dense LDS accumulator, one value
// and one bit per column; the row comes out in column order, 64 columns per
// wave and step, and leaves its values zero for the next row.  The symbolic
// pass (DN = 0) keeps only the bits.  Rows are taken by ticket, those of more
// than kHeavy products first.  Bound by the LDS atomics.  Values are summed in
// 64 bits where they fit (DN <= 16384; more columns keep float sums, R-MAT with
// 32768 vertices at edge factor 8: 976 us, symbolic 159): beside being exact, an
// LDS add of a double runs at the rate of the integer ones, 15-24 cycles per wave in a loop
// of its own against 192 for ds_add_f32, which takes its lanes one by one.
// DN and BLOCK are the smallest that hold the columns, so that a CU holds 16
// to 32 waves (a 128 KB accumulator leaves room for one block).  R-MAT-14
// squared, 156M products: 2037 -> 517 us (542 with half the loads in flight),
// symbolic 465 -> 200 (a block of 256 for its longest rows, 340,000 products,
// took 480).
template <int DN, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_rows_dense(
    const int32_t *heavy, const int32_t *rest, const uint32_t *ctl, uint32_t *ticket,
    int32_t ncols, const int32_t *__restrict__ arp, const int32_t *__restrict__ acol,
    const float *__restrict__ aval, const int32_t *__restrict__ brp,
    const int32_t *__restrict__ bcol, const float *__restrict__ bval, int32_t *row_nnz,
    const int32_t *crp, int32_t *ccol, float *cval) {
    constexpr bool NUMERIC = DN > 0;
    using Acc = std::conditional_t<(DN > kDenseN / 2), float, double>;
    // where 16 waves fill the CU's LDS, each keeps twice the loads in flight
    constexpr int RUN = DN > kDenseN / 4 ? 2 * kRun : kRun;
    constexpr int NWORD = (NUMERIC ? DN : kDenseN) / 32;
    static_assert(NWORD <= kChunk, "the words' places share the chunk staging");
    __shared__ Acc s_val[NUMERIC ? DN : 1];
    __shared__ uint32_t s_bits[NWORD];
    __shared__ int32_t pre[kChunk + 1];
    __shared__ Entry ent[kChunk];
    __shared__ uint64_t s_scan[BLOCK / 64];
    __shared__ uint32_t s_row;
    const int32_t nw = (ncols + 31) / 32;
    const uint32_t nheavy = ctl[3], nrows = nheavy + ctl[2];
    for (int32_t q = threadIdx.x; q < nw; q += BLOCK) s_bits[q] = 0;
    if (NUMERIC)
        for (int32_t q = threadIdx.x; q < ncols; q += BLOCK) s_val[q] = Acc(0);
    for (;;) {
        if (threadIdx.x == 0) s_row = dev::atomic_add_dev(ticket, 1u);
        __syncthreads();
        const uint32_t i = s_row;
        if (i >= nrows) return;
        const int32_t r = i < nheavy ? heavy[i] : rest[i - nheavy];
        for_products<BLOCK, RUN>(r, arp, acol, aval, brp, bcol, bval, pre, ent, s_scan,
                            [&](int32_t col, float v) {
                                // a set bit needs no atomic (a stale read only costs one)
                                const uint32_t bit = 1u << (col & 31);
                                if (!(s_bits[col >> 5] & bit)) atomicOr(s_bits + (col >> 5), bit);
                                if (NUMERIC) atomicAdd(s_val + col, Acc(v));
                            });
        // each word's first place in the row
        uint32_t carry = 0;
        for (int32_t q0 = 0; q0 < nw; q0 += BLOCK) {
            const int32_t q = q0 + threadIdx.x;
            if (q0 > 0) __syncthreads();  // s_scan is free again
            dev::Pair32 tot;
            const uint32_t ex = dev::block_exclusive_add_pair<BLOCK>(
                                    q < nw ? (uint32_t)__popc(s_bits[q]) : 0u, 0u, s_scan, tot)
                                    .a;
            if (NUMERIC && q < nw) pre[q] = (int32_t)(carry + ex);
            carry += tot.a;
        }
        if (!NUMERIC && threadIdx.x == 0) row_nnz[r] = (int32_t)carry;
        if (NUMERIC) {
            __syncthreads();
            const int32_t c0 = crp[r];
            for (int32_t col = threadIdx.x; col < ncols; col += BLOCK) {
                const uint32_t bits = s_bits[col >> 5], bit = 1u << (col & 31);
                if (!(bits & bit)) continue;
                const int32_t at = c0 + pre[col >> 5] + __popc(bits & (bit - 1u));
                ccol[at] = col;
                cval[at] = (float)s_val[col];
                s_val[col] = Acc(0);
            }
            __syncthreads();
        }
        // (the next row's first product lies behind two barriers)
        for (int32_t q = threadIdx.x; q < nw; q += BLOCK) s_bits[q] = 0;
    }
}

}  // namespace

// the dense accumulator takes every row above the smallest (see spgemm_run)
static bool spgemm_small_dense(Ctx *c, int32_t n) {
    return n <= kDenseN / 2 && opt(c, "spgemm_dense", 1) != 0;
}

bool spgemm_uses_bounds(Ctx *c, int32_t n) { return !spgemm_small_dense(c, n); }

Graph *spgemm_run(Ctx *c, const Graph *a, const Graph *b) {
    const int32_t m = a->m;
    const int grid = fill_grid(c, kBlock, 4);
    apspie_graph *C = new apspie_graph();
    C->owner = c;
    C->device = c->device;
    C->m = m;
    C->n = b->n;
    C->owns = true;
    try {
        C->rowptr = (int32_t *)graph_alloc(c, sizeof(int32_t) * (m + 1));
        int64_t *prods = (int64_t *)scratch(c, "sg_ub", sizeof(int64_t) * std::max(m, 1));
        int32_t *row_nnz = (int32_t *)scratch(c, "sg_rownnz", sizeof(int32_t) * (m + 1));
        int32_t *lists = (int32_t *)scratch(c, "sg_lists", sizeof(int32_t) * 4 * (size_t)std::max(m, 1));
        uint32_t *ctl = (uint32_t *)scratch(c, "sg_ctl", 64);
        fill_i32(c, (int32_t *)ctl, 0, 16);
        // tier bounds (tunable below the tables' capacity): the wave tier's
        // table holds rows of up to kWaveUb products, the block tier's up to
        // kBlockUb; longer rows use the dense accumulator (B with at most
        // kDenseN columns, unless switched off) or global-memory tables
        const bool dense_ok = b->n <= kDenseN && opt(c, "spgemm_dense", 1) != 0;
        // up to 16,384 columns the dense accumulator (128 KB and less, no probe
        // chains, nothing to sort) takes every row above kDenseFrom products:
        // R-MAT-12 in the block tier's tables 415 us + 152 symbolic, here 82 + 69;
        // the wave tier took 32 us for its rows of up to 256 products and takes
        // 9 for those of up to 64
        const bool small_dense = spgemm_small_dense(c, b->n);
        const int32_t wave_ub = (int32_t)std::min<int64_t>(
            std::max<int64_t>(opt(c, "spgemm_wave_ub", kWaveUb), 1),
            small_dense ? kDenseFrom : kWaveUb);
        const int32_t block_ub =
            small_dense ? wave_ub
                        : (int32_t)std::min<int64_t>(
                              std::max<int64_t>(opt(c, "spgemm_block_ub", kBlockUb), wave_ub),
                              kBlockUb);
        if (m > 0) {
            k_row_bound<<<(int)std::min<int64_t>(ceil_div(m, kBlock / 16), 2 * grid), kBlock, 0,
                          c->stream>>>(a->rowptr, a->col, b->rowptr, m, prods);
            k_bin_rows<<<(int)std::min<int64_t>(grid, ceil_div(m, kBlock)), kBlock, 0,
                         c->stream>>>(prods, a->rowptr, m, b->n, wave_ub, block_ub, dense_ok,
                                      lists, ctl, row_nnz);
            APSPIE_LAUNCH_CHECK();
        }
        uint32_t *h = (uint32_t *)c->pinned;
        APSPIE_HIP(hipMemcpyAsync(h, ctl, 64, hipMemcpyDeviceToHost, c->stream));
        sync(c);
        const int64_t nwave = h[0], nblock = h[1], ndense = dense_ok ? (int64_t)h[2] + h[3] : 0,
                      nglobal = dense_ok ? 0 : h[3], ntiny = h[kCtlTiny], umax = h[kCtlMaxU];
        fill_i32(c, row_nnz + m, 0, 1);
        int64_t gcap = 1;
        while (gcap < 2 * umax) gcap <<= 1;
        // global tables: at most ~2 GiB of keys + values in flight
        const int64_t by_mem = std::max<int64_t>(1, ((int64_t)1 << 31) / (8 * gcap));
        const int gblocks = (int)std::min<int64_t>(
            std::min<int64_t>(std::max<int64_t>(nglobal, 1), c->cus), by_mem);
        int32_t *gkeys = nglobal ? (int32_t *)scratch(c, "sg_gkeys", sizeof(int32_t) * gcap * gblocks) : nullptr;
        float *gvals = nglobal ? (float *)scratch(c, "sg_gvals", sizeof(float) * gcap * gblocks) : nullptr;
        auto dense = [&](auto dn, auto block, int per_cu, int32_t *crp, int32_t *ccol, float *cval) {
            constexpr int DN = decltype(dn)::value, BLOCK = decltype(block)::value;
            k_rows_dense<DN, BLOCK>
                <<<(int)std::min<int64_t>(ndense, (int64_t)per_cu * c->cus), BLOCK, 0, c->stream>>>(
                    lists + 3 * (size_t)m, lists + 2 * (size_t)m, ctl,
                    ctl + kCtlTicket + (DN ? 1 : 0), b->n, a->rowptr, a->col, a->val, b->rowptr,
                    b->col, b->val, row_nnz, crp, ccol, cval);
        };
        auto pass = [&](auto numeric_tag, int32_t *crp, int32_t *ccol, float *cval) {
            constexpr bool NUM = decltype(numeric_tag)::value;
            using std::integral_constant;
            if (nglobal)  // longest rows first
                k_rows_table<NUM, kBig, 0><<<gblocks, kBig, 0, c->stream>>>(
                    lists + 3 * (size_t)m, ctl + 3, a->rowptr, a->col, a->val, b->rowptr, b->col,
                    b->val, row_nnz, crp, ccol, cval, prods, gkeys, gvals, gcap, b->n);
            if (ndense) {
                // blocks per CU: what their LDS (12 KB of staging beside the
                // accumulator) and 32 waves allow
                if constexpr (!NUM) {
                    if (b->n <= 8192)
                        dense(integral_constant<int, 0>{}, integral_constant<int, 512>{}, 4, crp, ccol, cval);
                    else
                        dense(integral_constant<int, 0>{}, integral_constant<int, kBig>{}, 2, crp, ccol, cval);
                }
                else if (b->n <= 4096)
                    dense(integral_constant<int, 4096>{}, integral_constant<int, 512>{}, 3, crp, ccol, cval);
                else if (b->n <= 8192)
                    dense(integral_constant<int, 8192>{}, integral_constant<int, kBig>{}, 2, crp, ccol, cval);
                else if (b->n <= 16384)
                    dense(integral_constant<int, 16384>{}, integral_constant<int, kBig>{}, 1, crp, ccol, cval);
                else
                    dense(integral_constant<int, kDenseN>{}, integral_constant<int, kBig>{}, 1, crp, ccol, cval);
            }
            if (nblock)
                k_rows_table<NUM, kBlock, kBlockTable>
                    <<<(int)std::min<int64_t>(nblock, 4 * c->cus), kBlock, 0, c->stream>>>(
                        lists + m, ctl + 1, a->rowptr, a->col, a->val, b->rowptr, b->col, b->val,
                        row_nnz, crp, ccol, cval, prods, nullptr, nullptr, 0, b->n);
            if (nwave)
                k_rows_wave<NUM><<<(int)std::min<int64_t>(ceil_div(nwave, kBlock / 64), 8 * c->cus),
                                   kBlock, 0, c->stream>>>(lists, ctl + 0, a->rowptr, a->col,
                                                           a->val, b->rowptr, b->col, b->val,
                                                           prods, b->n, row_nnz, crp, ccol, cval);
            if (ntiny)
                k_rows_tiny<NUM><<<(int)std::min<int64_t>(ceil_div(ntiny, kBlock / 16), 32 * c->cus),
                                   kBlock, 0, c->stream>>>(
                    lists + 4 * (size_t)m - 1, ctl + kCtlTiny, a->rowptr, a->col, a->val,
                    b->rowptr, b->col, b->val, row_nnz, crp, ccol, cval);
            APSPIE_LAUNCH_CHECK();
        };
        pass(std::false_type{}, nullptr, nullptr, nullptr);
        const int64_t nnz = scan_exclusive_i32(c, row_nnz, C->rowptr, m + 1);
        APSPIE_CHECK(nnz < INT32_MAX, APSPIE_ERR_OVERFLOW, "product has more than 2^31 entries");
        C->nnz = nnz;
        C->col = (int32_t *)graph_alloc(c, sizeof(int32_t) * nnz);
        C->val = (float *)graph_alloc(c, sizeof(float) * nnz);
        C->bytes = (int64_t)(sizeof(int32_t) * (m + 1) + 8 * std::max<int64_t>(nnz, 1));
        if (nnz > 0) pass(std::true_type{}, C->rowptr, C->col, C->val);
        sync(c);
        c->stats.edges_traversed = nnz;
        c->stats.iterations = 1;
    } catch (...) {
        graph_release(c, C);
        delete C;
        throw;
    }
    return C;
}

}  // namespace apspie
