// Graph ingestion on the device: COO -> CSR (optionally symmetrized,
// deduplicated and loop-free) and CSR transpose.
//
// Reference: makeSymmetric (util.cuh:571-643: mirror, qsort by (row,col),
// dedup), buildMatrix (matrix.cpp:55-111: counting sort by row that keeps the
// input order inside a row), cusparseXcoo2csr (util.cuh:456-471) and
// cusparseScsr2csc (util.cuh:473-511).  An entry travels as one 64-bit key
// (row above column) with its value beside it through the stable radix sort,
// which orders entries by (row, column) with ties in input order, so a
// duplicate keeps the value of its first occurrence; everything after the
// sort then reads in order (sorting 32-bit keys with entry numbers and
// gathering rows, columns and values by them took 10.6 ms instead of 2.6 for
// the 16.8M edges of R-MAT-20); the reference leaves self-loops in and moves values
// out of step with indices during dedup (util.cuh:606-641) -- here loops are
// dropped and values travel with their entry.
#include "common.hpp"
#include "device.hpp"
#include "primitives.hpp"

namespace apspie {

namespace {

constexpr int kBlock = 256;

// Triples as keys (row << cb) | column with their values, and with MIRROR
// each entry's mirror image after all of them.
template <bool MIRROR>
__global__ void k_pack(const int32_t *row, const int32_t *col, const float *val, int64_t nnz,
                       int32_t m, int32_t n, int cb, uint64_t *keys, float *vals, int32_t *bad) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nnz;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int32_t r = row[i], c = col[i];
        if (r < 0 || r >= m || c < 0 || c >= n) bad[0] = 1;
        keys[i] = ((uint64_t)(uint32_t)r << cb) | (uint32_t)c;
        if (MIRROR) keys[nnz + i] = ((uint64_t)(uint32_t)c << cb) | (uint32_t)r;
        if (vals) {
            const float x = val[i];
            vals[i] = x;
            if (MIRROR) vals[nnz + i] = x;
        }
    }
}

// CSR entries as keys (column << rb) | row: each thread takes kPackRun
// consecutive entries, finds the first one's row by binary search and walks on
constexpr int kPackRun = 8;
__device__ __forceinline__ int32_t entry_row(const int32_t *rowptr, int32_t m, int64_t e) {
    int32_t r = 0, hi = m;  // largest r with rowptr[r] <= e
    while (hi - r > 1) {
        const int32_t mid = (int32_t)(((int64_t)r + hi) >> 1);
        if (rowptr[mid] <= e) r = mid; else hi = mid;
    }
    return r;
}
__global__ void k_pack_transposed(const int32_t *rowptr, const int32_t *col, int32_t m,
                                  int64_t nnz, int rb, uint64_t *keys) {
    for (int64_t e0 = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) * kPackRun; e0 < nnz;
         e0 += (int64_t)gridDim.x * blockDim.x * kPackRun) {
        int32_t r = entry_row(rowptr, m, e0), end = rowptr[r + 1];
        for (int64_t e = e0; e < min(e0 + kPackRun, nnz); ++e) {
            while (end <= e) end = rowptr[++r + 1];
            keys[e] = ((uint64_t)(uint32_t)col[e] << rb) | (uint32_t)r;
        }
    }
}

// The sorted keys as CSR.  Tiles of kEmitTile entries, a wave owning 512
// consecutive ones and taking them 64 at a time; with DEDUP an entry is
// dropped if it is a self-loop or repeats the one before it.
constexpr int kEmitItems = 8;
constexpr int kEmitTile = kBlock * kEmitItems;

__device__ __forceinline__ bool emit_keep(const uint64_t *keys, int64_t e, uint64_t key, int cb) {
    if ((key >> cb) == (key & ((uint64_t(1) << cb) - 1))) return false;
    return e == 0 || keys[e - 1] != key;
}

__global__ __launch_bounds__(kBlock) void k_kept_count(const uint64_t *keys, int64_t n, int cb,
                                                       int32_t *counts) {
    __shared__ uint32_t s[kBlock / 64];
    const int w = threadIdx.x / 64;
    const int64_t base = (int64_t)blockIdx.x * kEmitTile + w * (64 * kEmitItems) + dev::lane_id();
    uint32_t c = 0;
#pragma unroll
    for (int k = 0; k < kEmitItems; ++k) {
        const int64_t e = base + k * 64;
        c += __popcll(__ballot(e < n && emit_keep(keys, e, keys[e], cb)));
    }
    if (dev::lane_id() == 0) s[w] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int q = 0; q < kBlock / 64; ++q) t += s[q];
        counts[blockIdx.x] = (int32_t)t;
    }
}

// Row starts between two consecutive entries' rows are written by the thread
// of the second one; longer gaps go to a list in pieces of kGapPiece rows
// (ctl[0] counts them), so that one thread does not write a long run of
// empty rows.
constexpr int32_t kGapShort = 64, kGapPiece = 16384;
struct Gaps {
    int32_t *lo, *hi, *val;
    uint32_t *count;
};

__device__ __forceinline__ void row_starts(int32_t *rowptr, int64_t lo, int64_t hi, int32_t v,
                                           const Gaps &g) {
    if (hi - lo < kGapShort) {
        for (int64_t r = lo; r <= hi; ++r) rowptr[r] = v;
        return;
    }
    for (int64_t r = lo; r <= hi; r += kGapPiece) {
        const uint32_t q = dev::atomic_add_dev(g.count, 1u);
        g.lo[q] = (int32_t)r;
        g.hi[q] = (int32_t)min<int64_t>(hi, r + kGapPiece - 1);
        g.val[q] = v;
    }
}

__global__ void k_fill_gaps(int32_t *rowptr, Gaps g) {
    const uint32_t n = *g.count;
    for (uint32_t q = blockIdx.x; q < n; q += gridDim.x)
        for (int64_t r = (int64_t)g.lo[q] + threadIdx.x; r <= g.hi[q]; r += blockDim.x)
            rowptr[r] = g.val[q];
}

// offsets: entries kept before each tile (null: all are kept); vals null:
// values of 1.0 where oval is given
template <bool DEDUP>
__global__ __launch_bounds__(kBlock) void k_emit(const uint64_t *keys, const float *vals,
                                                 int64_t n, int cb, int32_t m,
                                                 const int32_t *offsets, int32_t *ocol,
                                                 float *oval, int32_t *rowptr, Gaps gaps) {
    __shared__ uint32_t s_cnt[kBlock / 64];
    const int w = threadIdx.x / 64;
    const uint64_t cmask = (uint64_t(1) << cb) - 1;
    const int64_t base = (int64_t)blockIdx.x * kEmitTile + w * (64 * kEmitItems) + dev::lane_id();
    uint64_t key[kEmitItems], kept[kEmitItems];
    uint32_t c = 0;
#pragma unroll
    for (int k = 0; k < kEmitItems; ++k) {
        const int64_t e = base + k * 64;
        key[k] = e < n ? keys[e] : 0;
        kept[k] = __ballot(e < n && (!DEDUP || emit_keep(keys, e, key[k], cb)));
        c += __popcll(kept[k]);
    }
    if (dev::lane_id() == 0) s_cnt[w] = c;
    __syncthreads();
    int64_t run = offsets ? offsets[blockIdx.x] : (int64_t)blockIdx.x * kEmitTile;
    for (int q = 0; q < w; ++q) run += s_cnt[q];
#pragma unroll
    for (int k = 0; k < kEmitItems; ++k) {
        const int64_t e = base + k * 64;
        const int32_t at = (int32_t)(run + __popcll(kept[k] & dev::lanemask_lt()));
        const bool mine = (kept[k] >> dev::lane_id()) & 1u;
        if (e < n) {
            const int64_t r = (int64_t)(key[k] >> cb);
            if (mine) {
                ocol[at] = (int32_t)(key[k] & cmask);
                if (oval) oval[at] = vals ? vals[e] : 1.0f;
            }
            // rows up to this one start here if the entry before is in another
            const int64_t before = e > 0 ? (int64_t)(keys[e - 1] >> cb) : -1;
            if (r != before) row_starts(rowptr, before + 1, r, at, gaps);
            if (e == n - 1) row_starts(rowptr, r + 1, m, at + (mine ? 1 : 0), gaps);
        }
        run += __popcll(kept[k]);
    }
}

__global__ void k_iota_key(const int32_t *src, int64_t n, uint32_t *keys, uint32_t *idx) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        idx[i] = (uint32_t)i;
        keys[i] = (uint32_t)src[i];
    }
}

// row id of every CSR entry (binary search over rowptr)
__global__ void k_entry_rows(const int32_t *rowptr, int32_t m, int64_t nnz, int32_t *rows) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < nnz;
         e += (int64_t)gridDim.x * blockDim.x) {
        int32_t lo = 0, hi = m;  // largest r with rowptr[r] <= e
        while (hi - lo > 1) {
            const int32_t mid = lo + ((hi - lo) >> 1);  // lo + hi can pass 2^31
            if (rowptr[mid] <= e) lo = mid; else hi = mid;
        }
        rows[e] = lo;
    }
}

// rowptr / col / val of g (allocated, k entries) from E sorted keys
template <bool DEDUP>
void emit_csr(Ctx *c, Graph *g, const uint64_t *keys, const float *vals, int64_t E, int cb,
              const int32_t *offsets) {
    if (E == 0) {
        fill_i32(c, g->rowptr, 0, (int64_t)g->m + 1);
        return;
    }
    const int64_t pieces = (int64_t)g->m / kGapShort + g->m / kGapPiece + 4;
    int32_t *mem = (int32_t *)scratch(c, "emit_gaps", sizeof(int32_t) * (3 * pieces + 1));
    const Gaps gaps{mem + 1, mem + 1 + pieces, mem + 1 + 2 * pieces, (uint32_t *)mem};
    fill_i32(c, mem, 0, 1);
    k_emit<DEDUP><<<(unsigned)ceil_div(E, kEmitTile), kBlock, 0, c->stream>>>(
        keys, vals, E, cb, g->m, offsets, g->col, g->val, g->rowptr, gaps);
    k_fill_gaps<<<fill_grid(c, kBlock, 2), kBlock, 0, c->stream>>>(g->rowptr, gaps);
    APSPIE_LAUNCH_CHECK();
}

// ---------------------------------------------------- row-block DCSC
// Part of CSR row r when the rows are cut into blocks of ps, the last of the
// pn parts taking every row from (pn - 1) * ps on.
__device__ __forceinline__ uint32_t dcsc_part(int32_t r, int32_t ps, int32_t pn) {
    return (uint32_t)min(r / ps, pn - 1);
}

__global__ void k_dcsc_part_keys(const int32_t *rows, const uint32_t *idx, int64_t n, int32_t ps,
                                 int32_t pn, uint32_t *keys) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        keys[i] = dcsc_part(rows[idx[i]], ps, pn);
}

// Entry j of the (part, column, row) order: its row and value, and whether
// it opens a (part, column) segment.
__global__ void k_dcsc_entries(const int32_t *rows, const int32_t *col, const float *val,
                               const uint32_t *part, const uint32_t *idx, int64_t n,
                               int32_t *row_ind, float *val_out, int32_t *opens) {
    for (int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; j < n;
         j += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t e = idx[j];
        row_ind[j] = rows[e];
        if (val_out) val_out[j] = val[e];
        opens[j] = j == 0 || part[j] != part[j - 1] || col[e] != col[idx[j - 1]];
    }
}

// Segment k starts at off[k]: its column and part; off[L] = n closes the last.
__global__ void k_dcsc_segments(const int32_t *col, const uint32_t *idx, const uint32_t *part,
                                int32_t *off, int64_t L, int64_t n, int32_t *col_ind,
                                uint32_t *seg_part) {
    const int64_t gid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    for (int64_t k = gid; k < L; k += (int64_t)gridDim.x * blockDim.x) {
        const int32_t j = off[k];
        col_ind[k] = col[idx[j]];
        seg_part[k] = part[j];
    }
    if (gid == 0) off[L] = (int32_t)n;
}

// part_ptr[p] = segments in parts before p (first k with seg_part[k] >= p)
__global__ void k_dcsc_part_ptr(const uint32_t *seg_part, int64_t L, int32_t pn,
                                int32_t *part_ptr) {
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p <= pn;
         p += (int64_t)gridDim.x * blockDim.x) {
        int64_t lo = 0, hi = L;
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if ((int64_t)seg_part[mid] < p) lo = mid + 1; else hi = mid;
        }
        part_ptr[p] = (int32_t)lo;
    }
}

}  // namespace

void graph_from_coo_dev(Ctx *c, Graph *g, const int32_t *row, const int32_t *col,
                        const float *val, int64_t nnz, int symmetrize) {
    const int grid = fill_grid(c, kBlock, 8);
    const int64_t E = symmetrize ? 2 * nnz : nnz;
    const int64_t Ea = std::max<int64_t>(E, 1);
    const int cb = bits_for(std::max(g->n - 1, 1)), rb = bits_for(std::max(g->m - 1, 1));
    uint64_t *ka = (uint64_t *)scratch(c, "ing_ka", sizeof(uint64_t) * Ea);
    uint64_t *kb = (uint64_t *)scratch(c, "ing_kb", sizeof(uint64_t) * Ea);
    float *va = nullptr, *vb = nullptr;
    if (val) {
        va = (float *)scratch(c, "ing_va", sizeof(float) * Ea);
        vb = (float *)scratch(c, "ing_vb", sizeof(float) * Ea);
    }
    const int64_t ntiles = ceil_div(Ea, kEmitTile);
    // [0] entries kept, [1] an index out of range
    int64_t *ctl = (int64_t *)scratch(c, "ing_ctl", 256);
    fill_i32(c, (int32_t *)ctl, 0, 4);
    if (nnz > 0) {
        if (symmetrize)
            k_pack<true><<<grid, kBlock, 0, c->stream>>>(row, col, val, nnz, g->m, g->n, cb, ka,
                                                         va, (int32_t *)(ctl + 1));
        else
            k_pack<false><<<grid, kBlock, 0, c->stream>>>(row, col, val, nnz, g->m, g->n, cb, ka,
                                                          va, (int32_t *)(ctl + 1));
        APSPIE_LAUNCH_CHECK();
    }
    int32_t *offsets = nullptr;
    if (E > 0) {
        // symmetrized: by (row, column); else by row only, input order inside
        // a row (buildMatrix).  (Keys of an index out of range sort as any
        // others do: every digit is masked.)
        const bool in_b = radix_sort(c, ka, (uint32_t *)va, kb, (uint32_t *)vb, E,
                                     symmetrize ? 0 : cb, symmetrize ? cb + rb : rb);
        if (in_b) {
            std::swap(ka, kb);
            std::swap(va, vb);
        }
        if (symmetrize) {
            int32_t *counts = (int32_t *)scratch(c, "ing_cnt", sizeof(int32_t) * ntiles);
            offsets = (int32_t *)scratch(c, "ing_off", sizeof(int32_t) * ntiles);
            k_kept_count<<<(unsigned)ntiles, kBlock, 0, c->stream>>>(ka, E, cb, counts);
            APSPIE_LAUNCH_CHECK();
            scan_exclusive_i32_async(c, counts, offsets, ntiles, ctl);
        }
    }
    int64_t h[2] = {0, 0};
    APSPIE_HIP(hipMemcpyAsync(h, ctl, sizeof h, hipMemcpyDeviceToHost, c->stream));
    sync(c);
    APSPIE_CHECK(h[1] == 0, APSPIE_ERR_INVALID, "COO index out of range");
    const int64_t k = symmetrize ? h[0] : E;
    g->nnz = k;
    g->rowptr = (int32_t *)graph_alloc(c, sizeof(int32_t) * (g->m + 1));
    g->col = (int32_t *)graph_alloc(c, sizeof(int32_t) * k);
    g->val = (float *)graph_alloc(c, sizeof(float) * k);
    g->bytes = (int64_t)(sizeof(int32_t) * (g->m + 1) + 8 * std::max<int64_t>(k, 1));
    if (symmetrize) emit_csr<true>(c, g, ka, va, E, cb, offsets);
    else emit_csr<false>(c, g, ka, va, E, cb, nullptr);
}

__global__ void k_neq(const int32_t *a, const int32_t *b, int64_t n, int32_t *flag) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        if (a[i] != b[i]) flag[0] = 1;
}

// Whether every entry of a symmetric CSR with sorted rows has its mirror
// image's value: kPackRun consecutive entries per thread, the mirror image by
// binary search in its row.
__global__ void k_check_mirror_values(const int32_t *rowptr, const int32_t *col,
                                      const float *val, int32_t m, int64_t nnz, int32_t *flag) {
    for (int64_t e0 = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) * kPackRun; e0 < nnz;
         e0 += (int64_t)gridDim.x * blockDim.x * kPackRun) {
        int32_t r = entry_row(rowptr, m, e0), end = rowptr[r + 1];
        for (int64_t e = e0; e < min(e0 + kPackRun, nnz); ++e) {
            while (end <= e) end = rowptr[++r + 1];
            const int32_t v = col[e];
            int32_t lo = rowptr[v], hi = rowptr[v + 1];  // first entry of row v not below r
            while (lo < hi) {
                const int32_t mid = lo + ((hi - lo) >> 1);  // lo + hi can pass 2^31
                if (col[mid] < r) lo = mid + 1; else hi = mid;
            }
            if (lo >= rowptr[v + 1] || col[lo] != r ||
                __float_as_int(val[lo]) != __float_as_int(val[e]))
                flag[0] = 1;
        }
    }
}

// Structure (and, for a weighted graph, values) compared with the transpose,
// once per graph.  The transpose's rows come out sorted, so with equal
// structure the values line up position by position.
static void check_symmetry(Ctx *c, Graph *g) {
    if (g->symmetric >= 0) return;
    if (g->m != g->n) {
        g->symmetric = 0;
        g->sym_weights = 0;
        return;
    }
    Graph t;  // a temporary in the context's scratch
    graph_transpose_dev(c, g, &t, "sym_t");
    int32_t *flag = (int32_t *)scratch(c, "sym_flag", 256);
    fill_i32(c, flag, 0, 2);
    const int grid = fill_grid(c, kBlock, 4);
    k_neq<<<grid, kBlock, 0, c->stream>>>(g->rowptr, t.rowptr, g->m + 1, flag);
    k_neq<<<grid, kBlock, 0, c->stream>>>(g->col, t.col, g->nnz, flag);
    if (g->val && t.val)
        k_neq<<<grid, kBlock, 0, c->stream>>>((const int32_t *)g->val, (const int32_t *)t.val,
                                               g->nnz, flag + 1);
    APSPIE_LAUNCH_CHECK();
    int32_t h[2] = {1, 1};
    APSPIE_HIP(hipMemcpyAsync(h, flag, 8, hipMemcpyDeviceToHost, c->stream));
    sync(c);
    g->symmetric = h[0] == 0 ? 1 : 0;
    g->sym_weights = (g->symmetric == 1 && g->val && h[1] == 0) ? 1 : 0;
}

// A graph built symmetrized is known to be symmetric (and its rows sorted),
// but not in its values: an edge listed both ways round keeps each one's own.
// Checked in place, with no scratch but a flag: the callers may have none left.
static void check_mirror_values(Ctx *c, Graph *g) {
    if (g->symmetric != 1 || g->sym_weights >= 0) return;
    int32_t *flag = (int32_t *)scratch(c, "sym_flag", 256);
    fill_i32(c, flag, 0, 1);
    if (g->val && g->nnz > 0) {
        k_check_mirror_values<<<fill_grid(c, kBlock, 8), kBlock, 0, c->stream>>>(
            g->rowptr, g->col, g->val, g->m, g->nnz, flag);
        APSPIE_LAUNCH_CHECK();
    }
    int32_t h = 1;
    APSPIE_HIP(hipMemcpyAsync(&h, flag, 4, hipMemcpyDeviceToHost, c->stream));
    sync(c);
    g->sym_weights = g->val && h == 0 ? 1 : 0;
}

__global__ void k_iso_bits(const int32_t *rowptr, int32_t m, uint32_t *bits) {
    const int64_t words = ((int64_t)m + 31) / 32;
    for (int64_t wi = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; wi < words;
         wi += (int64_t)gridDim.x * blockDim.x) {
        uint32_t x = 0;
        int32_t prev = rowptr[wi * 32];
        for (int b = 0; b < 32 && wi * 32 + b < m; ++b) {
            const int32_t next = rowptr[wi * 32 + b + 1];
            if (next == prev) x |= 1u << b;
            prev = next;
        }
        bits[wi] = x;
    }
}

__global__ void k_max_degree(const int32_t *rowptr, int32_t m, int32_t *out) {
    int32_t best = 0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m;
         i += (int64_t)gridDim.x * blockDim.x)
        best = max(best, rowptr[i + 1] - rowptr[i]);
    for (int off = 32; off > 0; off >>= 1) best = max(best, __shfl_xor(best, off, 64));
    if (dev::lane_id() == 0 && best > 0) atomicMax(out, best);
}

// Floats as unsigned keys that order like the floats (negative ones reversed).
__device__ __forceinline__ uint32_t f_order(float f) {
    const uint32_t b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

// One pair of atomics per block: one per wave on the same two words took 80 us
// whatever the size.
__global__ __launch_bounds__(kBlock) void k_weight_range(const float *w, int64_t n,
                                                         uint32_t *out) {
    constexpr int U = 8;
    __shared__ uint32_t s_lo[kBlock / 64], s_hi[kBlock / 64];
    uint32_t lo = 0xffffffffu, hi = 0;
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i0 = blockIdx.x * (int64_t)kBlock + threadIdx.x; i0 < n; i0 += stride * U) {
        float x[U];
#pragma unroll
        for (int k = 0; k < U; ++k) x[k] = w[min(i0 + k * stride, n - 1)];
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const uint32_t q = f_order(x[k]);
            lo = min(lo, q);
            hi = max(hi, q);
        }
    }
    lo = dev::wave_min_u32(lo);
    hi = dev::wave_max_u32(hi);
    if (dev::lane_id() == 0) {
        s_lo[threadIdx.x / 64] = lo;
        s_hi[threadIdx.x / 64] = hi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int q = 1; q < kBlock / 64; ++q) {
            lo = min(lo, s_lo[q]);
            hi = max(hi, s_hi[q]);
        }
        atomicMin(out, lo);
        atomicMax(out + 1, hi);
    }
}

bool graph_weight_range(Ctx *c, Graph *g, float *lo, float *hi) {
    if (!g->val || g->nnz == 0) return false;
    std::lock_guard<std::mutex> lock(g->derived_mu);
    if (g->w_range < 0) {
        uint32_t *d = (uint32_t *)scratch(c, "w_range", 256);
        fill_i32(c, (int32_t *)d, -1, 1);
        fill_i32(c, (int32_t *)d + 1, 0, 1);
        k_weight_range<<<(int)std::min<int64_t>(ceil_div(g->nnz, kBlock), 4 * c->cus), kBlock, 0,
                         c->stream>>>(g->val, g->nnz, d);
        APSPIE_LAUNCH_CHECK();
        uint32_t h[2];
        APSPIE_HIP(hipMemcpyAsync(h, d, 8, hipMemcpyDeviceToHost, c->stream));
        sync(c);
        auto back = [](uint32_t k) {
            const uint32_t b = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
            return __builtin_bit_cast(float, b);
        };
        g->w_lo = back(h[0]);
        g->w_hi = back(h[1]);
        g->w_range = 1;
    }
    *lo = g->w_lo;
    *hi = g->w_hi;
    return true;
}

// Longest row, computed once per graph.
int32_t graph_max_degree(Ctx *c, Graph *g) {
    std::lock_guard<std::mutex> lock(g->derived_mu);
    if (g->max_deg >= 0) return g->max_deg;
    int32_t *d = (int32_t *)scratch(c, "max_deg", 256);
    fill_i32(c, d, 0, 1);
    if (g->m > 0) {
        k_max_degree<<<(int)std::min<int64_t>(ceil_div(g->m, kBlock), 4 * c->cus), kBlock, 0,
                       c->stream>>>(g->rowptr, g->m, d);
        APSPIE_LAUNCH_CHECK();
    }
    int32_t h = 0;
    APSPIE_HIP(hipMemcpyAsync(&h, d, 4, hipMemcpyDeviceToHost, c->stream));
    sync(c);
    g->max_deg = h;
    return h;
}

// Bitmap of the vertices without entries, built once per graph.
const uint32_t *graph_iso_bits(Ctx *c, Graph *g) {
    std::lock_guard<std::mutex> lock(g->derived_mu);
    if (g->iso_bits) return g->iso_bits;
    const int64_t words = ((int64_t)g->m + 31) / 32;
    uint32_t *bits = nullptr;
    // owned by the graph (freed with it), like its other derived arrays
    APSPIE_HIP(device_malloc(c, (void **)&bits, sizeof(uint32_t) * std::max<int64_t>(words, 1)));
    if (words > 0) {
        k_iso_bits<<<(int)std::min<int64_t>(ceil_div(words, kBlock), 4 * c->cus), kBlock, 0,
                     c->stream>>>(g->rowptr, g->m, bits);
        APSPIE_LAUNCH_CHECK();
    }
    sync(c);
    g->iso_bits = bits;
    return bits;
}

// ------------------------------------------------- connected components
// Lock-free union-find over the edges of a symmetric CSR: every root hooks
// under a smaller root with one compare-and-swap on its parent pointer, so a
// tree's root is always the smallest id in it and the final label of a
// vertex is the smallest vertex id of its component.  Parents only ever move
// to smaller ids of the same set, so any value a parent pointer ever held is
// an ancestor: a find may halve its path, and a stale read only costs a
// retry.  Every write to the parent array while unions run is an atomic
// read-modify-write (the hook, the halving swap, the final label exchange):
// the workgroups of different XCDs write neighbouring words of one line.
__device__ __forceinline__ int32_t cc_parent(const int32_t *p, int32_t x) {
    return __hip_atomic_load(p + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int32_t cc_find(int32_t *p, int32_t x) {
    int32_t px = cc_parent(p, x);
    while (px != x) {
        const int32_t gp = cc_parent(p, px);
        if (gp != px) {  // halve: x's parent becomes its grandparent, if still px
            int32_t expected = px;
            __hip_atomic_compare_exchange_strong(p + x, &expected, gp, __ATOMIC_RELAXED,
                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        x = gp;
        px = cc_parent(p, x);
    }
    return x;
}

__device__ __forceinline__ void cc_unite(int32_t *p, int32_t u, int32_t v) {
    u = cc_find(p, u);
    v = cc_find(p, v);
    while (u != v) {
        if (u < v) {
            const int32_t t = u;
            u = v;
            v = t;
        }
        // hook the larger root u under v; a failed swap means u got a parent
        int32_t expected = u;
        if (__hip_atomic_compare_exchange_strong(p + u, &expected, v, __ATOMIC_RELAXED,
                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            return;
        u = cc_find(p, expected);
        v = cc_find(p, v);
    }
}

__global__ void k_cc_init(int32_t m, int32_t *p) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = (int32_t)i;
}

constexpr int32_t kCcShort = 32;

// rows of at most kCcShort entries: one thread per row; each undirected edge
// is united from its larger end only
__global__ void k_cc_short(const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col,
                           int32_t m, int32_t *p) {
    for (int64_t u = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; u < m;
         u += (int64_t)gridDim.x * blockDim.x) {
        const int32_t rs = rowptr[u], re = rowptr[u + 1];
        if (re - rs > kCcShort) continue;
        for (int32_t e = rs; e < re; ++e) {
            const int32_t v = col[e];
            if (v < u) cc_unite(p, (int32_t)u, v);
        }
    }
}

// longer rows: one wave per row, lanes striding it
__global__ void k_cc_long(const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col,
                          int32_t m, int32_t *p) {
    const int lane = dev::lane_id();
    const int64_t wave = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / 64;
    const int64_t nwaves = (int64_t)gridDim.x * blockDim.x / 64;
    for (int64_t u = wave; u < m; u += nwaves) {
        const int32_t rs = rowptr[u], re = rowptr[u + 1];
        if (re - rs <= kCcShort) continue;
        for (int32_t e = rs + lane; e < re; e += 64) {
            const int32_t v = col[e];
            if (v < u) cc_unite(p, (int32_t)u, v);
        }
    }
}

__global__ void k_cc_label(int32_t m, int32_t *p) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < m;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int32_t r = cc_find(p, (int32_t)i);
        __hip_atomic_exchange(p + i, r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

void components_into(Ctx *c, const Graph *g, int32_t *label) {
    if (g->m == 0) return;
    const int grid = fill_grid(c, kBlock, 8);
    k_cc_init<<<grid, kBlock, 0, c->stream>>>(g->m, label);
    k_cc_short<<<grid, kBlock, 0, c->stream>>>(g->rowptr, g->col, g->m, label);
    k_cc_long<<<grid, kBlock, 0, c->stream>>>(g->rowptr, g->col, g->m, label);
    k_cc_label<<<grid, kBlock, 0, c->stream>>>(g->m, label);
    APSPIE_LAUNCH_CHECK();
}

const int32_t *graph_components(Ctx *c, Graph *g) {
    std::lock_guard<std::mutex> lock(g->derived_mu);
    if (g->comp) return g->comp;
    int32_t *label = nullptr;
    // owned by the graph (freed with it), like its other derived arrays
    APSPIE_HIP(device_malloc(c, (void **)&label, sizeof(int32_t) * std::max<int64_t>(g->m, 1)));
    components_into(c, g, label);
    sync(c);
    g->comp = label;
    return label;
}

int graph_symmetry_known(Graph *g) {
    std::lock_guard<std::mutex> lock(g->derived_mu);
    return g->symmetric;
}

const uint32_t *graph_iso_bits_cached(Graph *g) {
    std::lock_guard<std::mutex> lock(g->derived_mu);
    return g->iso_bits;
}

void iso_bits_into(Ctx *c, const Graph *g, uint32_t *bits) {
    const int64_t words = ((int64_t)g->m + 31) / 32;
    if (words == 0) return;
    k_iso_bits<<<(int)std::min<int64_t>(ceil_div(words, kBlock), 4 * c->cus), kBlock, 0,
                 c->stream>>>(g->rowptr, g->m, bits);
    APSPIE_LAUNCH_CHECK();
}

bool graph_is_symmetric(Ctx *c, Graph *g) {
    std::lock_guard<std::mutex> lock(g->derived_mu);
    check_symmetry(c, g);
    return g->symmetric == 1;
}

bool graph_is_symmetric_weighted(Ctx *c, Graph *g) {
    std::lock_guard<std::mutex> lock(g->derived_mu);
    check_symmetry(c, g);
    check_mirror_values(c, g);
    return g->sym_weights == 1;
}

void graph_transpose_dev(Ctx *c, const Graph *g, Graph *t, const char *in_scratch) {
    const int grid = fill_grid(c, kBlock, 4);
    const int64_t E = g->nnz, Ea = std::max<int64_t>(E, 1);
    t->owner = c;
    t->device = c->device;
    t->m = g->n;
    t->n = g->m;
    t->nnz = E;
    t->owns = !in_scratch;
    // keys (new row = old column, new column = old row), sorted by the old
    // column alone: stable, so the old rows stay ascending
    const int rb = bits_for(std::max(g->m - 1, 1));
    uint64_t *ka = (uint64_t *)scratch(c, "tr_ka", sizeof(uint64_t) * Ea);
    uint64_t *kb = (uint64_t *)scratch(c, "tr_kb", sizeof(uint64_t) * Ea);
    float *va = nullptr, *vb = nullptr;
    if (g->val) {
        va = (float *)scratch(c, "tr_va", sizeof(float) * Ea);
        vb = (float *)scratch(c, "tr_vb", sizeof(float) * Ea);
    }
    if (E > 0) {
        k_pack_transposed<<<grid, kBlock, 0, c->stream>>>(g->rowptr, g->col, g->m, E, rb, ka);
        APSPIE_LAUNCH_CHECK();
        if (g->val)
            APSPIE_HIP(hipMemcpyAsync(va, g->val, sizeof(float) * E, hipMemcpyDeviceToDevice,
                                      c->stream));
        if (radix_sort(c, ka, (uint32_t *)va, kb, (uint32_t *)vb, E, rb, bits_for(std::max(g->n - 1, 1)))) {
            std::swap(ka, kb);
            std::swap(va, vb);
        }
    }
    if (in_scratch) {
        const std::string p(in_scratch);
        t->rowptr = (int32_t *)scratch(c, p + "_rowptr", sizeof(int32_t) * (t->m + 1));
        t->col = (int32_t *)scratch(c, p + "_col", sizeof(int32_t) * Ea);
        t->val = g->val ? (float *)scratch(c, p + "_val", sizeof(float) * Ea) : nullptr;
    } else {
        t->rowptr = (int32_t *)graph_alloc(c, sizeof(int32_t) * (t->m + 1));
        t->col = (int32_t *)graph_alloc(c, sizeof(int32_t) * E);
        t->val = g->val ? (float *)graph_alloc(c, sizeof(float) * E) : nullptr;
    }
    t->bytes = (int64_t)(sizeof(int32_t) * (t->m + 1) + (g->val ? 8 : 4) * Ea);
    emit_csr<false>(c, t, ka, va, E, rb, nullptr);
}


// Row-block DCSC (csr_to_dcsc, matrix.cpp:286-468): two stable radix passes
// order the entries by (part, column) with rows ascending inside, the
// segment openings are compacted into the column offsets, and each part's
// first segment is found by binary search.  Outputs are device pointers;
// returns the number of (part, column) segments.
int64_t graph_to_dcsc_dev(Ctx *c, const Graph *g, int32_t ps, int32_t pn, int32_t *part_ptr,
                          int32_t *col_ind, int32_t *col_off, int32_t *row_ind, float *val) {
    const int grid = fill_grid(c, kBlock, 4);
    const int64_t E = g->nnz, Ea = std::max<int64_t>(E, 1);
    int64_t L = 0;
    uint32_t *seg_part = (uint32_t *)scratch(c, "dc_sp", sizeof(uint32_t) * Ea);
    if (E > 0) {
        int32_t *rows = (int32_t *)scratch(c, "dc_rows", sizeof(int32_t) * Ea);
        uint32_t *keys = (uint32_t *)scratch(c, "dc_k", sizeof(uint32_t) * Ea);
        uint32_t *idx = (uint32_t *)scratch(c, "dc_i", sizeof(uint32_t) * Ea);
        int32_t *opens = (int32_t *)scratch(c, "dc_open", sizeof(int32_t) * Ea);
        k_entry_rows<<<grid, kBlock, 0, c->stream>>>(g->rowptr, g->m, E, rows);
        k_iota_key<<<grid, kBlock, 0, c->stream>>>(g->col, E, keys, idx);
        APSPIE_LAUNCH_CHECK();
        radix_sort_pairs(c, keys, idx, E, bits_for(g->n));  // by column, rows kept ascending
        k_dcsc_part_keys<<<grid, kBlock, 0, c->stream>>>(rows, idx, E, ps, pn, keys);
        APSPIE_LAUNCH_CHECK();
        radix_sort_pairs(c, keys, idx, E, bits_for(pn - 1));  // by part, stable
        k_dcsc_entries<<<grid, kBlock, 0, c->stream>>>(rows, g->col, g->val, keys, idx, E,
                                                       row_ind, g->val ? val : nullptr, opens);
        APSPIE_LAUNCH_CHECK();
        L = compact_flags(c, opens, E, col_off);
        k_dcsc_segments<<<grid, kBlock, 0, c->stream>>>(g->col, idx, keys, col_off, L, E,
                                                        col_ind, seg_part);
    } else {
        k_dcsc_segments<<<1, 64, 0, c->stream>>>(g->col, nullptr, nullptr, col_off, 0, 0,
                                                 col_ind, seg_part);
    }
    APSPIE_LAUNCH_CHECK();
    k_dcsc_part_ptr<<<std::max(1, std::min(grid, (pn + kBlock) / kBlock)), kBlock, 0,
                      c->stream>>>(seg_part, L, pn, part_ptr);
    APSPIE_LAUNCH_CHECK();
    return L;
}

}  // namespace apspie
