// SpMV kernels of the MLEM iteration for CDNA4 (gfx950, wave64).
//
//  * csr_vector_kernel<G, EPI>: a group of G work-items per row
//    (calcFwProj_csr_vector / calcBwProj_csr_vector, kernel.cu:118-153,
//    297-336).  Consecutive 4-byte non-temporal loads of col/val, eight
//    rounds in flight, fixed-order xor shuffle reduction, plain store
//    through the epilogue.  csr_long_rows_kernel<EPI>: the same for long rows.
//  * merge_*: block-level merge-path SpMV (calcFwProj_merge_based /
//    calcBwProj_merge_based, kernel.cu:52-105,190-286).  The merge path of
//    (row ends, nonzeros) is cut into tiles of 256*S items; each workgroup
//    stages its tile's products and row ends in LDS, every work-item walks S
//    items, a segmented scan over the workgroup joins rows split between
//    work-items, and rows split between tiles are finished by a fix-up kernel
//    that adds the tile carries in tile order.  No float atomics: results are
//    bitwise reproducible.
//  * scatter_kernel<G>, scatter_window_kernel: BP without a transpose
//    (calcBwProj_none_trans, kernel.cu:165-177,347-370), float atomics, one
//    per entry or summed in LDS first.
//  * elementwise ratio / update / fill, FP64 column sums, FP64 log-likelihood.
#include <algorithm>

#include "launch.hpp"

namespace mlem {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Streamed matrix data is read once per pass: non-temporal loads keep it from
// evicting the gathered image / ratio vector from L2.
template <typename T>
__device__ __forceinline__ T ldnt(const T *p) {
    return __builtin_nontemporal_load(p);
}

// The epilogue of row r with row sum y: calcCorrel (kernel.cu:16-18), g / y
// where y != 0, else y stays; calcUpdate (kernel.cu:33-37), (f * y) / norm,
// or f * y where norm == 0; or the plain sum.  epi_load reads the row's
// inputs (RATIO: the count; UPDATE: the image value and the sensitivity) and
// emit_with forms the result, so that a kernel can issue those reads before
// its row sum and their memory round trip overlaps the sum's.
struct EpiIn {
    float a, b;
};

template <int EPI>
__device__ __forceinline__ EpiIn epi_load(uint32_t r, const EpiArgs &ea) {
    if constexpr (EPI == EPI_RATIO) return {(float)ea.g[r], 0.0f};
    else if constexpr (EPI == EPI_UPDATE) return {ea.f[r], ea.norm[r]};
    else return {0.0f, 0.0f};
}

template <int EPI>
__device__ __forceinline__ void emit_with(uint32_t r, float y, const EpiIn &in, const EpiArgs &ea) {
    if constexpr (EPI == EPI_PLAIN) {
        ea.out[r] = y;
    } else if constexpr (EPI == EPI_RATIO) {
        ea.out[r] = (y != 0.0f) ? in.a / y : y;
    } else {
        const float v = in.a * y;
        ea.f[r] = (in.b == 0.0f) ? v : v / in.b;
    }
}

template <int EPI>
__device__ __forceinline__ void emit(uint32_t r, float y, const EpiArgs &ea) {
    emit_with<EPI>(r, y, epi_load<EPI>(r, ea), ea);
}

// ---------------------------------------------------------------------------
// CSR-vector
// ---------------------------------------------------------------------------
template <int G>
__device__ __forceinline__ float group_sum(float v) {
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

template <int G>
__device__ __forceinline__ double group_sum_f64(double v) {
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// Row sum of val[k] * x[col[k]] over [b, e) split over the G work-items of a
// group (this work-item is `lane`); per-lane partials, not yet reduced.
// Consecutive work-items take consecutive entries (4-byte loads), so one
// gather instruction reads neighbouring columns, which share cache lines.
// Rounds of U = 8 entries per work-item are loaded before any is used; the
// last (partial) round is issued the same way with the entries past the row
// end masked off, so a short row costs one load latency, not one per entry.
template <int G>
__device__ __forceinline__ float row_partial(const uint32_t *__restrict__ col, const float *__restrict__ val,
                                             const float *__restrict__ x, uint64_t b, uint64_t e, uint32_t lane) {
    constexpr int U = 8;
    float acc = 0.0f;
    uint64_t k = b + lane;
    for (; k + (uint64_t)(U - 1) * G < e; k += (uint64_t)U * G) {
        uint32_t c[U];
        float v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            c[u] = ldnt(col + k + (uint64_t)u * G);
            v[u] = ldnt(val + k + (uint64_t)u * G);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) acc += v[u] * x[c[u]];
    }
    if (k < e) {  // fewer than U rounds left
        uint32_t c[U];
        float v[U];
        bool in[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            in[u] = k + (uint64_t)u * G < e;
            c[u] = in[u] ? ldnt(col + k + (uint64_t)u * G) : 0u;
            v[u] = in[u] ? ldnt(val + k + (uint64_t)u * G) : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (in[u]) acc += v[u] * x[c[u]];
    }
    return acc;
}

template <int G, int EPI>
__global__ __launch_bounds__(kWG) void csr_vector_kernel(const uint64_t *__restrict__ rowptr,
                                                         const uint32_t *__restrict__ col,
                                                         const float *__restrict__ val, const float *__restrict__ x,
                                                         uint32_t rows, EpiArgs ea) {
    const uint32_t row = blockIdx.x * (uint32_t)(kWG / G) + threadIdx.x / G;
    const uint32_t lane = threadIdx.x % G;
    if (row >= rows) return;  // whole groups leave together
    const EpiIn in = epi_load<EPI>(row, ea);  // every work-item of the group: one address, one request
    const float acc = group_sum<G>(row_partial<G>(col, val, x, rowptr[row], rowptr[row + 1], lane));
    if (lane == 0) emit_with<EPI>(row, acc, in, ea);
}

// Long rows, a wave each: chunks of 1024 entries are loaded 16 bytes per
// work-item (a quarter of the load instructions) and turned in LDS, so that
// a gather instruction still reads 64 consecutive entries, whose columns
// share cache lines (gathering straight from the 16-byte pieces, four
// entries apart, misses L1 more than the saved loads are worth).  16 gathers
// per work-item are in flight, the next chunk's loads behind them.  Chunks
// start at a multiple of four entries (aligned pieces); pieces that reach
// past the row's end are read entry by entry.  A wave uses its own part of
// LDS: no barriers.
// Bound by L1 on the gathers of x (hits on lines still being fetched): on
// the mid-sized scanner (1085 entries per row, 1.8e8 nonzeros) FP takes 0.475
// ms (3.0 TB/s of matrix) and BP 0.461, csr_vector_kernel 0.549 and 0.560;
// on the 12 GB scanner 4.16 and 3.92 ms against 4.59 and 4.56.  Six pieces per
// chunk are within 1% of four, one or two 8% slower, eight (LDS for two
// workgroups of 256) 30%.
// Mean entries per row from which it is used (64 work-items per row by
// default too): rows of 440 gain 5%, of 550-620 7-23%; shorter rows leave
// most of a chunk empty.
constexpr uint32_t kLongMean = 384;
constexpr int kLongNT = 512;
constexpr int kLongQ = 4;  // 16-byte pieces of col and of val per work-item and chunk
template <int EPI>
__global__ __launch_bounds__(kLongNT) void csr_long_rows_kernel(const uint64_t *__restrict__ rowptr,
                                                                const uint32_t *__restrict__ col,
                                                                const float *__restrict__ val,
                                                                const float *__restrict__ x, uint32_t rows,
                                                                EpiArgs ea) {
    constexpr int Q = kLongQ, NW = kLongNT / 64;
    constexpr uint32_t CH = 256 * Q;  // entries per chunk
    __shared__ __attribute__((aligned(16))) uint32_t s_c[NW][CH];
    __shared__ __attribute__((aligned(16))) float s_v[NW][CH];
    const uint32_t wv = threadIdx.x / 64, lane = threadIdx.x % 64;
    const uint32_t row = blockIdx.x * (uint32_t)NW + wv;
    if (row >= rows) return;
    const EpiIn in = epi_load<EPI>(row, ea);
    const uint64_t b = rowptr[row], e = rowptr[row + 1];
    uint32_t *sc = s_c[wv];
    float *sv = s_v[wv];
    u32x4 c4[Q];
    f32x4 v4[Q];
    auto load = [&](uint64_t k) {
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const uint64_t i = k + 256 * q + 4 * lane;
            if (i + 4 <= e) {
                c4[q] = ldnt(reinterpret_cast<const u32x4 *>(col + i));
                v4[q] = ldnt(reinterpret_cast<const f32x4 *>(val + i));
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const bool ok = i + j < e;
                    c4[q][j] = ok ? col[i + j] : 0u;
                    v4[q][j] = ok ? val[i + j] : 0.0f;
                }
            }
        }
    };
    float acc = 0.0f;
    const uint64_t k0 = b & ~3ull;
    if (b < e) load(k0);
    for (uint64_t k = k0; k < e; k += CH) {
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            *reinterpret_cast<u32x4 *>(sc + 256 * q + 4 * lane) = c4[q];
            *reinterpret_cast<f32x4 *>(sv + 256 * q + 4 * lane) = v4[q];
        }
        if (k + CH < e) load(k + CH);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        float xv[4 * Q], vv[4 * Q];
#pragma unroll
        for (int u = 0; u < 4 * Q; ++u) {
            const uint64_t i = k + 64 * u + lane;
            vv[u] = sv[64 * u + lane];
            xv[u] = (i >= b && i < e) ? x[sc[64 * u + lane]] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < 4 * Q; ++u) {
            const uint64_t i = k + 64 * u + lane;
            if (i >= b && i < e) acc += vv[u] * xv[u];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    acc = group_sum<64>(acc);
    if (lane == 0) emit_with<EPI>(row, acc, in, ea);
}

// ---------------------------------------------------------------------------
// merge path
// ---------------------------------------------------------------------------

// Merge of the row ends a_i = rowptr[i+1] (i < rows) with the nonzero
// positions 0..nnz-1, a_i taken before nonzero j iff a_i <= j (the order of
// merge_based_work, kernel.cu:271-282).  The split point of diagonal d is the
// smallest i in [max(0, d-nnz), min(d, rows)] with rowptr[i+1] + i >= d,
// i.e. rowptr[i+1] > (d-i) - 1 (the search of merge_based_start,
// kernel.cu:202-229, without its read of rowptr[rows+1]).
__global__ void merge_partition_kernel(const uint64_t *__restrict__ rowptr, uint32_t rows, uint64_t nnz,
                                       uint64_t tile_items, uint32_t ntiles, uint32_t *__restrict__ tile_row,
                                       uint64_t *__restrict__ tile_nz) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t > ntiles) return;
    const uint64_t L = (uint64_t)rows + nnz;
    uint64_t d = (uint64_t)t * tile_items;
    if (d > L) d = L;
    uint64_t lo = d > nnz ? d - nnz : 0;
    uint64_t hi = d < rows ? d : rows;
    while (lo < hi) {
        const uint64_t mid = (lo + hi) >> 1;
        if (rowptr[mid + 1] + mid >= d)
            hi = mid;
        else
            lo = mid + 1;
    }
    tile_row[t] = (uint32_t)lo;
    tile_nz[t] = d - lo;
}

// The same split point found by a wave: 64 probes per round (three rounds of
// loads for 41,000 rows where one work-item takes sixteen).  Every lane gets
// it.
__device__ __forceinline__ uint32_t merge_split_wave(const uint64_t *__restrict__ rowptr, uint32_t rows, uint64_t nnz,
                                                     uint64_t d, uint32_t lane) {
    uint64_t lo = d > nnz ? d - nnz : 0, hi = d < rows ? d : rows;
    while (lo < hi) {  // ends: the range shrinks to less than a 64th, at least by one
        const uint64_t step = (hi - lo + 63) / 64, at = lo + lane * step;
        const bool past = at >= hi || rowptr[at + 1] + at >= d;
        const uint64_t m = __ballot(past);
        const uint32_t f = m ? (uint32_t)__builtin_ctzll(m) : 64u;  // the first probe at or past the split
        hi = f == 64u ? hi : (lo + f * step < hi ? lo + f * step : hi);
        lo = f == 0u ? lo : lo + (f - 1) * step + 1;
    }
    return (uint32_t)lo;
}

// SEARCH: the partition does not exist yet.  Two waves find the tile's two
// split points and the tile stores its own for the fix-up.
template <int EPI, bool SEARCH>
__global__ __launch_bounds__(kWG) void merge_spmv_kernel(const uint64_t *__restrict__ rowptr,
                                                         const uint32_t *__restrict__ col,
                                                         const float *__restrict__ val, const float *__restrict__ x,
                                                         uint32_t S, uint32_t rows, uint64_t nnz, uint32_t *tile_row,
                                                         uint64_t *tile_nz, float *__restrict__ tile_carry,
                                                         float *__restrict__ tile_head, EpiArgs ea) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    __shared__ float s_wv[kWG / 64];
    __shared__ int s_wf[kWG / 64];
    __shared__ uint32_t s_row[2];

    const uint32_t t = blockIdx.x;
    const uint32_t tid = threadIdx.x;
    uint32_t i0, i1;
    uint64_t j0, j1;
    if constexpr (SEARCH) {
        const uint64_t L = (uint64_t)rows + nnz, T = (uint64_t)kWG * S;
        const uint64_t d0 = t * T, d1 = d0 + T < L ? d0 + T : L;  // t * T < L
        const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);
        if (w < 2) {
            const uint32_t r = merge_split_wave(rowptr, rows, nnz, w ? d1 : d0, tid & 63u);
            if ((tid & 63u) == 0) s_row[w] = r;
        }
        __syncthreads();
        i0 = s_row[0];
        i1 = s_row[1];
        j0 = d0 - i0;
        j1 = d1 - i1;
        if (tid < 2 && (tid == 0 || t + 1 == gridDim.x)) {
            tile_row[t + tid] = tid ? i1 : i0;
            tile_nz[t + tid] = tid ? j1 : j0;
        }
    } else {
        i0 = tile_row[t];
        i1 = tile_row[t + 1];
        j0 = tile_nz[t];
        j1 = tile_nz[t + 1];
    }
    const uint32_t nr = i1 - i0;              // row ends in this tile
    const uint32_t nz = (uint32_t)(j1 - j0);  // nonzeros in this tile
    const uint32_t h = (uint32_t)(j0 & 3u);   // s_val[h + jl] holds nonzero j0 + jl
    float *s_val = smem;
    uint32_t *s_end = reinterpret_cast<uint32_t *>(smem + ((h + nz + 3u) & ~3u));

    // Stage products val*x[col] with aligned 16-byte loads and the local row
    // ends.  The tile's edge quads: on its own (SEARCH, a small matrix whose
    // tile is one chain of latencies) loaded whole, a neighbour's entries in
    // them unused; else element by element, which costs the chain another
    // round trip but was the faster on large matrices (mid-sized scanner,
    // 87,811 tiles, FP + BP: 1046 against 1110 us; 2D ring 36.7 against 35.0).
    const uint64_t ja = j0 - h;
    const uint32_t nq = (h + nz + 3u) >> 2;
    for (uint32_t q = tid; q < nq; q += kWG) {
        const uint64_t jq = ja + 4ull * q;
        if (SEARCH ? jq + 4 <= nnz : jq >= j0 && jq + 4 <= j1) {
            const u32x4 c = ldnt(reinterpret_cast<const u32x4 *>(col + jq));
            const f32x4 v = ldnt(reinterpret_cast<const f32x4 *>(val + jq));
            f32x4 p;
            p.x = v.x * x[c.x];
            p.y = v.y * x[c.y];
            p.z = v.z * x[c.z];
            p.w = v.w * x[c.w];
            *reinterpret_cast<f32x4 *>(s_val + 4u * q) = p;
        } else {
            for (uint32_t e = 0; e < 4; ++e) {
                const uint64_t j = jq + e;
                if (j >= j0 && j < j1) s_val[4u * q + e] = val[j] * x[col[j]];
            }
        }
    }
    for (uint32_t q = tid; q < nr; q += kWG) s_end[q] = (uint32_t)(rowptr[(uint64_t)i0 + 1 + q] - j0);
    __syncthreads();

    // Each work-item walks S consecutive merge items of the tile.
    const uint32_t Tt = nr + nz;
    uint32_t d0 = tid * S;
    if (d0 > Tt) d0 = Tt;
    const uint32_t d1 = (d0 + S < Tt) ? d0 + S : Tt;
    uint32_t lo = d0 > nz ? d0 - nz : 0u;
    uint32_t hi = d0 < nr ? d0 : nr;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (s_end[mid] + mid >= d0)
            hi = mid;
        else
            lo = mid + 1;
    }
    const uint32_t first = lo;
    uint32_t i = lo, j = d0 - lo;
    float acc = 0.0f, head = 0.0f;
    int has_end = 0;
    for (uint32_t d = d0; d < d1; ++d) {
        if (i < nr && s_end[i] <= j) {
            if (has_end)
                emit<EPI>(i0 + i, acc, ea);  // row started and ended in this work-item
            else {
                head = acc;
                has_end = 1;
            }
            acc = 0.0f;
            ++i;
        } else {
            acc += s_val[h + j];
            ++j;
        }
    }

    // Segmented inclusive scan of (has_end, carry) over the workgroup:
    // (f1,v1) (+) (f2,v2) = (f1|f2, f2 ? v2 : v1+v2), left operand first.
    const uint32_t lane = tid & 63u, w = tid >> 6;
    float v = acc;
    int f = has_end;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const float vu = __shfl_up(v, o);
        const int fu = __shfl_up(f, o);
        if (lane >= (uint32_t)o) {
            if (!f) v = vu + v;
            f |= fu;
        }
    }
    if (lane == 63) {
        s_wv[w] = v;
        s_wf[w] = f;
    }
    __syncthreads();
    float pv = 0.0f;
    int pf = 0;
    for (uint32_t u = 0; u < w; ++u) {
        pv = s_wf[u] ? s_wv[u] : pv + s_wv[u];
        pf |= s_wf[u];
    }
    const float iv = f ? v : pv + v;
    const int ifl = pf | f;
    float ev = __shfl_up(iv, 1);
    int ef = __shfl_up(ifl, 1);
    if (lane == 0) {
        ev = pv;
        ef = pf;
    }
    if (has_end) {
        const float tot = ev + head;
        // The tile's first finished row started in an earlier tile: leave its
        // partial to the fix-up kernel.
        if (!ef && rowptr[i0] < j0)
            tile_head[t] = tot;
        else
            emit<EPI>(i0 + first, tot, ea);
    }
    if (tid == kWG - 1) tile_carry[t] = iv;
}

// Rows whose nonzeros span tiles: sum the carries of the tiles before the
// one that ends the row, in tile order, then that tile's head partial.
template <int EPI>
__global__ void merge_fixup_kernel(const uint64_t *__restrict__ rowptr, uint32_t ntiles,
                                   const uint32_t *__restrict__ tile_row, const uint64_t *__restrict__ tile_nz,
                                   const float *__restrict__ tile_carry, const float *__restrict__ tile_head,
                                   EpiArgs ea) {
    const uint32_t u = blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= ntiles) return;
    const uint32_t r = tile_row[u];
    if (tile_row[u + 1] == r) return;       // no row ends in tile u
    if (!(rowptr[r] < tile_nz[u])) return;  // its first row starts inside tile u (always so for u == 0)
    uint32_t s = u - 1;
    while (s > 0 && tile_row[s] == r) --s;
    float tot = 0.0f;
    for (uint32_t q = s; q < u; ++q) tot += tile_carry[q];
    emit<EPI>(r, tot + tile_head[u], ea);
}

// ---------------------------------------------------------------------------
// scatter BP, elementwise, sensitivity, log-likelihood
// ---------------------------------------------------------------------------
template <int G>
__global__ __launch_bounds__(kWG) void scatter_kernel(const uint64_t *__restrict__ rowptr,
                                                      const uint32_t *__restrict__ col,
                                                      const float *__restrict__ val, const float *__restrict__ xrow,
                                                      float *__restrict__ out, uint32_t rows) {
    const uint32_t row = blockIdx.x * (uint32_t)(kWG / G) + threadIdx.x / G;
    const uint32_t lane = threadIdx.x % G;
    if (row >= rows) return;
    const float r = xrow[row];
    if (r == 0.0f) return;  // adding +0 leaves every (non-negative zero) sum unchanged
    const uint64_t b = rowptr[row], e = rowptr[row + 1];
    for (uint64_t k = b + lane; k < e; k += G) unsafeAtomicAdd(out + ldnt(col + k), ldnt(val + k) * r);
}

// Scatter BP with the sums of a window of columns in LDS: a workgroup owns up
// to kWinRows rows (one per lane of its waves) and walks them window by
// window; in a window every wave takes its rows that reach into it, a piece
// of 64 U entries at a time, S rows in flight, and adds into LDS.  The
// window's sums then go out as one run of consecutive atomics instead of one
// scattered atomic per entry (a wave's 64 entries touch 25 lines; the
// device-wide adds are done per line).  P is the next entry of the lane's
// row, NC its column.  A row leaves a window at its first entry outside it;
// what an unsorted row still holds after the last window is added entry by
// entry.  The walk ends: a slot advances a piece or closes, and each window
// opens a row once.
//
// The sums are FP64 where a row has many entries in a window: the LDS adds an
// FP32 value of one lane after the other (193 clocks per wave instruction
// whatever the addresses, measured), FP64 values in 20 to 60.  Half as many
// columns fit, so rows open twice as often, which is what short rows cost.
// Bound by the loads then (without the adds 0.50 ms, without what goes out
// 0.51 of the 0.55; loads that stay in the caches for the next window's
// pieces bring it to 0.51).  Rows dealt to the workgroups in turn, which
// balances them better, lose: neighbours share columns, so fewer sums go out
// (0.52, and 113 against 91 us with 4.4e7 nonzeros).  us with non-temporal
// loads, every row's factor nonzero; FP32 sums / FP64 with
// U = 1, S = 4 / FP64 with U = 2, S = 3, by the mean entries e of a row in
// 32,768 columns:
//   1e6 rows x 200,000, e = 3          938 / 1300 / 1581
//   200,000 x 100,000, e = 12          164 /  191 /  218
//   200,000 x 100,000, e = 25          212 /  208 /  241
//   200,000 x 100,000, e = 50          311 /  216 /  263
//   mid-sized scanner, e = 155        1153 /  574 /  550  (scattered atomics 4165)
//   500 rows x 100,000, e = 1000       103 /  102 /   85
// The 12 GB scanner takes 5.1 ms (FP32 sums 9.3, scattered atomics 34.7).
constexpr int kWinNT = 1024;
constexpr uint32_t kWinRows = 64 * (kWinNT / 64);  // rows per workgroup at most
constexpr uint32_t kWinColsF32 = 32768, kWinColsF64 = 20224;  // columns per window (128 and 158 KB)

__device__ __forceinline__ uint64_t readlane64(uint64_t v, uint32_t k) {
    return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), k) << 32) |
           (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, k);
}

template <typename T, uint32_t kWinCols, int U, int S>
__global__ __launch_bounds__(kWinNT) void scatter_window_kernel(const uint64_t *__restrict__ rowptr,
                                                                const uint32_t *__restrict__ col,
                                                                const float *__restrict__ val,
                                                                const float *__restrict__ xrow,
                                                                float *__restrict__ out, uint32_t rows, uint32_t cols,
                                                                uint32_t per_wg) {
    extern __shared__ __attribute__((aligned(16))) char win_mem[];
    T *win = reinterpret_cast<T *>(win_mem);         // [kWinCols]
    constexpr uint32_t NW = kWinNT / 64, PC = 64 * U;  // PC: entries per piece
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r0 = blockIdx.x * per_wg, nr = min(per_wg, rows - r0);
    const uint32_t mine = wv + NW * lane;  // lane k of wave w: row r0 + w + NW * k
    const float f = mine < nr ? xrow[r0 + mine] : 0.0f;
    const bool has = f != 0.0f;  // adding +0 leaves every (non-negative zero) sum unchanged
    const uint64_t base = rowptr[r0];
    uint64_t P = has ? rowptr[r0 + mine] : 0;
    const uint64_t E = has ? rowptr[r0 + mine + 1] : 0;
    uint32_t NC = P < E ? col[P] : 0xffffffffu;
    for (uint32_t w0 = 0; w0 < cols;) {
        const uint32_t wn = min(kWinCols, cols - w0), w1 = w0 + wn;
        if (!__syncthreads_or(NC < w1)) {  // no row of the workgroup reaches into this window
            w0 = w1;
            continue;
        }
        for (uint32_t i = tid; i < wn; i += kWinNT) win[i] = T(0);
        __syncthreads();
        uint64_t todo = __ballot(NC < w1);
        if (todo) {
            uint64_t p[S], left[S];  // next entry, entries from it on (0: no row)
            uint32_t row[S], c[S][U], nopen = 0;
            float a[S], v[S][U];
            auto take = [&](int j) {
                p[j] = base;
                left[j] = 0;
                row[j] = 0;
                a[j] = 0.0f;
                if (todo) {
                    const uint32_t k = (uint32_t)__builtin_ctzll(todo);
                    todo &= todo - 1;
                    row[j] = k;
                    p[j] = readlane64(P, k);
                    left[j] = readlane64(E, k) - p[j];
                    a[j] = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(f), k));
                    ++nopen;
                }
            };
            // Lanes past the row's end re-read its entry p (a slot without a
            // row: the workgroup's first entry), so the loads are unconditional.
            // Not non-temporal: a row's piece that ends in the next window is
            // read again there, from the MALL.
            auto fetch = [&](int j) {
#pragma unroll
                for (uint32_t u = 0; u < (uint32_t)U; ++u) {
                    const uint32_t l = lane + 64 * u < left[j] ? lane + 64 * u : 0u;
                    c[j][u] = col[p[j] + l];
                    v[j][u] = val[p[j] + l];
                }
            };
#pragma unroll
            for (int j = 0; j < S; ++j) {
                take(j);
                fetch(j);
            }
            while (nopen) {
#pragma unroll
                for (int j = 0; j < S; ++j) {
                    const uint32_t rj = row[j];
                    const uint64_t pj = p[j], lj = left[j];
                    uint32_t cc[U], n = 0;  // n: entries in the window
                    float t[U];
#pragma unroll
                    for (uint32_t u = 0; u < (uint32_t)U; ++u) {
                        cc[u] = c[j][u];
                        t[u] = v[j][u] * a[j];
                        const uint64_t m = ~__ballot(cc[u] >= w0 && cc[u] < w1 && lane + 64 * u < lj);
                        if (n == 64 * u) n += m ? (uint32_t)__builtin_ctzll(m) : 64u;
                    }
                    const bool more = n == PC && lj > PC;
                    if (more) {
                        p[j] += PC;
                        left[j] -= PC;
                    } else {
                        nopen -= lj ? 1u : 0u;
                        take(j);
                    }
                    fetch(j);
#pragma unroll
                    for (uint32_t u = 0; u < (uint32_t)U; ++u)
                        if (lane + 64 * u < n) unsafeAtomicAdd(win + (cc[u] - w0), (T)t[u]);
                    if (lj && !more) {
                        uint32_t nc = 0xffffffffu;
                        if (n < lj) {
                            nc = (uint32_t)__builtin_amdgcn_readlane((int)cc[0], n & 63u);
#pragma unroll
                            for (uint32_t u = 1; u < (uint32_t)U; ++u)
                                if (n >= 64 * u) nc = (uint32_t)__builtin_amdgcn_readlane((int)cc[u], n & 63u);
                        }
                        if (lane == rj) {
                            P = pj + n;
                            NC = nc;
                        }
                    }
                }
            }
        }
        __syncthreads();
        for (uint32_t i = tid; i < wn; i += kWinNT)
            if (win[i] != T(0)) unsafeAtomicAdd(out + w0 + i, (float)win[i]);
        __syncthreads();
        w0 = w1;
    }
    for (uint64_t rest = __ballot(P < E); rest; rest &= rest - 1) {  // unsorted rows
        const uint32_t k = (uint32_t)__builtin_ctzll(rest);
        const float a = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(f), k));
        const uint64_t e = readlane64(E, k);
        for (uint64_t i = readlane64(P, k) + lane; i < e; i += 64) unsafeAtomicAdd(out + col[i], val[i] * a);
    }
}

__global__ void ratio_kernel(const int32_t *__restrict__ g, float *__restrict__ fw, uint32_t rows) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < rows) {
        const float y = fw[i];
        if (y != 0.0f) fw[i] = (float)g[i] / y;
    }
}

__global__ void update_kernel(const float *__restrict__ f, const float *__restrict__ norm, float *__restrict__ bw,
                              uint32_t cols) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < cols) {
        const float v = f[i] * bw[i];
        const float n = norm[i];
        bw[i] = (n == 0.0f) ? v : v / n;
    }
}

__global__ void update_image_kernel(float *__restrict__ f, const float *__restrict__ norm, float *__restrict__ bp,
                                    uint32_t cols) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < cols) {
        const float v = f[i] * bp[i];
        const float n = norm[i];
        f[i] = (n == 0.0f) ? v : v / n;
        bp[i] = 0.0f;
    }
}

template <typename T>
__global__ void fill_kernel(T *__restrict__ dst, T v, uint64_t n) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        dst[i] = v;
}

// dst = src over n floats, 16 bytes per work-item per step.
__global__ __launch_bounds__(kWG) void copy_kernel(float *__restrict__ dst, const float *__restrict__ src,
                                                   uint64_t n) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    const uint64_t n4 = n / 4, stride = (uint64_t)gridDim.x * kWG;
    for (uint64_t i = blockIdx.x * (uint64_t)kWG + threadIdx.x; i < n4; i += stride)
        __builtin_nontemporal_store(__builtin_nontemporal_load(reinterpret_cast<const f4 *>(src) + i),
                                    reinterpret_cast<f4 *>(dst) + i);
    for (uint64_t i = 4 * n4 + blockIdx.x * (uint64_t)kWG + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

// csr4 AoS {u32 col, f32 val} entries [first, first+n) of the matrix -> SoA;
// bit 1 of *bad: a column index >= cols.
__global__ __launch_bounds__(kWG) void aos_split_kernel(const uint32_t *__restrict__ aos, uint64_t n, uint64_t first,
                                                        uint32_t cols, uint32_t *__restrict__ col,
                                                        float *__restrict__ val, uint32_t *__restrict__ bad) {
    const uint64_t stride = (uint64_t)gridDim.x * kWG;
    uint32_t flag = 0;
    for (uint64_t i = blockIdx.x * (uint64_t)kWG + threadIdx.x; i < n; i += stride) {
        const uint32_t c = __builtin_nontemporal_load(aos + 2 * i);
        const uint32_t v = __builtin_nontemporal_load(aos + 2 * i + 1);
        flag |= c >= cols ? 1u : 0u;
        col[first + i] = c;
        val[first + i] = __uint_as_float(v);
    }
    if (flag) atomicOr(bad, 1u);
}

// *first = the smallest k with col[k] >= cols (unchanged when there is none;
// the caller starts it at UINT64_MAX).
__global__ void first_bad_column_kernel(const uint32_t *__restrict__ col, uint64_t n, uint32_t cols,
                                        unsigned long long *__restrict__ first) {
    for (uint64_t k = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; k < n; k += (uint64_t)gridDim.x * blockDim.x)
        if (col[k] >= cols) {
            atomicMin(first, (unsigned long long)k);
            return;
        }
}

// One slot of an interleaved [n][stride] array <-> a contiguous vector.
template <typename T>
__global__ void strided_put_kernel(T *__restrict__ dst, uint32_t stride, const T *__restrict__ src, uint64_t n) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        dst[i * stride] = src[i];
}
template <typename T>
__global__ void strided_get_kernel(T *__restrict__ dst, const T *__restrict__ src, uint32_t stride, uint64_t n) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        dst[i] = src[i * stride];
}

__global__ void f64_to_f32_kernel(const double *__restrict__ a, float *__restrict__ b, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = (float)a[i];
}

// Row sums of A^T (= column sums of A) in FP64, 64 work-items per row.
__global__ __launch_bounds__(kWG) void colsum_rows_kernel(const uint64_t *__restrict__ rowptrT,
                                                          const float *__restrict__ valT, uint32_t cols,
                                                          double *__restrict__ s64, float *__restrict__ s32) {
    const uint32_t row = blockIdx.x * (uint32_t)(kWG / 64) + threadIdx.x / 64;
    const uint32_t lane = threadIdx.x % 64;
    if (row >= cols) return;
    double acc = 0.0;
    for (uint64_t k = rowptrT[row] + lane; k < rowptrT[row + 1]; k += 64) acc += (double)valT[k];
    acc = group_sum_f64<64>(acc);
    if (lane == 0) {
        if (s64) s64[row] = acc;
        if (s32) s32[row] = (float)acc;
    }
}

// s[c] = sum over row c of A^T of valT[k] * w[rowT[k]] (FP64): the column
// sums of a matrix given as row weights times codes.
__global__ __launch_bounds__(kWG) void colsum_weighted_kernel(const uint64_t *__restrict__ rowptrT,
                                                              const uint32_t *__restrict__ rowT,
                                                              const float *__restrict__ valT,
                                                              const float *__restrict__ w, uint32_t cols,
                                                              double *__restrict__ s64, float *__restrict__ s32) {
    const uint32_t row = blockIdx.x * (uint32_t)(kWG / 64) + threadIdx.x / 64;
    const uint32_t lane = threadIdx.x % 64;
    if (row >= cols) return;
    double acc = 0.0;
    for (uint64_t k = rowptrT[row] + lane; k < rowptrT[row + 1]; k += 64) acc += (double)valT[k] * (double)w[rowT[k]];
    acc = group_sum_f64<64>(acc);
    if (lane == 0) {
        if (s64) s64[row] = acc;
        if (s32) s32[row] = (float)acc;
    }
}

__global__ __launch_bounds__(kWG) void colsum_scatter_kernel(const uint64_t *__restrict__ rowptr,
                                                             const uint32_t *__restrict__ col,
                                                             const float *__restrict__ val, uint32_t rows,
                                                             double *__restrict__ s64) {
    const uint32_t row = blockIdx.x * (uint32_t)(kWG / 64) + threadIdx.x / 64;
    const uint32_t lane = threadIdx.x % 64;
    if (row >= rows) return;
    for (uint64_t k = rowptr[row] + lane; k < rowptr[row + 1]; k += 64) unsafeAtomicAdd(s64 + col[k], (double)val[k]);
}

// Per-row l_i = g_i log(y_i) - y_i with y = A x (terms with y_i <= 0
// contribute -y_i), FP64, one partial per workgroup in a fixed order.
template <int G>
__global__ __launch_bounds__(kWG) void loglik_kernel(const uint64_t *__restrict__ rowptr,
                                                     const uint32_t *__restrict__ col, const float *__restrict__ val,
                                                     const float *__restrict__ x, const int32_t *__restrict__ g,
                                                     uint32_t rows, double *__restrict__ part) {
    __shared__ double s[kWG / G];
    const uint32_t row = blockIdx.x * (uint32_t)(kWG / G) + threadIdx.x / G;
    const uint32_t lane = threadIdx.x % G;
    double l = 0.0;
    if (row < rows) {
        const float y = group_sum<G>(row_partial<G>(col, val, x, rowptr[row], rowptr[row + 1], lane));
        const double yd = (double)y;
        l = (yd > 0.0) ? (double)g[row] * log(yd) - yd : -yd;
    }
    if (lane == 0) s[threadIdx.x / G] = l;
    __syncthreads();
    if (threadIdx.x == 0) {
        double acc = 0.0;
        for (int q = 0; q < kWG / G; ++q) acc += s[q];
        part[blockIdx.x] = acc;
    }
}

inline uint32_t blocks_for(uint64_t n, uint32_t per) { return (uint32_t)((n + per - 1) / per); }

template <int EPI>
hipError_t launch_merge_epi(const MergePlan &p, bool search, uint32_t *tile_row, uint64_t *tile_nz, float *carry,
                            float *head, const uint64_t *rowptr, const uint32_t *col, const float *val,
                            const float *x, const EpiArgs &ea, hipStream_t s) {
    const size_t lds = (p.tile_items + 8) * sizeof(float);
    if (search)
        hipLaunchKernelGGL((merge_spmv_kernel<EPI, true>), dim3(p.ntiles), dim3(kWG), lds, s, rowptr, col, val, x,
                           p.secsize, p.rows, p.nnz, tile_row, tile_nz, carry, head, ea);
    else
        hipLaunchKernelGGL((merge_spmv_kernel<EPI, false>), dim3(p.ntiles), dim3(kWG), lds, s, rowptr, col, val, x,
                           p.secsize, p.rows, p.nnz, tile_row, tile_nz, carry, head, ea);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || p.ntiles == 1) return e;  // one tile: no row spans two
    hipLaunchKernelGGL(merge_fixup_kernel<EPI>, dim3(blocks_for(p.ntiles, kWG)), dim3(kWG), 0, s, rowptr, p.ntiles,
                       tile_row, tile_nz, carry, head, ea);
    return hipGetLastError();
}

template <int G>
hipError_t launch_csr_vector_g(const uint64_t *rowptr, const uint32_t *col, const float *val, const float *x,
                               uint32_t rows, Epi epi, const EpiArgs &ea, hipStream_t s) {
    const dim3 grid(blocks_for(rows, kWG / G)), block(kWG);
    switch (epi) {
        case EPI_PLAIN: hipLaunchKernelGGL((csr_vector_kernel<G, EPI_PLAIN>), grid, block, 0, s, rowptr, col, val, x, rows, ea); break;
        case EPI_RATIO: hipLaunchKernelGGL((csr_vector_kernel<G, EPI_RATIO>), grid, block, 0, s, rowptr, col, val, x, rows, ea); break;
        default: hipLaunchKernelGGL((csr_vector_kernel<G, EPI_UPDATE>), grid, block, 0, s, rowptr, col, val, x, rows, ea); break;
    }
    return hipGetLastError();
}

template <typename T, uint32_t COLS, int U, int S>
hipError_t launch_window(const uint64_t *rowptr, const uint32_t *col, const float *val, const float *xrow, float *out,
                         uint32_t rows, uint32_t cols, uint32_t per, hipStream_t s) {
    hipLaunchKernelGGL((scatter_window_kernel<T, COLS, U, S>), dim3(blocks_for(rows, per)), dim3(kWinNT),
                       COLS * sizeof(T), s, rowptr, col, val, xrow, out, rows, cols, per);
    return hipGetLastError();
}

template <int G>
hipError_t launch_scatter_g(const uint64_t *rowptr, const uint32_t *col, const float *val, const float *xrow,
                            float *out, uint32_t rows, hipStream_t s) {
    hipLaunchKernelGGL(scatter_kernel<G>, dim3(blocks_for(rows, kWG / G)), dim3(kWG), 0, s, rowptr, col, val, xrow,
                       out, rows);
    return hipGetLastError();
}

template <int G>
hipError_t launch_loglik_g(const uint64_t *rowptr, const uint32_t *col, const float *val, const float *x,
                           const int32_t *g, uint32_t rows, double *part, hipStream_t s) {
    hipLaunchKernelGGL(loglik_kernel<G>, dim3(blocks_for(rows, kWG / G)), dim3(kWG), 0, s, rowptr, col, val, x, g,
                       rows, part);
    return hipGetLastError();
}

constexpr size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

}  // namespace

MergePlan merge_plan(uint32_t rows, uint64_t nnz, uint32_t secsize) {
    MergePlan p;
    p.rows = rows;
    p.nnz = nnz;
    p.secsize = secsize;
    p.tile_items = (uint64_t)kWG * secsize;
    const uint64_t L = (uint64_t)rows + nnz;
    p.ntiles = secsize ? (uint32_t)((L + p.tile_items - 1) / p.tile_items) : 0;
    return p;
}

size_t merge_partition_bytes(const MergePlan &p) {
    return align256(sizeof(uint32_t) * ((size_t)p.ntiles + 1)) + align256(sizeof(uint64_t) * ((size_t)p.ntiles + 1));
}

size_t merge_scratch_bytes(const MergePlan &p) { return 2 * align256(sizeof(float) * ((size_t)p.ntiles + 1)); }

hipError_t launch_merge_partition(const MergePlan &p, const uint64_t *rowptr, void *partition, hipStream_t s) {
    if (p.rows == 0) return hipSuccess;
    uint32_t *tile_row = static_cast<uint32_t *>(partition);
    uint64_t *tile_nz = reinterpret_cast<uint64_t *>(static_cast<char *>(partition) +
                                                     align256(sizeof(uint32_t) * ((size_t)p.ntiles + 1)));
    hipLaunchKernelGGL(merge_partition_kernel, dim3(blocks_for((uint64_t)p.ntiles + 1, kWG)), dim3(kWG), 0, s,
                       rowptr, p.rows, p.nnz, p.tile_items, p.ntiles, tile_row, tile_nz);
    return hipGetLastError();
}

namespace {
hipError_t merge_launch(const MergePlan &p, bool search, void *partition, void *scratch, const uint64_t *rowptr,
                        const uint32_t *col, const float *val, const float *x, Epi epi, const EpiArgs &ea,
                        hipStream_t s) {
    uint32_t *tile_row = static_cast<uint32_t *>(partition);
    uint64_t *tile_nz = reinterpret_cast<uint64_t *>(static_cast<char *>(partition) +
                                                     align256(sizeof(uint32_t) * ((size_t)p.ntiles + 1)));
    float *carry = static_cast<float *>(scratch);
    float *head = reinterpret_cast<float *>(static_cast<char *>(scratch) + align256(sizeof(float) * ((size_t)p.ntiles + 1)));
    switch (epi) {
        case EPI_PLAIN: return launch_merge_epi<EPI_PLAIN>(p, search, tile_row, tile_nz, carry, head, rowptr, col, val, x, ea, s);
        case EPI_RATIO: return launch_merge_epi<EPI_RATIO>(p, search, tile_row, tile_nz, carry, head, rowptr, col, val, x, ea, s);
        default: return launch_merge_epi<EPI_UPDATE>(p, search, tile_row, tile_nz, carry, head, rowptr, col, val, x, ea, s);
    }
}
}  // namespace

hipError_t launch_merge_spmv(const MergePlan &p, const void *partition, void *scratch, const uint64_t *rowptr,
                             const uint32_t *col, const float *val, const float *x, Epi epi, const EpiArgs &ea,
                             hipStream_t s) {
    if (p.rows == 0) return hipSuccess;
    return merge_launch(p, false, const_cast<void *>(partition), scratch, rowptr, col, val, x, epi, ea, s);
}

// A small product is a chain of launches: the partition's own launch and its
// binary search (one work-item per tile, a memory latency per step) took as
// long as the search by waves inside the product takes for thousands of
// tiles.  FP + ratio + BP + update, us, partition launch / search: 2D ring
// (987 tiles) 36.7 / 30.5, 4262 tiles 74.0 / 69.1, 7804 tiles 116.7 / 113.0,
// 24497 tiles 301 / 319.
constexpr uint32_t kSearchTiles = 8192;
hipError_t launch_merge_once(const MergePlan &p, void *ws, const uint64_t *rowptr, const uint32_t *col,
                             const float *val, const float *x, Epi epi, const EpiArgs &ea, hipStream_t s) {
    if (p.rows == 0) return hipSuccess;
    const bool search = p.ntiles <= kSearchTiles;
    if (!search) {
        const hipError_t e = launch_merge_partition(p, rowptr, ws, s);
        if (e != hipSuccess) return e;
    }
    return merge_launch(p, search, ws, static_cast<char *>(ws) + merge_partition_bytes(p), rowptr, col, val, x, epi, ea, s);
}

// Rows per workgroup of the windowed scatter: whole rounds of a workgroup per
// CU (its LDS fills one), at most kWinRows each.
uint32_t scatter_window_rows(uint32_t rows) {
    const uint64_t wgs = 256ull * blocks_for(rows, 256 * kWinRows);
    return (uint32_t)((rows + wgs - 1) / wgs);
}

bool valid_lanes(uint32_t lanes) { return lanes == 4 || lanes == 8 || lanes == 16 || lanes == 32 || lanes == 64; }

// Lanes per row from the mean row length: one 16-byte load per lane should
// cover a mean row in about one to two rounds.
uint32_t auto_lanes(uint32_t rows, uint64_t nnz) {
    const double m = rows ? (double)nnz / rows : 0.0;
    if (m <= 16) return 4;
    // Rows of a few dozen entries with 8 lanes take two rounds of loads
    // (one memory latency each); 16 lanes take one: on the 2D ring (48 per
    // row, at most 115) FP ran 15.0 -> 11.1 us per launch.
    if (m <= 32) return 8;
    if (m <= 128) return 16;
    if (m <= 384) return 32;
    return 64;
}

template <int EPI>
hipError_t launch_csr_long(const uint64_t *rowptr, const uint32_t *col, const float *val, const float *x,
                           uint32_t rows, const EpiArgs &ea, hipStream_t s) {
    hipLaunchKernelGGL(csr_long_rows_kernel<EPI>, dim3(blocks_for(rows, kLongNT / 64)), dim3(kLongNT), 0, s, rowptr, col,
                       val, x, rows, ea);
    return hipGetLastError();
}

hipError_t launch_csr_vector(uint32_t lanes, const uint64_t *rowptr, const uint32_t *col, const float *val,
                             const float *x, uint32_t rows, uint64_t nnz, Epi epi, const EpiArgs &ea, hipStream_t s) {
    if (rows == 0) return hipSuccess;
    switch (lanes ? lanes : auto_lanes(rows, nnz)) {
        case 4: return launch_csr_vector_g<4>(rowptr, col, val, x, rows, epi, ea, s);
        case 8: return launch_csr_vector_g<8>(rowptr, col, val, x, rows, epi, ea, s);
        case 16: return launch_csr_vector_g<16>(rowptr, col, val, x, rows, epi, ea, s);
        case 32: return launch_csr_vector_g<32>(rowptr, col, val, x, rows, epi, ea, s);
        default: break;
    }
    if (nnz < (uint64_t)kLongMean * rows) return launch_csr_vector_g<64>(rowptr, col, val, x, rows, epi, ea, s);
    switch (epi) {
        case EPI_PLAIN: return launch_csr_long<EPI_PLAIN>(rowptr, col, val, x, rows, ea, s);
        case EPI_RATIO: return launch_csr_long<EPI_RATIO>(rowptr, col, val, x, rows, ea, s);
        default: return launch_csr_long<EPI_UPDATE>(rowptr, col, val, x, rows, ea, s);
    }
}

hipError_t launch_scatter(uint32_t lanes, const uint64_t *rowptr, const uint32_t *col, const float *val,
                          const float *xrow, float *out, uint32_t rows, uint32_t cols, uint64_t nnz, hipStream_t s) {
    if (rows == 0) return hipSuccess;
    if (lanes == 0) {
        const uint32_t per = scatter_window_rows(rows);
        const uint64_t nwg = blocks_for(rows, per);
        // Each workgroup clears and sends out its columns once, so the windows
        // pay from about one nonzero per 16 columns and workgroup on; windows /
        // scattered atomics, us: with one per 10 (1e6 x 200,000) 938 / 974,
        // per 6 (500 x 100,000) 108 / 142, per 25 (1e6 x 200,000) 754 / 394.
        if (16 * nnz >= nwg * cols) {
            const uint64_t wins = (uint64_t)rows * blocks_for(cols, kWinColsF32);  // nnz / wins: e above
            if (nnz < 25 * wins) return launch_window<float, kWinColsF32, 1, 4>(rowptr, col, val, xrow, out, rows, cols, per, s);
            if (nnz < 100 * wins) return launch_window<double, kWinColsF64, 1, 4>(rowptr, col, val, xrow, out, rows, cols, per, s);
            return launch_window<double, kWinColsF64, 2, 3>(rowptr, col, val, xrow, out, rows, cols, per, s);
        }
        lanes = auto_lanes(rows, nnz);
    }
    switch (lanes) {
        case 4: return launch_scatter_g<4>(rowptr, col, val, xrow, out, rows, s);
        case 8: return launch_scatter_g<8>(rowptr, col, val, xrow, out, rows, s);
        case 16: return launch_scatter_g<16>(rowptr, col, val, xrow, out, rows, s);
        case 32: return launch_scatter_g<32>(rowptr, col, val, xrow, out, rows, s);
        default: return launch_scatter_g<64>(rowptr, col, val, xrow, out, rows, s);
    }
}

hipError_t launch_ratio(const int32_t *g, float *fwproj, uint32_t rows, hipStream_t s) {
    if (rows == 0) return hipSuccess;
    hipLaunchKernelGGL(ratio_kernel, dim3(blocks_for(rows, kWG)), dim3(kWG), 0, s, g, fwproj, rows);
    return hipGetLastError();
}

hipError_t launch_update(const float *f, const float *norm, float *bwproj, uint32_t cols, hipStream_t s) {
    if (cols == 0) return hipSuccess;
    hipLaunchKernelGGL(update_kernel, dim3(blocks_for(cols, kWG)), dim3(kWG), 0, s, f, norm, bwproj, cols);
    return hipGetLastError();
}

hipError_t launch_update_image(float *f, const float *norm, float *bp, uint32_t cols, hipStream_t s) {
    if (cols == 0) return hipSuccess;
    hipLaunchKernelGGL(update_image_kernel, dim3(blocks_for(cols, kWG)), dim3(kWG), 0, s, f, norm, bp, cols);
    return hipGetLastError();
}

hipError_t launch_fill(float *dst, float v, uint64_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    uint64_t blocks = (n + kWG - 1) / kWG;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(fill_kernel<float>, dim3((uint32_t)blocks), dim3(kWG), 0, s, dst, v, n);
    return hipGetLastError();
}

hipError_t launch_copy(float *dst, const float *src, uint64_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    uint64_t blocks = (n / 4 + kWG - 1) / kWG;
    blocks = std::max<uint64_t>(1, std::min<uint64_t>(blocks, 8192));
    hipLaunchKernelGGL(copy_kernel, dim3((uint32_t)blocks), dim3(kWG), 0, s, dst, src, n);
    return hipGetLastError();
}

hipError_t launch_aos_split(const void *aos, uint64_t n, uint64_t first, uint32_t cols, uint32_t *col, float *val,
                            uint32_t *bad, hipStream_t s) {
    if (n == 0) return hipSuccess;
    const uint64_t blocks = std::max<uint64_t>(1, std::min<uint64_t>((n + kWG - 1) / kWG, 16384));
    hipLaunchKernelGGL(aos_split_kernel, dim3((uint32_t)blocks), dim3(kWG), 0, s, static_cast<const uint32_t *>(aos),
                       n, first, cols, col, val, bad);
    return hipGetLastError();
}

hipError_t launch_first_bad_column(const uint32_t *col, uint64_t n, uint32_t cols, uint64_t *first, hipStream_t s) {
    if (n == 0) return hipSuccess;
    const uint64_t blocks = std::max<uint64_t>(1, std::min<uint64_t>((n + kWG - 1) / kWG, 16384));
    hipLaunchKernelGGL(first_bad_column_kernel, dim3((uint32_t)blocks), dim3(kWG), 0, s, col, n, cols,
                       reinterpret_cast<unsigned long long *>(first));
    return hipGetLastError();
}

hipError_t launch_strided_put(void *dst, uint32_t stride, const void *src, uint64_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    const uint64_t blocks = std::max<uint64_t>(1, std::min<uint64_t>((n + kWG - 1) / kWG, 8192));
    hipLaunchKernelGGL(strided_put_kernel<uint32_t>, dim3((uint32_t)blocks), dim3(kWG), 0, s,
                       static_cast<uint32_t *>(dst), stride, static_cast<const uint32_t *>(src), n);
    return hipGetLastError();
}

hipError_t launch_strided_get(void *dst, const void *src, uint32_t stride, uint64_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    const uint64_t blocks = std::max<uint64_t>(1, std::min<uint64_t>((n + kWG - 1) / kWG, 8192));
    hipLaunchKernelGGL(strided_get_kernel<uint32_t>, dim3((uint32_t)blocks), dim3(kWG), 0, s,
                       static_cast<uint32_t *>(dst), static_cast<const uint32_t *>(src), stride, n);
    return hipGetLastError();
}

hipError_t launch_fill_u32(uint32_t *dst, uint32_t v, uint64_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    uint64_t blocks = (n + kWG - 1) / kWG;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(fill_kernel<uint32_t>, dim3((uint32_t)blocks), dim3(kWG), 0, s, dst, v, n);
    return hipGetLastError();
}

hipError_t launch_fill_f64(double *dst, double v, uint64_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    uint64_t blocks = (n + kWG - 1) / kWG;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(fill_kernel<double>, dim3((uint32_t)blocks), dim3(kWG), 0, s, dst, v, n);
    return hipGetLastError();
}

hipError_t launch_f64_to_f32(const double *a, float *b, uint32_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(f64_to_f32_kernel, dim3(blocks_for(n, kWG)), dim3(kWG), 0, s, a, b, n);
    return hipGetLastError();
}

hipError_t launch_colsum_rows_f64(const uint64_t *rowptrT, const float *valT, uint32_t cols, double *s64, float *s32,
                                  hipStream_t s) {
    if (cols == 0) return hipSuccess;
    hipLaunchKernelGGL(colsum_rows_kernel, dim3(blocks_for(cols, kWG / 64)), dim3(kWG), 0, s, rowptrT, valT, cols,
                       s64, s32);
    return hipGetLastError();
}

hipError_t launch_colsum_weighted_f64(const uint64_t *rowptrT, const uint32_t *rowT, const float *valT, const float *w,
                                      uint32_t cols, double *s64, float *s32, hipStream_t s) {
    if (cols == 0) return hipSuccess;
    hipLaunchKernelGGL(colsum_weighted_kernel, dim3(blocks_for(cols, kWG / 64)), dim3(kWG), 0, s, rowptrT, rowT, valT,
                       w, cols, s64, s32);
    return hipGetLastError();
}

hipError_t launch_colsum_scatter_f64(const uint64_t *rowptr, const uint32_t *col, const float *val, uint32_t rows,
                                     double *s64, hipStream_t s) {
    if (rows == 0) return hipSuccess;
    hipLaunchKernelGGL(colsum_scatter_kernel, dim3(blocks_for(rows, kWG / 64)), dim3(kWG), 0, s, rowptr, col, val,
                       rows, s64);
    return hipGetLastError();
}

uint32_t loglik_blocks(uint32_t rows) { return blocks_for(rows, kWG / 16); }

// The same terms from y = A x given (16 rows per block, as loglik_kernel<16>).
__global__ void loglik_y_kernel(const float *__restrict__ y, const int32_t *__restrict__ g, uint32_t rows,
                                double *__restrict__ part) {
    __shared__ double s[16];
    const uint32_t row = blockIdx.x * 16u + threadIdx.x;
    double l = 0.0;
    if (row < rows) {
        const double yd = (double)y[row];
        l = (yd > 0.0) ? (double)g[row] * log(yd) - yd : -yd;
    }
    s[threadIdx.x] = l;
    __syncthreads();
    if (threadIdx.x == 0) {
        double acc = 0.0;
        for (int q = 0; q < 16; ++q) acc += s[q];
        part[blockIdx.x] = acc;
    }
}

hipError_t launch_loglik_y(const float *y, const int32_t *g, uint32_t rows, double *part, hipStream_t s) {
    if (rows == 0) return hipSuccess;
    hipLaunchKernelGGL(loglik_y_kernel, dim3(loglik_blocks(rows)), dim3(16), 0, s, y, g, rows, part);
    return hipGetLastError();
}

hipError_t launch_loglik(const uint64_t *rowptr, const uint32_t *col, const float *val, const float *x,
                         const int32_t *g, uint32_t rows, double *part, hipStream_t s) {
    if (rows == 0) return hipSuccess;
    return launch_loglik_g<16>(rowptr, col, val, x, g, rows, part, s);
}

}  // namespace mlem
