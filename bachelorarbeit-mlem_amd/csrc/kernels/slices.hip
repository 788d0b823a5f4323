// Row slices: the layout of the batched kernels (several right-hand sides)
// for matrices whose rows are short in a tile, and its SpMV kernel.
//
// Why: with several right-hand sides the SpMV is bound by instructions and
// LDS, not by HBM.  In the block streams of tiled.hip consecutive work-items
// take consecutive quads, so a row is spread over several of them and joined
// by a segmented scan: of about 22 lane instructions per stored entry only 10
// decode, gather and multiply.  Here a row of a tile stays with the same four
// work-items from its first entry to its last, and their sums meet once per
// row: about 11 lane instructions, no scan, and one barrier per tile instead
// of three per 4096 entries.
//
// Layout, per tile (row block b of R rows, segment s of W columns) built on
// the device from a CSR with column-sorted rows:
//   The tile's non-empty rows are sorted by their steps (a step is four
//   entries; ties by row) and cut into slices of 16 rows; a slice has the
//   steps of its longest row.  A step of a slice is 64 entries, four
//   consecutive ones of each row: work-item 4r + q holds entry 4k + q of row
//   r in step k.  The slices of a tile go to kStreams = 8 streams, one per
//   computing wave of a workgroup, each with about the same number of
//   steps.  The steps of stream w of row block b, segment after segment, are
//   contiguous: a wave walks one array.
//   wbase u32[nblk * 8 * nseg + 1]: first step of (b, w, s).
//   A step of 16-bit values is 64 words: value << 16 | meta; one of f32
//   values 64 floats, then 64 16-bit metas.  meta: bits 0-3 four bits of the
//   row - b*R (the 4q-th from below: a row's four work-items hold all 16),
//   bits 4-14 the column - s*W (W: padding, whose x is 0; in place, it is a
//   byte offset into x of four right-hand sides), bit 15 set in the last
//   step of a slice.  So the stream is all a wave reads: no row lists, no
//   lengths.  Padding: 11-15% of a PET matrix's entries at 1024 columns,
//   19-23% at 512 (the quads: 11-20%).
//
// Work: a run is up to 64 consecutive non-empty tiles of a row block, all
// streams of them; one run per workgroup: a wave per stream, and kStagers
// waves that stage the x segments, the next tile's while one is computed
// (two LDS slots), one barrier per tile.  At the end of a slice every row's
// four sums are added (two DPP adds per right-hand side) and the row's
// accumulator in LDS is updated, by one wave per tile, so without atomics;
// the sums' order depends on the matrix alone, whatever the pass and the
// number of passes.  Partial sums, their reduction and the epilogue are
// those of tiled.hip.
//
// What bounds it: instructions (VALU 75% busy, 12 per step) and the LDS
// gather (16 bytes per entry and 4 right-hand sides; LDS 69% busy, half of
// that bank conflicts), then the barriers (a tile waits for its longest
// stream; with about 5 steps per stream and tile VALU 59%, LDS 64%).  us per launch, 4
// passes of 4 right-hand sides over 683 M entries (16-bit) and 2 passes of 8
// over 135 M (f32):
//   block streams                                        2702 / 629
//   slices, every wave stages x too                      2830 / 618
//   two staging waves, 1024 rows per tile                2630 / 516
//   the passes of a run on one XCD (its 4 MB of L2
//   serves all but the first; HBM reads of one pass)     2518 / 495
//   slices to the stream with the fewest steps, 2048
//   rows (4 right-hand sides), four staging waves        2116 / 474
//   steps taken in groups, 16-24 in flight               1589 / 430
// (us per iteration before the fifth: 4940 / 964, 4740 / 946 with the
// dealing, 4190 with 2048 rows, 4144 / 935 with four staging waves.)
// Non-temporal loads of the steps lose the L2 (2769); x of two or three tiles
// in flight instead of one, and 32-row slices of two work-items per row,
// gained nothing.
#include <algorithm>
#include <vector>

#include "tiled_common.hpp"

namespace mlem {
namespace {

constexpr uint32_t kStreams = 8;                            // waves that compute, one per stream
constexpr uint32_t kStagers = 4;                            // waves that stage x
constexpr int kSliceNT = 64 * (int)(kStreams + kStagers);
constexpr uint32_t kSliceRows = 16;
constexpr uint32_t kRowSteps = 255;            // steps of a row in a tile at most
constexpr uint32_t kSliceMaxR = 2048;          // rows per block at most
constexpr uint32_t kStreamSteps = 1u << 14;    // steps of a stream in a tile are fewer
static_assert(kSliceMaxR / kSliceRows * kRowSteps < kStreamSteps * kStreams &&
                  (kSliceMaxR / kSliceRows / kStreams + 1) * kRowSteps < kStreamSteps,
              "each slice goes to the shortest stream, so a stream exceeds the mean by one slice at most");
constexpr uint32_t kRunTiles = 64;             // tiles per run at most (one per lane)
// Steps in flight per wave, G taken together.  683 M entries in 16 bits, 4
// right-hand sides, fours, us per iteration with 8 / 12 / 16 / 24 in flight:
// 3600 / 3340 / 3216 / 3109.  (A loop of more groups than these is not
// unrolled, and then the steps are not in registers: 8544.)
constexpr int step_depth(uint32_t vt, uint32_t G) { return G == 1 ? 8 : G == 2 || vt == VAL_F32 ? 16 : 24; }
constexpr uint32_t kPadSteps = 48;         // readable past the last step

constexpr uint32_t step_bytes(uint32_t vt) { return vt == VAL_F32 ? 384u : 256u; }

// Value of a 16-bit word's upper half.
template <int VT>
__device__ __forceinline__ float word_val(uint32_t w) {
    if constexpr (VT == VAL_BF16) {
        return __uint_as_float(w & 0xffff0000u);
    } else if constexpr (is_uf16(VT)) {
        // (w >> 16) * 2^SH + bias in one instruction
        constexpr int SH = 7 + kUf16ExpBits, EMAX = (1 << kUf16ExpBits) - 1;
        uint32_t r;
        asm("v_mad_u32_u16 %0, %1, %2, %3 op_sel:[1,0,0,0]"
            : "=v"(r)
            : "v"(w), "s"(1u << SH), "v"((uint32_t)(127 - EMAX) << 23));
        return __uint_as_float(r);
    } else {
        return __half2float(__ushort_as_half((unsigned short)(w >> 16)));
    }
}

template <int CTRL>
__device__ __forceinline__ uint32_t quad_get(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ float quad_getf(float v) {
    return __uint_as_float(quad_get<CTRL>(__float_as_uint(v)));
}

// The epilogue of the rows r0 .. r0 + R - 1 from their sums: what
// blocked_reduce_kernel makes of one run's partial sums.
template <int EPI, int BC>
__device__ __forceinline__ void finish_rows(uint32_t r0, uint32_t R, const float *acc, const SliceEpi &se,
                                            const EpiArgs &ea) {
    const uint32_t nr = min(R, se.rows - r0);
    for (uint32_t i = threadIdx.x; i < nr; i += kSliceNT) {
        const ReduceIn<BC> in = reduce_load<EPI, BC>(r0 + i, se.scale, ea);
        float y[BC];
#pragma unroll
        for (int q = 0; q < BC; ++q) y[q] = acc[i * BC + q];
        reduce_epilogue<EPI, BC>(r0 + i, y, in, se.scale != nullptr, ea);
    }
}

// wl[run] = {row block, first tile (index into tiles), tiles}; tiles[i].x =
// segment.  One launch takes several passes of a batch, as
// stream_spmv_kernel does: workgroups go round the 8 XCDs, so 8 runs of one
// pass are followed by the same runs of the next, each on its XCD.
// G steps are taken together, their gathers in flight at once.  DIRECT: whole
// row blocks and their epilogue instead of partial sums (a variant of its
// own: as a branch it cost launches that do not take it 1%).
template <int W, int VT, int BC, int G, bool DIRECT>
__global__ __launch_bounds__(kSliceNT) void slice_spmv_kernel(uint32_t R, uint32_t nseg,
                                                              const uint32_t *__restrict__ wbase,
                                                              const uint4 *__restrict__ wl,
                                                              const uint32_t *__restrict__ order,
                                                              const uint4 *__restrict__ tiles,
                                                              const uint8_t *__restrict__ tdata, PassX px,
                                                              uint32_t nwg, float *__restrict__ part, SliceEpi se) {
    constexpr uint32_t SB = step_bytes(VT);
    constexpr int kDepth = step_depth(VT, G);
    static_assert(kDepth % G == 0 && 2 * kDepth <= (int)kPadSteps, "whole groups in flight, nothing read past the end");
    constexpr uint32_t XS = (W + 4) * BC;  // floats per x slot (column W holds 0)
    constexpr int XP = W * BC / 4 / (64 * kStagers);  // 16-byte pieces of an x segment per staging work-item
    static_assert(XP * 4 * 64 * kStagers == W * BC && (BC == 4 || BC == 8), "x moves in 16-byte pieces");
    extern __shared__ __attribute__((aligned(16))) float smem[];
    float *xs = smem;            // [2][XS]
    float *acc = smem + 2 * XS;  // [(R + 1) * BC]; row R: the empty rows of slices

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t grp = blockIdx.x / (8 * px.n), rem = blockIdx.x - grp * 8 * px.n;
    const uint32_t place = grp * 8 + (rem & 7u), pass = rem >> 3;
    if (place >= nwg) return;
    const uint32_t run = order[place];
    const float *__restrict__ x = px.x[pass];
    const uint4 w = wl[run];
    const uint32_t nt = w.z;
    // Lane i: the segment of tile i of the run.
    const uint32_t seg = tiles[w.y + min(lane, max(nt, 1u) - 1)].x;
    for (uint32_t i = tid; i < (R + 1) * BC; i += kSliceNT) acc[i] = 0.0f;
    if (tid < BC) {
        xs[W * BC + tid] = 0.0f;
        xs[XS + W * BC + tid] = 0.0f;
    }
    // Every wave passes nt + 1 barriers.  Barrier t: x of tile t is staged and
    // tile t - 1 is done, so that its slot may be written.
    if (wv >= kStreams) {
        const uint32_t st = tid - 64 * kStreams;
        f32x4 r[XP];
        for (uint32_t t = 0; t < nt; ++t) {
            // x is padded to whole segments: no clamping
            const f32x4 *xb = reinterpret_cast<const f32x4 *>(x + (uint64_t)__builtin_amdgcn_readlane(seg, t) * W * BC);
            f32x4 *slot = reinterpret_cast<f32x4 *>(xs + (t & 1u) * XS);
#pragma unroll
            for (int q = 0; q < XP; ++q) r[q] = xb[st + 64 * kStagers * q];
#pragma unroll
            for (int q = 0; q < XP; ++q) slot[st + 64 * kStagers * q] = r[q];
            __syncthreads();
        }
    } else {
        // Lane i: this wave's steps in tile i.
        const uint64_t wb = ((uint64_t)w.x * kStreams + wv) * nseg + seg;
        const uint32_t s0 = wbase[wb], s1 = wbase[wb + 1], cnt = s1 - s0;
        const uint32_t first = __builtin_amdgcn_readfirstlane(s0);
        const uint32_t total = nt ? __builtin_amdgcn_readlane(s1, nt - 1) - first : 0u;
        // The wave's steps, kDepth in flight (past its last step: whatever follows).
        const uint8_t *src = tdata + (uint64_t)first * SB;
        uint32_t rw[kDepth];  // 16-bit values: the words; f32: the metas
        float rv[kDepth];
        auto fetch = [&](int j, const uint8_t *at) {
            if constexpr (VT == VAL_F32) {
                rv[j] = reinterpret_cast<const float *>(at)[lane];
                rw[j] = reinterpret_cast<const uint16_t *>(at + 256)[lane];
            } else {
                rw[j] = reinterpret_cast<const uint32_t *>(at)[lane];
            }
        };
#pragma unroll
        for (int j = 0; j < kDepth; ++j) fetch(j, src + j * SB);

        const char *xw = reinterpret_cast<const char *>(xs);
        uint32_t t = 0, left = 0;  // the next tile; this wave's steps left in the current one
        auto enter = [&]() {
            __syncthreads();
            xw = reinterpret_cast<const char *>(xs + (t & 1u) * XS);
            left = __builtin_amdgcn_readlane(cnt, t);
            ++t;
        };

        float a[BC];
#pragma unroll
        for (int b = 0; b < BC; ++b) a[b] = 0.0f;
        for (uint32_t done = 0; done < total;) {
#pragma unroll
            for (int j0 = 0; j0 < kDepth; j0 += G) {
                if (done == total) break;
                while (left == 0) enter();  // ends: a tile with steps is left
                f32x4 xv[G][BC / 4];
                float v[G];
#pragma unroll
                for (int i = 0; i < G; ++i) {
                    const float *xg = reinterpret_cast<const float *>(xw + (rw[j0 + i] & 0x7ff0u) * (BC / 4));
#pragma unroll
                    for (int q = 0; q < BC / 4; ++q) xv[i][q] = *reinterpret_cast<const f32x4 *>(xg + 4 * q);
                    if constexpr (VT == VAL_F32)
                        v[i] = rv[j0 + i];
                    else
                        v[i] = word_val<VT>(rw[j0 + i]);
                }
                done += G;
                left -= G;
#pragma unroll
                for (int i = 0; i < G; ++i) {
                    const uint32_t m = rw[j0 + i];
#pragma unroll
                    for (int q = 0; q < BC / 4; ++q)
#pragma unroll
                        for (int b = 0; b < 4; ++b) a[4 * q + b] = fmaf(v[i], xv[i][q][b], a[4 * q + b]);
                    if (__builtin_amdgcn_readfirstlane(m) & 0x8000u) {  // the slice ends: its 16 rows
                        uint32_t row = (m & 15u) << (4u * (lane & 3u));
                        row |= quad_get<0xB1>(row);
                        row |= quad_get<0x4E>(row);
                        // Sums over the row's four work-items, halved between
                        // neighbours: work-item q keeps BC/4 right-hand sides.
                        const bool o1 = lane & 1u, o2 = lane & 2u;
                        float h[BC / 2];
#pragma unroll
                        for (int b = 0; b < BC / 2; ++b)
                            h[b] = (o1 ? a[b + BC / 2] : a[b]) + quad_getf<0xB1>(o1 ? a[b] : a[b + BC / 2]);
                        float *p = acc + row * BC + (o1 ? BC / 2 : 0) + (o2 ? BC / 4 : 0);
                        if constexpr (BC == 4) {
                            *p += (o2 ? h[1] : h[0]) + quad_getf<0x4E>(o2 ? h[0] : h[1]);
                        } else {
                            typedef float f32x2 __attribute__((ext_vector_type(2)));
                            f32x2 o = *reinterpret_cast<f32x2 *>(p);
                            o.x += (o2 ? h[2] : h[0]) + quad_getf<0x4E>(o2 ? h[0] : h[2]);
                            o.y += (o2 ? h[3] : h[1]) + quad_getf<0x4E>(o2 ? h[1] : h[3]);
                            *reinterpret_cast<f32x2 *>(p) = o;
                        }
#pragma unroll
                        for (int b = 0; b < BC; ++b) a[b] = 0.0f;
                    }
                }
                // The steps' registers are used up: loading into them earlier
                // would make the compiler copy them, and a copy waits.
#pragma unroll
                for (int i = 0; i < G; ++i) fetch(j0 + i, src + (kDepth + j0 + i) * SB);
            }
            src += kDepth * SB;
        }
        while (t < nt) enter();  // tiles without steps for this wave
    }
    __syncthreads();
    if constexpr (DIRECT) {
        const EpiArgs ea = se.pe.ea[pass];
        switch (se.epi) {
            case EPI_PLAIN: finish_rows<EPI_PLAIN, BC>(w.x * R, R, acc, se, ea); break;
            case EPI_RATIO: finish_rows<EPI_RATIO, BC>(w.x * R, R, acc, se, ea); break;
            default: finish_rows<EPI_UPDATE, BC>(w.x * R, R, acc, se, ea); break;
        }
    } else {
        float *pw = part + ((uint64_t)pass * nwg + run) * R * BC;
        for (uint32_t i = tid; i < R * BC; i += kSliceNT) pw[i] = acc[i];
    }
}

// ----------------------------------------------------------------- builder
// The place of row r's entries in tile (b, s), packed: its slice's steps,
// the slice's first step in the stream's part of the tile, the stream, the
// row's place in the slice.
__device__ __forceinline__ uint32_t loc_pack(uint32_t slice, uint32_t place) { return slice | (place << 25); }
__device__ __forceinline__ uint32_t loc_steps(uint32_t l) { return l & 0xffu; }
__device__ __forceinline__ uint32_t loc_first(uint32_t l) { return (l >> 8) & (kStreamSteps - 1); }
__device__ __forceinline__ uint32_t loc_stream(uint32_t l) { return (l >> 22) & 7u; }
__device__ __forceinline__ uint32_t loc_place(uint32_t l) { return (l >> 25) & 15u; }

__device__ __forceinline__ void wave_lds_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

// A wave per tile: a counting sort of its rows by steps (longest first,
// stable), their slices and streams.  rowloc as above for rows with entries;
// wsteps[(b * 8 + w) * nseg + s] = steps of stream w; *most = the most of
// any; bit 16 of *bad: a row with more steps than the layout holds.
__global__ __launch_bounds__(kWG) void slice_rows_kernel(const uint32_t *__restrict__ cnt, uint32_t rows, uint32_t R,
                                                         uint32_t nseg, uint64_t ntiles,
                                                         uint32_t *__restrict__ rowloc,
                                                         uint32_t *__restrict__ wsteps, uint32_t *__restrict__ most,
                                                         uint32_t *__restrict__ bad) {
    __shared__ uint32_t s_hist[kWG / 64][kRowSteps + 1];
    __shared__ uint32_t s_slice[kWG / 64][kSliceMaxR / kSliceRows];
    const uint32_t wv = threadIdx.x / 64, lane = threadIdx.x % 64;
    const uint64_t t = blockIdx.x * (uint64_t)(kWG / 64) + wv;
    if (t >= ntiles) return;  // whole waves, no barriers below
    const uint32_t b = (uint32_t)(t / nseg), s = (uint32_t)(t % nseg);
    const uint64_t r0 = (uint64_t)b * R;
    const uint32_t nr = (uint32_t)std::min<uint64_t>(R, rows - r0);
    uint32_t *h = s_hist[wv], *sl = s_slice[wv];  // bin 255 - steps: longest first
#pragma unroll
    for (int i = 0; i < 4; ++i) h[lane + 64 * i] = 0;
    wave_lds_fence();
    auto steps_of = [&](uint32_t i) { return i < nr ? (cnt[(r0 + i) * nseg + s] + 3u) / 4u : 0u; };
    bool over = false;
    for (uint32_t i0 = 0; i0 < nr; i0 += 64) {
        const uint32_t st = steps_of(i0 + lane);
        over = over || st > kRowSteps;
        if (st) atomicAdd(h + (kRowSteps - min(st, kRowSteps)), 1u);
    }
    wave_lds_fence();
    // Bin starts: lane l scans bins 4l .. 4l + 3.
    uint32_t c[4], sum = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        c[i] = h[4 * lane + i];
        sum += c[i];
    }
    uint32_t incl = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t u = __shfl_up(incl, o);
        if (lane >= (uint32_t)o) incl += u;
    }
    const uint32_t M = __shfl(incl, 63), nsl = (M + kSliceRows - 1) / kSliceRows;
    uint32_t start = incl - sum;
    wave_lds_fence();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        h[4 * lane + i] = start;
        start += c[i];
    }
    wave_lds_fence();
    for (uint32_t i = lane; i < nsl; i += 64) {  // a slice's steps: those of its first row
        uint32_t lo = 0, hi = kRowSteps + 1;     // the last bin that starts at or before it
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) / 2;
            if (h[mid] <= i * kSliceRows)
                lo = mid;
            else
                hi = mid;
        }
        sl[i] = kRowSteps - lo;
    }
    wave_lds_fence();
    // Longest first, each to the stream with the fewest steps so far (a tile
    // ends when its longest stream does: 9-27% above the mean this way,
    // 13-46% when dealt in turn).  Lane w counts for stream w; ties go to
    // another stream in every segment.
    uint32_t n = 0;
    for (uint32_t i = 0; i < nsl; ++i) {
        const uint32_t w8 = lane & (kStreams - 1), key0 = (n << 3) | ((lane + s) & (kStreams - 1));
        uint32_t key = key0;
#pragma unroll
        for (uint32_t o = 1; o < kStreams; o <<= 1) key = min(key, __shfl_xor(key, o));
        if (key == key0) {
            const uint32_t st = sl[i];
            if (lane < kStreams) sl[i] = st | (n << 8) | (w8 << 22);
            n += st;
        }
    }
    if (lane < kStreams) {
        wsteps[((uint64_t)b * kStreams + lane) * nseg + s] = n;
        if (n) atomicMax(most, n);
    }
    wave_lds_fence();
    for (uint32_t i0 = 0; i0 < nr; i0 += 64) {
        const uint32_t i = i0 + lane, st = min(steps_of(i), kRowSteps), bin = kRowSteps - st;
        uint64_t same = __ballot(st != 0);
#pragma unroll
        for (int bit = 0; bit < 8; ++bit) {
            const uint64_t m = __ballot((bin >> bit) & 1u);
            same &= ((bin >> bit) & 1u) ? m : ~m;
        }
        const uint32_t rank = __popcll(same & ((1ull << lane) - 1ull)), at = h[bin];
        wave_lds_fence();
        if (st && rank == 0) h[bin] = at + __popcll(same);
        wave_lds_fence();
        if (st) {
            const uint32_t pos = at + rank;
            rowloc[(r0 + i) * nseg + s] = loc_pack(sl[pos / kSliceRows], pos % kSliceRows);
        }
    }
    if (over) atomicOr(bad, 16u);
}

// Every entry's meta is that of an empty row of a slice (row R, padding
// column W), every value 0, until the rows are placed.
__global__ __launch_bounds__(kWG) void slice_clear_kernel(uint8_t *__restrict__ tdata, uint64_t first, uint64_t steps,
                                                          bool f32, uint32_t R, uint32_t W) {
    const uint64_t n = steps * 64, stride = (uint64_t)gridDim.x * kWG;
    for (uint64_t i = blockIdx.x * (uint64_t)kWG + threadIdx.x; i < n; i += stride) {
        const uint32_t lane = (uint32_t)(i & 63u), meta = ((R >> (4 * (lane & 3u))) & 15u) | (W << 4);
        const uint64_t st = first + i / 64;
        if (f32) {
            reinterpret_cast<float *>(tdata + st * 384)[lane] = 0.0f;
            reinterpret_cast<uint16_t *>(tdata + st * 384 + 256)[lane] = (uint16_t)meta;
        } else {
            reinterpret_cast<uint32_t *>(tdata + st * 256)[lane] = meta;
        }
    }
}

// A wave per row: every entry into its step, and the padding up to its
// slice's steps behind the last one.  wbase: of the row blocks of `rows`.
__global__ __launch_bounds__(kWG) void slice_scatter_kernel(const uint64_t *__restrict__ rowptr,
                                                            const uint32_t *__restrict__ col,
                                                            const float *__restrict__ val,
                                                            const uint16_t *__restrict__ qval, uint32_t rows,
                                                            uint32_t R, uint32_t nseg, uint32_t wshift,
                                                            const uint32_t *__restrict__ rowloc,
                                                            const uint32_t *__restrict__ wbase,
                                                            uint8_t *__restrict__ tdata) {
    const uint32_t row = blockIdx.x * (kWG / 64) + threadIdx.x / 64, lane = threadIdx.x % 64;
    if (row >= rows) return;
    const uint32_t b = row / R, i = row % R, W = 1u << wshift;
    const uint64_t rs = rowptr[row], re = rowptr[row + 1];
    SegWalk w{rs, 0u};
    for (uint64_t k0 = rs; k0 < re; k0 += 64) {
        const uint64_t k = k0 + lane;
        const uint32_t c = k < re ? col[k] : 0u, next = k0 + 64 < re ? col[k0 + 64] : 0u;
        bool last, unsorted;
        const uint64_t head = w.step(rs, re, k0, lane, c, next, wshift, &last, &unsorted);
        if (k >= re) continue;
        const uint32_t s = c >> wshift, loc = rowloc[(uint64_t)row * nseg + s], S = loc_steps(loc);
        const uint64_t at =
            (uint64_t)wbase[((uint64_t)b * kStreams + loc_stream(loc)) * nseg + s] + loc_first(loc);
        auto put = [&](uint32_t j, uint32_t cl, uint64_t from, bool pad) {
            const uint32_t st = j / 4, q = j % 4, l = loc_place(loc) * 4 + q;
            const uint32_t meta = (st + 1 == S ? 0x8000u : 0u) | ((i >> (4 * q)) & 15u) | (cl << 4);
            if (qval) {
                reinterpret_cast<uint32_t *>(tdata + (at + st) * 256)[l] =
                    (pad ? 0u : (uint32_t)qval[from] << 16) | meta;
            } else {
                reinterpret_cast<float *>(tdata + (at + st) * 384)[l] = pad ? 0.0f : val[from];
                reinterpret_cast<uint16_t *>(tdata + (at + st) * 384 + 256)[l] = (uint16_t)meta;
            }
        };
        const uint32_t j = (uint32_t)(k - head);
        put(j, c & (W - 1), k, false);
        if (last)
            for (uint32_t p = j + 1; p < 4 * S; ++p) put(p, W, 0, true);
    }
}

template <int W, int VT, int BC, int G>
hipError_t launch_slices(const TilePlan &p, const TiledMatrix &tm, const TileWork &wk, const PassX &x, float *part,
                         const SliceEpi &se, hipStream_t s) {
    const dim3 grid((wk.nwg + 7) / 8 * 8 * x.n);
    if (se.direct)
        hipLaunchKernelGGL((slice_spmv_kernel<W, VT, BC, G, true>), grid, dim3(kSliceNT), slice_lds_bytes(p, BC), s, p.R,
                           p.nseg, tm.wbase, wk.wl, wk.order, wk.tiles, tm.tdata, x, wk.nwg, part, se);
    else
        hipLaunchKernelGGL((slice_spmv_kernel<W, VT, BC, G, false>), grid, dim3(kSliceNT), slice_lds_bytes(p, BC), s,
                           p.R, p.nseg, tm.wbase, wk.wl, wk.order, wk.tiles, tm.tdata, x, wk.nwg, part, se);
    return hipGetLastError();
}

template <int VT>
hipError_t launch_slices_vt(const TilePlan &p, const TiledMatrix &tm, const TileWork &wk, const PassX &x, float *part,
                            uint32_t BC, const SliceEpi &se, hipStream_t s) {
    if (BC == 4 && p.W == 1024) {
        switch (p.group) {
            case 1: return launch_slices<1024, VT, 4, 1>(p, tm, wk, x, part, se, s);
            case 2: return launch_slices<1024, VT, 4, 2>(p, tm, wk, x, part, se, s);
            case 4: return launch_slices<1024, VT, 4, 4>(p, tm, wk, x, part, se, s);
        }
    } else if (BC == 4 && p.W == 512) {
        if (p.group == 1) return launch_slices<512, VT, 4, 1>(p, tm, wk, x, part, se, s);
        if (p.group == 2) return launch_slices<512, VT, 4, 2>(p, tm, wk, x, part, se, s);
    } else if (BC == 8 && p.W == 512) {
        if (p.group == 1) return launch_slices<512, VT, 8, 1>(p, tm, wk, x, part, se, s);
        if (p.group == 2) return launch_slices<512, VT, 8, 2>(p, tm, wk, x, part, se, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace

size_t slice_lds_bytes(const TilePlan &p, uint32_t BC) { return (2 * ((size_t)p.W + 4) + p.R + 1) * BC * 4; }

// Two workgroups' rows fit a CU's LDS, with 8 right-hand sides (512 columns)
// up to 1024 rows: with 2048 one is left, and the block streams win.
bool slices_possible(const TilePlan &p) { return p.quad && p.R <= (p.W == 512 ? kSliceMaxR / 2 : kSliceMaxR) && p.ntiles > 0; }

// A stream's part of a tile is padded to whole groups of steps: up to four
// (two of 512 columns, whose x of 8 right-hand sides takes the registers of
// four), as long as that adds at most an eighth.  us per iteration in single
// steps / pairs / fours, 8 steps in flight: 16 slots of 4 over 683 M entries
// 4242 / 3728 / 3600; 13 slots of 8 over 135 M, about 5 steps per part,
// 935 / 870 (+9% padding) / 1262 (+28%).
bool slice_prefix(uint32_t W, std::vector<uint32_t> *w, uint64_t *steps, uint32_t *group) {
    w->back() = 0;  // becomes the end
    uint64_t sum[3] = {};
    for (uint32_t n : *w)
        for (uint32_t i = 0; i < 3; ++i) sum[i] += (n + (1u << i) - 1) >> i << i;
    uint32_t i = W == 512 ? 1u : 2u;
    while (i && sum[i] * 8 > sum[0] * 9) --i;
    *group = 1u << i;
    uint64_t run = 0;
    for (uint32_t &v : *w) {
        const uint32_t n = (v + (1u << i) - 1) >> i << i;
        v = (uint32_t)run;
        run += n;
    }
    *steps = run;
    return run < 0xffffff00ull;
}

size_t slice_stream_count(const TilePlan &p) { return (size_t)p.nblk * kStreams * p.nseg; }

// Slices unless they store over a quarter more entries than the quads (a few
// long rows among short ones), or one tile holds so large a share of a small
// matrix that whole tiles per workgroup leave the chip idle (a run of a
// block stream may hold part of a tile).  Within the rule they were the
// faster on every matrix tried; us per iteration of 8 slots in 16-bit
// values, 4 / 8 right-hand sides per pass, block streams -> slices:
//   20000 x 2000, 200 a row, uniform     73 ->  34 /  53 ->  39
//   300000 x 300000, 60 a row, a band   151 ->  91 / 138 ->  91
//   100000 x 100000, 200 a row, uniform 239 -> 217 / 263 -> 234
//   200000 x 200000, 40 a row, uniform  556 -> 400 / 808 -> 403
bool slices_suit(const TilePlan &quads, uint64_t steps, uint32_t most) {
    const uint64_t per_run = std::max<uint64_t>(1, steps / 2048);
    return steps * 64 * 4 <= (quads.cap - 8) * 5 && (most <= 256 || most <= per_run);
}

// A row block summed by one workgroup needs no partial sums and no reduction
// (two launches in one), but its tiles are one chain: up to 16 segments, and
// as many entries per block as there are other blocks to run beside it.
// 4 right-hand sides per pass, 16 bits, us per iteration (FP and BP, FP's
// blocks of 512 rows as one run or not), one pass / four / eight:
//   64 x 64, 81 blocks of 24 Ki entries      32.7 -> 30.4 / 43.4 -> 37.1 / 55.8 -> 49.5
//   40 x 40, 22 blocks of 15 Ki              24.2 -> 21.3 / 25.1 -> 22.2 / 26.7 -> 23.2
//   96 x 96, 156 blocks of 36 Ki             47.0 -> 45.6 / 79.5 -> 70.1 /  129 ->  108
//   128 x 128, 324 blocks of 48 Ki           75.5 -> 72.3 /  156 ->  140 /  310 ->  272
//   128 x 128, 88 blocks of 48 Ki            43.0 -> 48.3 /   73 ->   65 /  119 ->  101
// With 8 right-hand sides 24 Ki entries gain only in several passes (one
// 40.1 -> 41.4, four 70.3 -> 57.7) and 10 Ki in one (977 blocks: 113 -> 94).
bool slices_direct(uint32_t cols, uint32_t W, uint32_t R, uint64_t rows, uint64_t nnz, uint32_t BC) {
    const uint64_t blocks = (rows + R - 1) / R;
    const uint64_t most = BC == 8 ? 12288 : std::min<uint64_t>(65536, std::max<uint64_t>(16384, 400 * blocks));
    return cols <= 16ull * W && nnz <= blocks * most;
}

size_t slice_data_bytes(const TilePlan &p) {
    return align256(4 * (slice_stream_count(p) + 1)) + align256((p.steps + kPadSteps) * step_bytes(p.vt));
}

void slice_view(const TilePlan &p, void *mem, TiledMatrix *t) {
    char *c = static_cast<char *>(mem);
    t->wbase = reinterpret_cast<uint32_t *>(c);
    t->tdata = reinterpret_cast<uint8_t *>(c + align256(4 * (slice_stream_count(p) + 1)));
}

hipError_t launch_slice_count(const TilePlan &p, const uint32_t *cnt, uint32_t *rowloc, uint32_t *wsteps,
                              uint32_t *flags, uint32_t *flags_host, hipStream_t s) {
    hipError_t e;
    if ((e = hipMemsetAsync(flags, 0, 8, s)) != hipSuccess) return e;
    hipLaunchKernelGGL(slice_rows_kernel, dim3(blocks_for(p.ntiles, kWG / 64)), dim3(kWG), 0, s, cnt, p.rows, p.R,
                       p.nseg, p.ntiles, rowloc, wsteps, flags + 1, flags);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = hipMemcpyAsync(flags_host, flags, 8, hipMemcpyDeviceToHost, s)) != hipSuccess) return e;
    return hipStreamSynchronize(s);
}

hipError_t launch_slice_clear(const TilePlan &p, const TiledMatrix &tm, hipStream_t s) {
    if (!p.steps) return hipSuccess;
    const uint64_t blocks = std::min<uint64_t>((p.steps * 64 + kWG - 1) / kWG, 16384);
    hipLaunchKernelGGL(slice_clear_kernel, dim3((uint32_t)blocks), dim3(kWG), 0, s, tm.tdata, (uint64_t)0, p.steps,
                       p.vt == VAL_F32, p.R, p.W);
    return hipGetLastError();
}

hipError_t launch_slice_scatter(const TilePlan &p, const uint64_t *rowptr, const uint32_t *col, const float *val,
                                const uint16_t *qval, const uint32_t *rowloc, const uint32_t *wbase, uint8_t *tdata,
                                hipStream_t s) {
    if (!p.rows) return hipSuccess;
    uint32_t wshift = 0;
    while ((1u << wshift) < p.W) ++wshift;
    hipLaunchKernelGGL(slice_scatter_kernel, dim3(blocks_for(p.rows, kWG / 64)), dim3(kWG), 0, s, rowptr, col, val,
                       qval, p.rows, p.R, p.nseg, wshift, rowloc, wbase, tdata);
    return hipGetLastError();
}

TileWorkList slice_work_list(const TilePlan &p, const uint32_t *wbase, uint32_t target_wgs) {
    TileWorkList L;
    const uint64_t per_run = std::max<uint64_t>(1, (p.steps + std::max(1u, target_wgs) - 1) / std::max(1u, target_wgs));
    L.wl_first.assign((size_t)p.nblk + 1, 0);
    std::vector<uint64_t> n;  // steps of each non-empty tile of the block
    for (uint32_t b = 0; b < p.nblk; ++b) {
        L.wl_first[b] = L.nwg;
        const uint32_t first = L.ntl;
        uint64_t left = 0;
        n.clear();
        for (uint32_t sg = 0; sg < p.nseg; ++sg) {
            uint64_t st = 0;
            for (uint32_t w = 0; w < kStreams; ++w) {
                const uint32_t *q = wbase + ((size_t)b * kStreams + w) * p.nseg + sg;
                st += q[1] - q[0];
            }
            if (!st) continue;
            L.tiles.insert(L.tiles.end(), {sg, 0u, 0u, 0u});
            ++L.ntl;
            n.push_back(st);
            left += st;
        }
        if (n.empty() && target_wgs == 1) {  // one run per block: an empty one too (launch_tiled_spmv)
            L.wl.insert(L.wl.end(), {b, 0u, 0u, 0u});
            ++L.nwg;
        }
        // Runs of nearly equal steps over the block's tiles.
        uint64_t runs = (left + per_run - 1) / per_run;
        for (size_t i = 0; i < n.size();) {
            const uint64_t want = (left + runs - 1) / runs;
            const size_t i0 = i;
            uint64_t got = 0;
            while (i < n.size() && i - i0 < kRunTiles && (got == 0 || got + n[i] / 2 <= want)) got += n[i++];
            L.wl.insert(L.wl.end(), {b, first + (uint32_t)i0, (uint32_t)(i - i0), 0u});
            ++L.nwg;
            left -= got;
            runs = runs > 1 ? runs - 1 : 1;
        }
    }
    if (L.ntl == 0) {  // no entries at all: no runs
        L.wl.clear();
        L.nwg = 0;
        std::fill(L.wl_first.begin(), L.wl_first.end(), 0u);
    }
    L.wl_first[p.nblk] = L.nwg;
    // Launch order: by the column segment each run starts in, as for the
    // block streams.
    L.order.resize(L.nwg);
    for (uint32_t r = 0; r < L.nwg; ++r) L.order[r] = r;
    auto first_seg = [&](uint32_t r) { return L.tiles[4 * (size_t)L.wl[4 * (size_t)r + 1]]; };
    std::stable_sort(L.order.begin(), L.order.end(),
                     [&](uint32_t a, uint32_t b) { return first_seg(a) < first_seg(b); });
    return L;
}

hipError_t launch_slice_spmv(const TilePlan &p, const TiledMatrix &tm, const TileWork &wk, const PassX &x, float *part,
                             uint32_t BC, const SliceEpi &se, hipStream_t s) {
    switch (p.vt) {
        case VAL_F32: return launch_slices_vt<VAL_F32>(p, tm, wk, x, part, BC, se, s);
        case VAL_BF16: return launch_slices_vt<VAL_BF16>(p, tm, wk, x, part, BC, se, s);
        case VAL_UF16: return launch_slices_vt<VAL_UF16>(p, tm, wk, x, part, BC, se, s);
        default: return launch_slices_vt<VAL_F16>(p, tm, wk, x, part, BC, se, s);
    }
}

}  // namespace mlem
