// Device helpers shared by the blocked kernels' files (tiled.hip, slices.hip).
#pragma once

#include <hip/hip_fp16.h>

#include "launch.hpp"

namespace mlem {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));

// Streamed matrix data is read once per pass: non-temporal loads.
template <typename T>
__device__ __forceinline__ T ldnt(const T *p) {
    return __builtin_nontemporal_load(p);
}

inline uint32_t blocks_for(uint64_t n, uint32_t per) { return (uint32_t)((n + per - 1) / per); }
constexpr size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

// A wave walking the entries of one row, 64 at a time, in rows sorted by
// column: where the run of entries in the same segment that each entry
// belongs to started (`head`, an entry index) and whether it ends there.
struct SegWalk {
    uint64_t head;    // start of the run that the last step ended in
    uint32_t prev_c;  // column of the last step's last entry
    // Entries k0..k0+63 of the row [rs, re) with column c in lane k - k0
    // (lanes past re: any); next_c: the column of entry k0 + 64 where it is
    // in the row.  Returns the head of this lane's run.
    __device__ __forceinline__ uint64_t step(uint64_t rs, uint64_t re, uint64_t k0, uint32_t lane, uint32_t c,
                                             uint32_t next_c, uint32_t wshift, bool *last, bool *unsorted) {
        const uint64_t k = k0 + lane;
        const bool in = k < re;
        uint32_t p = __shfl_up(c, 1), n = __shfl_down(c, 1);
        if (lane == 0) p = prev_c;
        if (lane == 63) n = next_c;
        const uint32_t seg = c >> wshift;
        const bool starts = in && (k == rs || (p >> wshift) != seg);
        *unsorted = in && k != rs && c < p;
        *last = in && (k + 1 == re || (n >> wshift) != seg);
        const uint64_t m = __ballot(starts), below = m & (~0ull >> (63u - lane));
        const uint64_t mine = below ? k0 + (63u - __clzll(below)) : head;
        if (m) head = k0 + (63u - __clzll(m));
        prev_c = __shfl(c, 63);
        return mine;
    }
};

// The epilogue of row r from its sum y over the block's workgroups: the
// row's value scale (16-bit values), then the ratio, the update or the plain
// sum.  Vectors are [rows][BC].  Its inputs are read by reduce_load before
// the partials are summed, so that their memory round trip overlaps the
// sum's instead of following it (a small matrix's reduction is a chain of
// dependent round trips).
template <int BC>
struct ReduceIn {
    float sc;     // the row's value scale (1 without scales)
    float a[BC];  // RATIO: the counts; UPDATE: the image values
    float n;      // UPDATE: the sensitivity
    bool act[BC]; // UPDATE: the right-hand side is active
};

template <int EPI, int BC>
__device__ __forceinline__ ReduceIn<BC> reduce_load(uint32_t r, const float *__restrict__ scale, const EpiArgs &ea) {
    ReduceIn<BC> in;
    in.sc = scale ? scale[r] : 1.0f;
    in.n = 0.0f;
#pragma unroll
    for (int q = 0; q < BC; ++q) {
        const uint64_t k = (uint64_t)r * BC + q;
        in.a[q] = 0.0f;
        in.act[q] = true;
        if constexpr (EPI == EPI_RATIO) in.a[q] = (float)ea.g[k];
        if constexpr (EPI == EPI_UPDATE) {
            in.a[q] = ea.f[k];
            in.act[q] = !ea.active || ea.active[q];
        }
    }
    if constexpr (EPI == EPI_UPDATE) in.n = ea.norm[r];
    return in;
}

template <int EPI, int BC>
__device__ __forceinline__ void reduce_epilogue(uint32_t r, const float (&y)[BC], const ReduceIn<BC> &in,
                                                bool scaled, const EpiArgs &ea) {
#pragma unroll
    for (int q = 0; q < BC; ++q) {
        const uint64_t k = (uint64_t)r * BC + q;
        const float yq = scaled ? y[q] * in.sc : y[q];
        if constexpr (EPI == EPI_PLAIN) {
            ea.out[k] = yq;
        } else if constexpr (EPI == EPI_RATIO) {
            // 16-bit values: the back projection's tiles hold the same codes
            // without the row scales, so the ratio g / (scale * sum) goes on
            // multiplied by the scale, that is g / sum.
            ea.out[k] = (y[q] != 0.0f) ? in.a[q] / y[q] : 0.0f;
        } else {
            const float v = in.a[q] * yq;
            if (in.act[q]) ea.f[k] = (in.n == 0.0f) ? v : v / in.n;
        }
    }
}

}  // namespace
}  // namespace mlem
