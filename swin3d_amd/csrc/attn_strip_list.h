// The strip list of the attention forward's strip kernel (attn_strip_fwd.hip), which the sweep's list builder may make along with
// its own (attn_sweep.hip).
#pragma once

#include "s3d_common.h"

namespace s3d {
namespace tile {

constexpr int kStrip = 16;               // voxels of a strip
__host__ __device__ __forceinline__ int strips_of(int n) { return (n + kStrip - 1) / kStrip; }

// A window of n voxels is ceil(n / 16) strips of equal size.  A strip: first sorted position of the window, n, and which of
// the window's strips it is, in 22, 22 and 20 bits.
constexpr int kPosBits = 22;
struct StripList {
    const int32_t *total;
    const uint64_t *strips;
};
inline size_t strip_list_most(int64_t N, int64_t W) { return static_cast<size_t>(N > 0 ? N : 0) / kStrip + static_cast<size_t>(W > 0 ? W : 0); }

#ifdef __HIPCC__
// By one workgroup: the strips of the largest windows first, bins of one size by a counting sort in LDS.  (A strip's result does
// not depend on its place, so the order inside a bin may be any.)  place_strips leaves the places of the bins in `at`, from which
// the windows then draw theirs.
constexpr int kSizeBins = 256;
__device__ __forceinline__ int size_bin(int n) { return kSizeBins - min(n, kSizeBins); }
template <int kThreads>
__device__ __forceinline__ void place_strips(const int32_t *__restrict__ w_sizes, int W, int32_t *__restrict__ total, int *at)
{
    const int t = threadIdx.x;
    for (int b = t; b < kSizeBins; b += kThreads) at[b] = 0;
    __syncthreads();
    for (int w = t; w < W; w += kThreads) {
        const int n = w_sizes[w];
        if (n > 0) atomicAdd(&at[size_bin(n)], strips_of(n));
    }
    __syncthreads();
    if (t < 64) {
        int own[kSizeBins / 64], sum = 0;
#pragma unroll
        for (int e = 0; e < kSizeBins / 64; ++e) sum += own[e] = at[t * (kSizeBins / 64) + e];
        int incl = sum;
        for (int off = 1; off < 64; off <<= 1) {
            const int up = __shfl_up(incl, off);
            if (t >= off) incl += up;
        }
        int run = incl - sum;
#pragma unroll
        for (int e = 0; e < kSizeBins / 64; ++e) {
            at[t * (kSizeBins / 64) + e] = run;
            run += own[e];
        }
        if (t == 63) total[0] = incl;
    }
    __syncthreads();
}
template <int kThreads>
__device__ __forceinline__ void build_strip_list(const int32_t *__restrict__ w_sizes, const int32_t *__restrict__ w2n, int W,
                                                 int32_t *__restrict__ total, uint64_t *__restrict__ strips)
{
    __shared__ int at[kSizeBins];
    place_strips<kThreads>(w_sizes, W, total, at);
    for (int w = threadIdx.x; w < W; w += kThreads) {
        const int n = w_sizes[w];
        if (n <= 0) continue;
        const int count = strips_of(n), first = atomicAdd(&at[size_bin(n)], count);
        const uint64_t window = static_cast<uint64_t>(static_cast<uint32_t>(w2n[w])) | static_cast<uint64_t>(n) << kPosBits;
        for (int q = 0; q < count; ++q) strips[first + q] = window | static_cast<uint64_t>(q) << (2 * kPosBits);
    }
}
#endif

}  // namespace tile
}  // namespace s3d
