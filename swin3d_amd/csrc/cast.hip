// Several fp32 arrays to fp16 in one launch: the casts of parameters that autocast makes are a launch and some ten
// microseconds of host time each otherwise, for tens of kilobytes.
#include "s3d_common.h"

namespace s3d {
namespace {

constexpr int kCastThreads = 256, kCastArrays = 16;

struct CastArgs {
    const float *from[kCastArrays];
    _Float16 *to[kCastArrays];
    int64_t count[kCastArrays];
};

typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// blockIdx.y: the array; four neighbouring elements a thread and step, where both addresses allow it
__global__ __launch_bounds__(kCastThreads) void cast_half_kernel(CastArgs a)
{
    const float *from = a.from[0];
    _Float16 *to = a.to[0];
    int64_t count = a.count[0];
#pragma unroll
    for (int i = 1; i < kCastArrays; ++i) {
        const bool here = static_cast<int>(blockIdx.y) == i;
        from = here ? a.from[i] : from;
        to = here ? a.to[i] : to;
        count = here ? a.count[i] : count;
    }
    const int64_t first = static_cast<int64_t>(blockIdx.x) * kCastThreads + threadIdx.x, step = static_cast<int64_t>(gridDim.x) * kCastThreads;
    const int64_t fours = reinterpret_cast<uintptr_t>(from) % 16 == 0 && reinterpret_cast<uintptr_t>(to) % 8 == 0 ? count / 4 : 0;
    for (int64_t i = first; i < fours; i += step)
        reinterpret_cast<f16x4 *>(to)[i] = __builtin_convertvector(reinterpret_cast<const f32x4 *>(from)[i], f16x4);
    for (int64_t i = 4 * fours + first; i < count; i += step) to[i] = static_cast<_Float16>(from[i]);
}

constexpr int kMostCopies = 24, kFlat = 4096, kSquare = 64;

struct HalfCopies {
    const float *from[kMostCopies];
    s3d_half_copy of[kMostCopies];
    int first[kMostCopies];        // the first workgroup of each
    int num;
    _Float16 *half;
    float *same;
};

// Parameters of a block in fp16: a workgroup takes 4096 elements of an array, or 64 x 64 of one that is wanted transposed as
// well, which it turns in LDS.  A block's seventeen arrays are 2 to 9 MB; one by one they were some thirty launches (the
// products with the scale of q, casts, concatenations and, in the backward, transposing copies) of 4 us each and 0.1 ms of
// the host's time.
__global__ __launch_bounds__(kCastThreads) void half_copies_kernel(HalfCopies a)
{
    __shared__ _Float16 turned[kSquare * (kSquare + 4)];
    // (a lane looks at an array's first workgroup: one by one they were a chain of sixteen loads)
    const int lane = threadIdx.x & 63;
    const int at = __popcll(__ballot(lane < a.num && static_cast<int>(blockIdx.x) >= a.first[min(lane, kMostCopies - 1)])) - 1;
    const s3d_half_copy &c = a.of[at];
    const float *from = a.from[at];
    const float scale = c.scale;
    const int tile = static_cast<int>(blockIdx.x) - a.first[at], tid = threadIdx.x;
    _Float16 *to = c.to < 0 ? nullptr : a.half + c.to;
    float *same = c.same < 0 ? nullptr : a.same + c.same;
    if (c.transposed < 0) {
        const int64_t begin = static_cast<int64_t>(tile) * kFlat, end = min(begin + kFlat, c.rows * c.cols), scaled = c.scaled_rows * c.cols;
        const bool whole = reinterpret_cast<uintptr_t>(from) % 16 == 0 && (!to || c.to % 4 == 0) && (!same || c.same % 4 == 0);
        const int64_t fours = whole ? (end - begin) / 4 : 0;
        for (int64_t i = begin + 4 * tid; i < begin + 4 * fours; i += 4 * kCastThreads) {
            f32x4 v = *reinterpret_cast<const f32x4 *>(from + i);
            if (same) *reinterpret_cast<f32x4 *>(same + i) = v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = i + e < scaled ? v[e] * scale : v[e];
            if (to) *reinterpret_cast<f16x4 *>(to + i) = __builtin_convertvector(v, f16x4);
        }
        for (int64_t i = begin + 4 * fours + tid; i < end; i += kCastThreads) {
            const float v = from[i];
            if (same) same[i] = v;
            if (to) to[i] = static_cast<_Float16>(i < scaled ? v * scale : v);
        }
        return;
    }
    // (rows and cols multiples of 8)
    constexpr int kPitch = kSquare + 4;
    const int across = static_cast<int>((c.cols + kSquare - 1) / kSquare), part = 4 * (tid & 15);
    const int64_t row0 = static_cast<int64_t>(tile / across) * kSquare, col0 = static_cast<int64_t>(tile % across) * kSquare;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = tid / 16 + 16 * i;
        if (row0 + r >= c.rows || col0 + part >= c.cols) continue;
        const int64_t e = (row0 + r) * c.cols + col0 + part;
        f32x4 v = *reinterpret_cast<const f32x4 *>(from + e);
        if (same) *reinterpret_cast<f32x4 *>(same + e) = v;
        if (row0 + r < c.scaled_rows) v *= scale;
        const f16x4 h = __builtin_convertvector(v, f16x4);
        if (to) *reinterpret_cast<f16x4 *>(to + e) = h;
#pragma unroll
        for (int k = 0; k < 4; ++k) turned[(part + k) * kPitch + r] = h[k];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int col = tid / 16 + 16 * i;
        if (col0 + col >= c.cols || row0 + part >= c.rows) continue;
        *reinterpret_cast<f16x4 *>(a.half + c.transposed + (col0 + col) * c.rows + row0 + part) = *reinterpret_cast<const f16x4 *>(turned + col * kPitch + part);
    }
}

// out = x + residual: widened first, which is exact, then one fp32 sum.  (Two launches, or at a tenth of the rate a sum of two
// types, in the framework: 9.7 + 6.2 us for 49,682 x 96.)
__global__ __launch_bounds__(kCastThreads) void add_half_kernel(const f32x4 *__restrict__ x, const f16x4 *__restrict__ residual,
                                                                f32x4 *__restrict__ out, int64_t fours)
{
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kCastThreads + threadIdx.x; i < fours; i += static_cast<int64_t>(gridDim.x) * kCastThreads)
        out[i] = x[i] + __builtin_convertvector(residual[i], f32x4);
}

}  // namespace
}  // namespace s3d

extern "C" __attribute__((visibility("default"))) int s3d_cast_half(const float *const *from, void *const *to, const int64_t *counts,
                                                                    int32_t num, void *stream)
{
    using namespace s3d;
    if (num < 0 || num > kCastArrays) return fail(S3D_ERR_BAD_SHAPE, "s3d_cast_half: %d arrays (0..%d)", num, kCastArrays);
    if (num > 0 && (!from || !to || !counts)) return fail(S3D_ERR_NULL_POINTER, "s3d_cast_half: null array of addresses");
    CastArgs a{};
    int64_t most = 0;
    for (int i = 0; i < num; ++i) {
        if (counts[i] < 0) return fail(S3D_ERR_BAD_SHAPE, "s3d_cast_half: %lld elements", (long long)counts[i]);
        if (counts[i] > 0 && (!from[i] || !to[i])) return fail(S3D_ERR_NULL_POINTER, "s3d_cast_half: null device pointer");
        a.from[i] = from[i];
        a.to[i] = static_cast<_Float16 *>(to[i]);
        a.count[i] = counts[i];
        most = counts[i] > most ? counts[i] : most;
    }
    if (most == 0) return S3D_OK;
    const int64_t blocks = ceil_div(ceil_div(most, 4), kCastThreads);
    hipLaunchKernelGGL(cast_half_kernel, dim3(static_cast<unsigned>(blocks < 512 ? blocks : 512), static_cast<unsigned>(num)), dim3(kCastThreads), 0,
                       static_cast<hipStream_t>(stream), a);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

extern "C" __attribute__((visibility("default"))) int s3d_half_copies(const float *const *from, const s3d_half_copy *copies, int32_t num,
                                                                      void *half, float *same, void *stream)
{
    using namespace s3d;
    if (num < 0 || num > kMostCopies) return fail(S3D_ERR_BAD_SHAPE, "s3d_half_copies: %d arrays (0..%d)", num, kMostCopies);
    if (num > 0 && (!from || !copies)) return fail(S3D_ERR_NULL_POINTER, "s3d_half_copies: null array");
    HalfCopies a{};
    int64_t blocks = 0;
    for (int i = 0; i < num; ++i) {
        const s3d_half_copy &c = copies[i];
        if (c.rows < 1 || c.cols < 1 || c.rows > 0x7fffffff || c.cols > 0x7fffffff || c.rows * c.cols > (int64_t(1) << 34) || c.scaled_rows < 0 ||
            (c.transposed >= 0 && (c.rows % 8 || c.cols % 8 || c.transposed % 8 || (c.to >= 0 && c.to % 8) || (c.same >= 0 && c.same % 4))))
            return fail(S3D_ERR_BAD_SHAPE, "s3d_half_copies: array %d of %lld x %lld (a transposed one: multiples of 8)", i, (long long)c.rows,
                        (long long)c.cols);
        if (!from[i] || ((c.to >= 0 || c.transposed >= 0) && !half) || (c.same >= 0 && !same))
            return fail(S3D_ERR_NULL_POINTER, "s3d_half_copies: null device pointer");
        if (reinterpret_cast<uintptr_t>(half) % 16 || reinterpret_cast<uintptr_t>(same) % 16 ||
            (c.transposed >= 0 && reinterpret_cast<uintptr_t>(from[i]) % 16))
            return fail(S3D_ERR_BAD_SHAPE, "s3d_half_copies: array %d is not aligned to 16 bytes", i);
        a.from[i] = from[i];
        a.of[i] = c;
        a.first[i] = static_cast<int>(blocks);
        blocks += c.transposed >= 0 ? ceil_div(c.rows, kSquare) * ceil_div(c.cols, kSquare) : ceil_div(c.rows * c.cols, kFlat);
    }
    if (blocks == 0) return S3D_OK;
    a.num = num;
    a.half = static_cast<_Float16 *>(half);
    a.same = same;
    hipLaunchKernelGGL(half_copies_kernel, dim3(static_cast<unsigned>(blocks)), dim3(kCastThreads), 0, static_cast<hipStream_t>(stream), a);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

extern "C" __attribute__((visibility("default"))) int s3d_add_half(const float *x, const void *residual, float *out, int64_t count, void *stream)
{
    using namespace s3d;
    if (count < 0 || count % 4) return fail(S3D_ERR_BAD_SHAPE, "s3d_add_half: %lld elements (a multiple of 4)", (long long)count);
    if (count == 0) return S3D_OK;
    if (!x || !residual || !out) return fail(S3D_ERR_NULL_POINTER, "s3d_add_half: null device pointer");
    const int64_t blocks = ceil_div(count / 4, kCastThreads);
    hipLaunchKernelGGL(add_half_kernel, dim3(static_cast<unsigned>(blocks < 4096 ? blocks : 4096)), dim3(kCastThreads), 0, static_cast<hipStream_t>(stream),
                       reinterpret_cast<const f32x4 *>(x), static_cast<const f16x4 *>(residual), reinterpret_cast<f32x4 *>(out), count / 4);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}
