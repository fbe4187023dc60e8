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
