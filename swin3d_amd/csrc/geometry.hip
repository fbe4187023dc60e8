// The small steps of a level's geometry, a launch each where the tensor statements take three to nine (gfx950): what bounds
// them on a small scan is the host, some six to ten microseconds a launch.
#include "s3d_common.h"

namespace s3d {
namespace {

constexpr int kThreads = 256;

// ends of the batch elements: a thread each searches the ascending batch ids
__global__ __launch_bounds__(kThreads) void segment_ends_kernel(const int32_t *__restrict__ batch, int64_t stride, int64_t N, int B,
                                                                int32_t *__restrict__ out)
{
    const int b = static_cast<int>(blockIdx.x) * kThreads + static_cast<int>(threadIdx.x);
    if (b >= B) return;
    int64_t lo = 0, hi = N;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (batch[mid * stride] <= b) lo = mid + 1;
        else hi = mid;
    }
    out[b] = static_cast<int32_t>(lo);
}

// key of a voxel, ascending as (batch, x, y, z)
__global__ __launch_bounds__(kThreads) void pack_keys_kernel(const int4 *__restrict__ coords, int64_t N, int field, int64_t *__restrict__ out)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= N) return;
    const int4 c = coords[i];
    const int64_t bias = int64_t(1) << (field - 1);
    out[i] = (((static_cast<int64_t>(c.x) * (bias << 1) + (c.y + bias)) * (bias << 1)) + (c.z + bias)) * (bias << 1) + (c.w + bias);
}

// Sixteen lanes a cell (= window of the sort).  The mean of the members' signal rows, a column per lane, members in sorted
// order; then the member nearest to it, a member per lane, columns in order; then what the level above is made of: the
// cell's coordinates and the chosen member's signals.
constexpr int kLanes = 16;
__global__ __launch_bounds__(kThreads) void pool_cells_kernel(
    const int32_t *__restrict__ n2n, const int32_t *__restrict__ w2n, const int32_t *__restrict__ w_sizes, int64_t W,
    const int4 *__restrict__ coords, int step, const float *__restrict__ signals, int64_t stride, int S,
    int64_t *__restrict__ pick, int4 *__restrict__ out_coords, float *__restrict__ out_signals)
{
#pragma clang fp contract(off)
    const int t = threadIdx.x % kLanes;
    const int64_t w_raw = (static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x) / kLanes, w = min(w_raw, W - 1);
    const int begin = w2n[w], size = w_sizes[w];
    float mean = 0.0f;
    for (int p0 = 0; p0 < size; p0 += kLanes) {
        const int row = n2n[begin + min(p0 + t, size - 1)];
        for (int m = 0; m < min(kLanes, size - p0); ++m) {
            const int64_t from = __shfl(row, m, kLanes);
            if (t < S) mean += signals[from * stride + t];
        }
    }
    mean /= static_cast<float>(size);
    float best = INFINITY;
    int best_row = 0x7fffffff;
    for (int p0 = 0; p0 < size; p0 += kLanes) {
        const int row = n2n[begin + min(p0 + t, size - 1)];
        float sq = 0.0f;
        for (int c = 0; c < S; ++c) {
            const float d = signals[static_cast<int64_t>(row) * stride + c] - __shfl(mean, c, kLanes);
            sq += d * d;
        }
        const float dist = sqrtf(sq);
        if (p0 + t < size && (dist < best || (dist == best && row < best_row))) {
            best = dist;
            best_row = row;
        }
    }
#pragma unroll
    for (int other = 1; other < kLanes; other <<= 1) {
        const float d = __shfl_xor(best, other, kLanes);
        const int r = __shfl_xor(best_row, other, kLanes);
        if (d < best || (d == best && r < best_row)) {
            best = d;
            best_row = r;
        }
    }
    if (w_raw >= W) return;
    if (t == 0) {
        pick[w] = best_row;
        const int4 c = coords[n2n[begin]];
        auto down = [&](int x) { return (x >= 0 ? x / step : -((-x + step - 1) / step)) * step; };
        out_coords[w] = make_int4(c.x, down(c.y), down(c.z), down(c.w));
    }
    // (no member is nearest where a signal is NaN: the row is then the caller's to trip over, as without this kernel)
    if (t < S) out_signals[w * S + t] = best_row == 0x7fffffff ? __int_as_float(0x7fc00000) : signals[static_cast<int64_t>(best_row) * stride + t];
}

// As window_signals_kernel, from what a level holds: voxels and the points' signals (batch, x, y, z in voxels, others).
// The position inside the voxel is a difference times the stride's reciprocal, as the framework divides by a number.
__global__ __launch_bounds__(kThreads) void level_signals_kernel(
    const int32_t *__restrict__ w_w_id, const int32_t *__restrict__ n2n, const int4 *__restrict__ coords, float inv_stride,
    const float *__restrict__ signals, int64_t signals_stride, int columns, int window, float xyz_scale, float other_scale,
    float *__restrict__ out, int64_t N)
{
#pragma clang fp contract(off)
    extern __shared__ float tile[];
    const int64_t p0 = static_cast<int64_t>(blockIdx.x) * kThreads, p = p0 + threadIdx.x;
    if (p < N) {
        float *to = tile + threadIdx.x * columns;
        const int64_t row = n2n[p];
        const int id = w_w_id[p];
        const int x = id / (window * window), rest = id - x * (window * window), y = rest / window, z = rest - y * window;
        const int4 c = coords[row];
        const float *from = signals + row * signals_stride;
        to[0] = (static_cast<float>(x) + (from[1] - static_cast<float>(c.y)) * inv_stride) * xyz_scale;
        to[1] = (static_cast<float>(y) + (from[2] - static_cast<float>(c.z)) * inv_stride) * xyz_scale;
        to[2] = (static_cast<float>(z) + (from[3] - static_cast<float>(c.w)) * inv_stride) * xyz_scale;
#pragma unroll 6
        for (int k = 3; k < columns; ++k) to[k] = from[k + 1] * other_scale;
    }
    __syncthreads();
    const int here = static_cast<int>(min(static_cast<int64_t>(kThreads), N - p0)) * columns;
    for (int t = threadIdx.x; t < here; t += kThreads) out[p0 * columns + t] = tile[t];
}

}  // namespace
}  // namespace s3d

extern "C" __attribute__((visibility("default"))) int s3d_segment_ends(const int32_t *batch, int64_t stride, int64_t N, int32_t B,
                                                                       int32_t *out, void *stream)
{
    using namespace s3d;
    if (N < 0 || N > 0x7fffffffLL || B < 0 || stride < 1) return fail(S3D_ERR_BAD_SHAPE, "s3d_segment_ends: N=%lld B=%d stride=%lld", (long long)N, B, (long long)stride);
    if (B == 0) return S3D_OK;
    if (!out || (N > 0 && !batch)) return fail(S3D_ERR_NULL_POINTER, "s3d_segment_ends: null device pointer");
    hipLaunchKernelGGL(segment_ends_kernel, dim3(static_cast<unsigned>(ceil_div(B, kThreads))), dim3(kThreads), 0,
                       static_cast<hipStream_t>(stream), batch, stride, N, B, out);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

extern "C" __attribute__((visibility("default"))) int s3d_pack_keys(const int32_t *coords, int64_t N, int32_t field, int64_t *out, void *stream)
{
    using namespace s3d;
    if (N < 0 || field < 2 || field > 20) return fail(S3D_ERR_BAD_SHAPE, "s3d_pack_keys: N=%lld field=%d (2..20 bits)", (long long)N, field);
    if (N == 0) return S3D_OK;
    if (!coords || !out) return fail(S3D_ERR_NULL_POINTER, "s3d_pack_keys: null device pointer");
    if (reinterpret_cast<uintptr_t>(coords) % 16 != 0) return fail(S3D_ERR_BAD_SHAPE, "s3d_pack_keys: coords must be 16-byte aligned");
    hipLaunchKernelGGL(pack_keys_kernel, dim3(static_cast<unsigned>(ceil_div(N, kThreads))), dim3(kThreads), 0,
                       static_cast<hipStream_t>(stream), reinterpret_cast<const int4 *>(coords), N, field, out);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

extern "C" __attribute__((visibility("default"))) int s3d_pool_cells(
    const int32_t *n2n, const int32_t *w2n, const int32_t *w_sizes, int64_t W, const int32_t *coords, int32_t step,
    const float *signals, int64_t signals_stride, int32_t num_signals, int64_t *pick, int32_t *out_coords, float *out_signals,
    void *stream)
{
    using namespace s3d;
    if (W < 0 || step < 1 || num_signals < 1 || num_signals > kLanes || signals_stride < num_signals)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_pool_cells: W=%lld step=%d num_signals=%d (1..%d) signals_stride=%lld", (long long)W, step,
                    num_signals, kLanes, (long long)signals_stride);
    if (W == 0) return S3D_OK;
    if (!n2n || !w2n || !w_sizes || !coords || !signals || !pick || !out_coords || !out_signals)
        return fail(S3D_ERR_NULL_POINTER, "s3d_pool_cells: null device pointer");
    if (reinterpret_cast<uintptr_t>(coords) % 16 != 0 || reinterpret_cast<uintptr_t>(out_coords) % 16 != 0)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_pool_cells: coordinates must be 16-byte aligned");
    hipLaunchKernelGGL(pool_cells_kernel, dim3(static_cast<unsigned>(ceil_div(W * kLanes, kThreads))), dim3(kThreads), 0,
                       static_cast<hipStream_t>(stream), n2n, w2n, w_sizes, W, reinterpret_cast<const int4 *>(coords), step, signals,
                       signals_stride, num_signals, pick, reinterpret_cast<int4 *>(out_coords), out_signals);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

extern "C" __attribute__((visibility("default"))) int s3d_level_signals(
    const int32_t *w_w_id, const int32_t *n2n, const int32_t *coords, int32_t stride, const float *signals, int64_t signals_stride,
    int32_t num_signals, int32_t window, float xyz_scale, float other_scale, float *out, int64_t N, void *stream)
{
    using namespace s3d;
    if (N < 0 || stride < 1 || num_signals < 0 || num_signals > 29 || window < 1 || window > 10 || signals_stride < 4 + num_signals)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_level_signals: N=%lld stride=%d num_signals=%d (0..29) signals_stride=%lld window=%d", (long long)N,
                    stride, num_signals, (long long)signals_stride, window);
    if (N == 0) return S3D_OK;
    if (!w_w_id || !n2n || !coords || !signals || !out) return fail(S3D_ERR_NULL_POINTER, "s3d_level_signals: null device pointer");
    if (reinterpret_cast<uintptr_t>(coords) % 16 != 0) return fail(S3D_ERR_BAD_SHAPE, "s3d_level_signals: coords must be 16-byte aligned");
    const int columns = 3 + num_signals;
    hipLaunchKernelGGL(level_signals_kernel, dim3(static_cast<unsigned>(ceil_div(N, kThreads))), dim3(kThreads),
                       kThreads * columns * sizeof(float), static_cast<hipStream_t>(stream), w_w_id, n2n,
                       reinterpret_cast<const int4 *>(coords), 1.0f / static_cast<float>(stride), signals, signals_stride, columns, window,
                       xyz_scale, other_scale, out, N);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}
