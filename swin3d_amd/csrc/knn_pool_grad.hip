// The gradient of the maximum over the K nearest rows (s3d_knn_max_pool) for the gathered rows (gfx950): every query's
// gradient goes to the rows that hold its maximum, in equal shares, and a row adds up what its queries give it
// (Swin3D/modules/swin3d_layers.py:292-312 under autograd).
//
// The tensor statement writes masks and gradients for all Nq K C gathered numbers and sorts the rows for the scatter.
// Here the rows get the list of their queries by a counting sort, a kernel divides every query's gradient by the number
// of rows that hold its maximum, and a thread per row and 16 bytes of channels adds up its queries' shares: no atomics on
// data.  Shares of fp16 are multiples of 2^-24 below 2^17, whose sums are exact in fp64, so the lists' order, which varies,
// shows in no result; for fp32 it shows below the last place of fp64.
//
// Bound by the gathered 16-byte pieces.  49,682 queries of 16 among 199,327 rows of 96, fp16: 110 us (lists 33, shares 24,
// rows 53) against 1170 through torch's operations, 240 of them the scatter and 150 its sort.
#include "s3d_common.h"

#include <cstring>

#include <rocprim/rocprim.hpp>

namespace s3d {
namespace {

constexpr int kThreads = 256;

__global__ __launch_bounds__(kThreads) void pool_zero_kernel(int32_t *counts, int64_t n)
{
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (t < n) counts[t] = 0;
}

__device__ __forceinline__ int32_t row_of(const int32_t *idx, int64_t t, int64_t Ns)
{
    return static_cast<int32_t>(min(static_cast<int64_t>(max(idx[t], 0)), Ns - 1));
}

__global__ __launch_bounds__(kThreads) void pool_count_kernel(const int32_t *__restrict__ idx, int64_t entries, int64_t Ns,
                                                              int32_t *__restrict__ counts, int32_t *__restrict__ place)
{
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (t < entries) place[t] = atomicAdd(counts + row_of(idx, t, Ns), 1);
}

__global__ __launch_bounds__(kThreads) void pool_fill_kernel(const int32_t *__restrict__ idx, int64_t entries, int K, int64_t Ns,
                                                             const int32_t *__restrict__ starts, const int32_t *__restrict__ place,
                                                             int32_t *__restrict__ queries)
{
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (t < entries) queries[starts[row_of(idx, t, Ns)] + place[t]] = static_cast<int32_t>(t / K);
}

template <typename T, int VEC> struct alignas(sizeof(T) * VEC) Vec { T x[VEC]; };
template <typename T, int VEC> __device__ __forceinline__ Vec<T, VEC> load(const T *p) { return *reinterpret_cast<const Vec<T, VEC> *>(p); }

template <typename T, int VEC>
__global__ __launch_bounds__(kThreads) void pool_share_kernel(const int32_t *__restrict__ idx, int K, int64_t Nq, int64_t Ns,
                                                              const T *__restrict__ feat, const T *__restrict__ out,
                                                              const T *__restrict__ dout, int C, T *__restrict__ share)
{
    const int groups = C / VEC;
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (t >= Nq * groups) return;
    const int64_t q = t / groups, at = q * C + (t - q * groups) * VEC;
    const int c0 = static_cast<int>(t - q * groups) * VEC;
    const Vec<T, VEC> top = load<T, VEC>(out + at), given = load<T, VEC>(dout + at);
    int holders[VEC] = {};
    constexpr int kAhead = 8;
    for (int i0 = 0; i0 < K; i0 += kAhead) {
        Vec<T, VEC> v[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) v[i] = load<T, VEC>(feat + static_cast<int64_t>(row_of(idx, q * K + min(i0 + i, K - 1), Ns)) * C + c0);
#pragma unroll
        for (int i = 0; i < kAhead; ++i)
#pragma unroll
            for (int e = 0; e < VEC; ++e) holders[e] += i0 + i < K && v[i].x[e] == top.x[e];
    }
    Vec<T, VEC> s;
    // (a maximum that is not a number is held by no row: 0 / 0)
#pragma unroll
    for (int e = 0; e < VEC; ++e)
        s.x[e] = holders[e] == 1 ? given.x[e] : static_cast<T>(holders[e] == 0 ? __int_as_float(0x7fc00000) : static_cast<float>(given.x[e]) / static_cast<float>(holders[e]));
    *reinterpret_cast<Vec<T, VEC> *>(share + at) = s;
}

template <typename T, int VEC>
__global__ __launch_bounds__(kThreads) void pool_gather_kernel(const int32_t *__restrict__ starts, const int32_t *__restrict__ queries,
                                                               int64_t Ns, const T *__restrict__ feat, const T *__restrict__ out,
                                                               const T *__restrict__ share, int C, T *__restrict__ dfeat)
{
    const int groups = C / VEC;
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (t >= Ns * groups) return;
    const int64_t row = t / groups;
    const int c0 = static_cast<int>(t - row * groups) * VEC;
    const Vec<T, VEC> v = load<T, VEC>(feat + row * C + c0);
    double sum[VEC] = {};
    const int begin = starts[row], end = starts[row + 1];
    constexpr int kAhead = 2;
    for (int i0 = begin; i0 < end; i0 += kAhead) {
        Vec<T, VEC> top[kAhead], s[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const int64_t at = static_cast<int64_t>(queries[min(i0 + i, end - 1)]) * C + c0;
            top[i] = load<T, VEC>(out + at);
            s[i] = load<T, VEC>(share + at);
        }
#pragma unroll
        for (int i = 0; i < kAhead; ++i)
#pragma unroll
            for (int e = 0; e < VEC; ++e)
                if (i0 + i < end && (top[i].x[e] == v.x[e] || top[i].x[e] != top[i].x[e])) sum[e] += static_cast<double>(s[i].x[e]);
    }
    Vec<T, VEC> d;
#pragma unroll
    for (int e = 0; e < VEC; ++e) d.x[e] = static_cast<T>(sum[e]);
    *reinterpret_cast<Vec<T, VEC> *>(dfeat + row * C + c0) = d;
}

struct PoolLayout {
    size_t counts, starts, place, queries, share, temp, temp_bytes, total;
};

PoolLayout pool_layout(int64_t Nq, int32_t K, int64_t Ns, int32_t C, int32_t dtype)
{
    PoolLayout l{};
    auto take = [&](size_t bytes) {
        const size_t at = l.total;
        l.total += align_up(bytes, 256);
        return at;
    };
    l.counts = take(static_cast<size_t>(Ns + 1) * 4);
    l.starts = take(static_cast<size_t>(Ns + 1) * 4);
    l.place = take(static_cast<size_t>(Nq) * K * 4);
    l.queries = take(static_cast<size_t>(Nq) * K * 4);
    l.share = take(static_cast<size_t>(Nq) * C * (dtype == S3D_DTYPE_F16 ? 2 : 4));
    int32_t *p = nullptr;
    (void)rocprim::exclusive_scan(nullptr, l.temp_bytes, p, p, 0, static_cast<size_t>(Ns + 1), rocprim::plus<int32_t>(), hipStream_t(0));
    l.temp = take(l.temp_bytes);
    return l;
}

bool pool_fits(int64_t Nq, int32_t K, int64_t Ns, int32_t C, int32_t dtype)
{
    return K >= 1 && K <= S3D_KNN_KMAX && Nq >= 1 && Ns >= 1 && C >= 1 && Ns < 0x7fffffffLL && Nq * K < 0x7fffffffLL &&
           Nq * static_cast<int64_t>(C) <= 0x3fffffffffLL && Ns * static_cast<int64_t>(C) <= 0x3fffffffffLL &&
           (dtype == S3D_DTYPE_F32 || dtype == S3D_DTYPE_F16);
}

dim3 grid_of(int64_t threads) { return dim3(static_cast<unsigned>(ceil_div(threads, kThreads))); }

template <typename T, int VEC>
int launch_pool_grad(const PoolLayout &l, char *ws, const int32_t *idx, int K, int64_t Nq, const T *feat, int64_t Ns, int C, const T *out,
                     const T *dout, T *dfeat, hipStream_t s)
{
    int32_t *starts = reinterpret_cast<int32_t *>(ws + l.starts), *queries = reinterpret_cast<int32_t *>(ws + l.queries);
    T *share = reinterpret_cast<T *>(ws + l.share);
    hipLaunchKernelGGL((pool_share_kernel<T, VEC>), grid_of(Nq * (C / VEC)), dim3(kThreads), 0, s, idx, K, Nq, Ns, feat, out, dout, C, share);
    S3D_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL((pool_gather_kernel<T, VEC>), grid_of(Ns * (C / VEC)), dim3(kThreads), 0, s, starts, queries, Ns, feat, out, share, C, dfeat);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

// 16 bytes of channels a thread where rows and pointers allow it
template <typename T>
int launch_pool_grad(const PoolLayout &l, char *ws, const int32_t *idx, int K, int64_t Nq, const void *feat, int64_t Ns, int C, const void *out,
                     const void *dout, void *dfeat, hipStream_t s)
{
    constexpr int kVec = 16 / static_cast<int>(sizeof(T));
    const uintptr_t all = reinterpret_cast<uintptr_t>(feat) | reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(dout) | reinterpret_cast<uintptr_t>(dfeat);
    auto launch = C % kVec == 0 && all % 16 == 0 ? launch_pool_grad<T, kVec> : launch_pool_grad<T, 1>;
    return launch(l, ws, idx, K, Nq, static_cast<const T *>(feat), Ns, C, static_cast<const T *>(out), static_cast<const T *>(dout), static_cast<T *>(dfeat), s);
}

}  // namespace
}  // namespace s3d

extern "C" __attribute__((visibility("default"))) size_t s3d_knn_max_pool_grad_workspace_bytes(int64_t Nq, int32_t K, int64_t Ns, int32_t C, int32_t dtype)
{
    return s3d::pool_fits(Nq, K, Ns, C, dtype) ? s3d::pool_layout(Nq, K, Ns, C, dtype).total : 0;
}

extern "C" __attribute__((visibility("default"))) int s3d_knn_max_pool_grad(
    const int32_t *idx, int32_t K, int64_t Nq, const void *src_feat, int64_t Ns, int32_t C, int32_t dtype, const void *out,
    const void *dout, void *dsrc_feat, void *workspace, size_t workspace_bytes, void *stream)
{
    using namespace s3d;
    if (!pool_fits(Nq, K, Ns, C, dtype))
        return fail(S3D_ERR_BAD_SHAPE, "s3d_knn_max_pool_grad: Nq=%lld K=%d Ns=%lld C=%d dtype=%d out of range", (long long)Nq, K, (long long)Ns, C, dtype);
    if (!idx || !src_feat || !out || !dout || !dsrc_feat) return fail(S3D_ERR_NULL_POINTER, "s3d_knn_max_pool_grad: null device pointer");
    const PoolLayout l = pool_layout(Nq, K, Ns, C, dtype);
    if (!workspace || workspace_bytes < l.total)
        return fail(S3D_ERR_WORKSPACE, "s3d_knn_max_pool_grad: workspace %zu B < required %zu B", workspace ? workspace_bytes : size_t(0), l.total);
    hipStream_t s = static_cast<hipStream_t>(stream);
    char *ws = static_cast<char *>(workspace);
    int32_t *counts = reinterpret_cast<int32_t *>(ws + l.counts), *starts = reinterpret_cast<int32_t *>(ws + l.starts);
    int32_t *place = reinterpret_cast<int32_t *>(ws + l.place);
    const int64_t entries = Nq * K;
    hipLaunchKernelGGL(pool_zero_kernel, grid_of(Ns + 1), dim3(kThreads), 0, s, counts, Ns + 1);
    hipLaunchKernelGGL(pool_count_kernel, grid_of(entries), dim3(kThreads), 0, s, idx, entries, Ns, counts, place);
    S3D_HIP_CHECK(hipGetLastError());
    size_t temp_bytes = l.temp_bytes;
    S3D_HIP_CHECK(rocprim::exclusive_scan(ws + l.temp, temp_bytes, counts, starts, 0, static_cast<size_t>(Ns + 1), rocprim::plus<int32_t>(), s));
    hipLaunchKernelGGL(pool_fill_kernel, grid_of(entries), dim3(kThreads), 0, s, idx, entries, K, Ns, starts, place,
                       reinterpret_cast<int32_t *>(ws + l.queries));
    S3D_HIP_CHECK(hipGetLastError());
    return dtype == S3D_DTYPE_F16 ? launch_pool_grad<_Float16>(l, ws, idx, K, Nq, src_feat, Ns, C, out, dout, dsrc_feat, s)
                                  : launch_pool_grad<float>(l, ws, idx, K, Nq, src_feat, Ns, C, out, dout, dsrc_feat, s);
}
