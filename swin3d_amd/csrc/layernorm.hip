// Residual add fused with LayerNorm for the Swin block around the attention operator (gfx950).
//
// The block (Swin3D/modules/swin3d_layers.py:617-623) computes
//   feats = short_cut + attn(norm1(feats));  feats = feats + mlp(norm2(feats))
// on an fp32 residual stream whose normalised copies feed fp16 GEMMs under autocast.  As separate torch kernels
// that is an add (read two rows, write one), a LayerNorm (read one, write one in fp32) and a cast (read fp32,
// write fp16) per use; this kernel reads the row and the branch output once and writes the updated residual
// row and the normalised row in the GEMM's input type.  Memory bound: 4*C (+2*C) bytes in, 4*C + 2*C out per row.
//
// One group of G lanes per row (G = 16, 32 or 64 by row length), 16-byte loads, two-pass mean / variance in
// registers (the row stays in registers between the passes), fp32 arithmetic.
#include "s3d_common.h"
#include "linear.h"

#include <hip/hip_fp16.h>

namespace s3d {
namespace {

constexpr int kLnThreads = 256;
constexpr int kMaxChunks = 4;   // float4 chunks per lane: rows of up to 4 * 4 * 64 = 1024 channels

template <int kControl> __device__ __forceinline__ float moved(float v)
{
    return __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), kControl, 0xf, 0xf, true));
}
// The sum over G lanes in all of them, pairs first: within rows of sixteen lanes by moves of the VALU (neighbours, pairs, then the
// mirror images of eight and of sixteen, whose quads and eights hold the sums already), where a shuffle goes through LDS.  The same sums in the same pairs.  us with
// shuffles / so: LayerNorm of 390 rows of 384 2.9 / 2.7, of 600 of 640 3.5 / 3.1, of 50,000 of 96 10.7 / 10.6; its gradients, with the
// sums below in sixteen shares / so, 811 rows of 384 9.8 / 8.1, 3,000 11.2 / 9.5, 50,000 of 96 20.1 / 19.5, 199,327 of 48 30.1 / 28.2.
template <int G> __device__ __forceinline__ float group_sum(float v)
{
    v += moved<0xb1>(v);
    v += moved<0x4e>(v);
    v += moved<0x141>(v);
    v += moved<0x140>(v);
    if (G >= 32) {
        const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    }
    if (G >= 64) {
        const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    }
    return v;
}

// RES: 0 = no residual, 1 = fp32 residual, 2 = fp16 residual.  OUT16: normalised rows in fp16 (else fp32).  FOURS: of a lane.
//
// What bounds it: memory for many rows, for few the trips to it, of which there was one for each four and one more for gamma and
// beta behind the sums.  Now all loads of a row are under way together (lanes without a four read the last one).  us, fp16 residual and
// result, before / so: 390 rows of 384, 3.3 / 2.9 (2.7 with group_sum as it is); 600 of 640, 3.8 / 3.5 (3.1); 50,000 of 96, 11.5 / 10.7;
// 600,000 of 80, 111 / 107; no residual, 37,000 of 320, 18.5 / 14.5.
template <int G, int FOURS, int RES, bool OUT16>
__global__ __launch_bounds__(kLnThreads) void add_layernorm_kernel(const float *x, const void *residual, const float *__restrict__ gamma,
                                                                   const float *__restrict__ beta, float eps, float *x_out, void *y,
                                                                   int64_t N, int C)
{
    const int lane = threadIdx.x % G;
    const int64_t row = (static_cast<int64_t>(blockIdx.x) * kLnThreads + threadIdx.x) / G;
    if (row >= N) return;   // whole groups leave together: the shuffles below stay inside a group
    const int chunks = C / 4;   // C is a multiple of 4
    float4 v[FOURS], r[FOURS], g[FOURS], b[FOURS];
    uint2 raw[FOURS];
#pragma unroll
    for (int i = 0; i < FOURS; ++i) {
        const int ch = min(lane + i * G, chunks - 1);
        v[i] = *reinterpret_cast<const float4 *>(x + row * C + 4 * ch);
        if (RES == 1) r[i] = *reinterpret_cast<const float4 *>(static_cast<const float *>(residual) + row * C + 4 * ch);
        if (RES == 2) raw[i] = *reinterpret_cast<const uint2 *>(static_cast<const __half *>(residual) + row * C + 4 * ch);
    }
#pragma unroll
    for (int i = 0; i < FOURS; ++i) {
        const int ch = min(lane + i * G, chunks - 1);
        g[i] = *reinterpret_cast<const float4 *>(gamma + 4 * ch);
        b[i] = *reinterpret_cast<const float4 *>(beta + 4 * ch);
    }
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < FOURS; ++i) {
        if (RES == 2) {
            const float2 lo = __half22float2(*reinterpret_cast<const __half2 *>(&raw[i].x));
            const float2 hi = __half22float2(*reinterpret_cast<const __half2 *>(&raw[i].y));
            r[i] = make_float4(lo.x, lo.y, hi.x, hi.y);
        }
        if (RES != 0) {
            v[i].x += r[i].x; v[i].y += r[i].y; v[i].z += r[i].z; v[i].w += r[i].w;
        }
        if (lane + i * G < chunks) sum += (v[i].x + v[i].y) + (v[i].z + v[i].w);
    }
    const float mean = group_sum<G>(sum) / static_cast<float>(C);
    float sq = 0.0f;
#pragma unroll
    for (int i = 0; i < FOURS; ++i) {
        const float p = v[i].x - mean, q = v[i].y - mean, s = v[i].z - mean, t = v[i].w - mean;
        if (lane + i * G < chunks) sq += (p * p + q * q) + (s * s + t * t);
    }
    const float rstd = rsqrtf(group_sum<G>(sq) / static_cast<float>(C) + eps);
#pragma unroll
    for (int i = 0; i < FOURS; ++i) {
        const int ch = lane + i * G;
        if (ch >= chunks) continue;
        if (RES != 0 && x_out) *reinterpret_cast<float4 *>(x_out + row * C + 4 * ch) = v[i];
        float4 o;
        o.x = (v[i].x - mean) * rstd * g[i].x + b[i].x;
        o.y = (v[i].y - mean) * rstd * g[i].y + b[i].y;
        o.z = (v[i].z - mean) * rstd * g[i].z + b[i].z;
        o.w = (v[i].w - mean) * rstd * g[i].w + b[i].w;
        if (OUT16) {
            uint2 packed;
            *reinterpret_cast<__half2 *>(&packed.x) = __floats2half2_rn(o.x, o.y);
            *reinterpret_cast<__half2 *>(&packed.y) = __floats2half2_rn(o.z, o.w);
            *reinterpret_cast<uint2 *>(static_cast<__half *>(y) + row * C + 4 * ch) = packed;
        } else {
            *reinterpret_cast<float4 *>(static_cast<float *>(y) + row * C + 4 * ch) = o;
        }
    }
}

template <int G, int FOURS, int RES>
void launch_ln(bool out16, const float *x, const void *residual, const float *gamma, const float *beta, float eps,
               float *x_out, void *y, int64_t N, int C, hipStream_t stream)
{
    const int64_t threads = N * G;
    const dim3 grid(static_cast<unsigned>((threads + kLnThreads - 1) / kLnThreads));
    if (out16)
        hipLaunchKernelGGL((add_layernorm_kernel<G, FOURS, RES, true>), grid, dim3(kLnThreads), 0, stream, x, residual, gamma, beta,
                           eps, x_out, y, N, C);
    else
        hipLaunchKernelGGL((add_layernorm_kernel<G, FOURS, RES, false>), grid, dim3(kLnThreads), 0, stream, x, residual, gamma, beta,
                           eps, x_out, y, N, C);
}

template <int G, int FOURS>
void launch_ln_res(int res, bool out16, const float *x, const void *residual, const float *gamma, const float *beta,
                   float eps, float *x_out, void *y, int64_t N, int C, hipStream_t stream)
{
    if (res == 0) launch_ln<G, FOURS, 0>(out16, x, residual, gamma, beta, eps, x_out, y, N, C, stream);
    else if (res == 1) launch_ln<G, FOURS, 1>(out16, x, residual, gamma, beta, eps, x_out, y, N, C, stream);
    else launch_ln<G, FOURS, 2>(out16, x, residual, gamma, beta, eps, x_out, y, N, C, stream);
}

}  // namespace
}  // namespace s3d

extern "C" __attribute__((visibility("default"))) int s3d_add_layernorm(
    const float *x, const void *residual, int32_t residual_dtype, const float *gamma, const float *beta, float eps,
    float *x_out, void *y, int32_t y_dtype, int64_t N, int32_t C, void *stream)
{
    using namespace s3d;
    if (N < 0 || C < 4 || C % 4 != 0 || C > 4 * kMaxChunks * 64)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_add_layernorm: N=%lld C=%d (C a multiple of 4, 4..%d)", (long long)N, C,
                    4 * kMaxChunks * 64);
    if (y_dtype != S3D_DTYPE_F32 && y_dtype != S3D_DTYPE_F16)
        return fail(S3D_ERR_BAD_DTYPE, "s3d_add_layernorm: y_dtype %d (0 = fp32, 1 = fp16)", y_dtype);
    if (residual && residual_dtype != S3D_DTYPE_F32 && residual_dtype != S3D_DTYPE_F16)
        return fail(S3D_ERR_BAD_DTYPE, "s3d_add_layernorm: residual_dtype %d (0 = fp32, 1 = fp16)", residual_dtype);
    if (N == 0) return S3D_OK;
    if (!x || !gamma || !beta || !y) return fail(S3D_ERR_NULL_POINTER, "s3d_add_layernorm: null device pointer");
    const int res = !residual ? 0 : (residual_dtype == S3D_DTYPE_F32 ? 1 : 2);
    const bool out16 = y_dtype == S3D_DTYPE_F16;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int chunks = C / 4;
    auto launch = chunks <= 16 ? launch_ln_res<16, 1> : chunks <= 32 ? launch_ln_res<16, 2> : chunks <= 64 ? launch_ln_res<32, 2>
                  : chunks <= 128 ? launch_ln_res<64, 2> : launch_ln_res<64, kMaxChunks>;
    launch(res, out16, x, residual, gamma, beta, eps, x_out, y, N, C, s);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

// The same for training: (x + residual, LayerNorm of it in fp16) with the bits of torch's forward, since another rounding of a
// row's mean moves single fp16 roundings and with them the gradients of a network on a small scan.  Its sums are running means and
// squared deviations (Welford's recurrence, Chan's rule for two parts): 256 threads a row with four neighbouring numbers each, whose
// parts meet over a wavefront's lanes, the lower halves taking in the upper ones, and then over the wavefronts, two apart first.
// That this is torch's order (2.10.0 for ROCm 7.0) rests on results alone: the test compares every bit of rows of these widths.
// Here a lane holds up to four of those threads' parts, 64 apart, so that all of a row's numbers are loaded at once and none is
// read again, and rows of up to 64 or 128 channels share a wavefront; threads without numbers are parts of no weight.
// Bound by memory: 199,327 rows of 48 with a residual 18.3 us, 6.3 TB/s, where a sum, torch's norm (185 us: a workgroup a row) and a
// cast took 223; 600,000 of 80, 800 -> 115; 49,682 of 96, 73 -> 11; 12,421 of 192, 32 -> 8.  A training pass of Swin3D-S on
// 199,327 voxels 34.0 -> 31.8 ms, of which norms 0.6 (2.6, with 0.3 for the sums before and 0.35 for the casts behind).
namespace s3d {
namespace {

struct Part { float mean, m2, count; };

// the part of four numbers; thirds is the card's reciprocal of 3, which is not the nearest to a third
__device__ __forceinline__ Part part_of(const float4 &v, float thirds)
{
#pragma clang fp contract(off)
    const float x[4] = {v.x, v.y, v.z, v.w}, inverse[4] = {1.0f, 0.5f, thirds, 0.25f};
    float mean = 0.0f, m2 = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float delta = x[e] - mean;
        mean = __builtin_fmaf(delta, inverse[e], mean);
        const float product = delta * (x[e] - mean);      // (rounded before it is added)
        m2 = m2 + product;
    }
    return {mean, m2, 4.0f};
}
// kLanes: of two lanes, the own part and that of a higher one; else of two wavefronts
template <bool kLanes> __device__ __forceinline__ Part joined(const Part &own, const Part &other)
{
#pragma clang fp contract(off)
    const float delta = own.mean - other.mean, count = own.count + other.count;
    const float inverse = __builtin_amdgcn_rcpf(count), to_own = own.count * inverse, to_other = other.count * inverse;
    const float mean = kLanes ? __builtin_fmaf(to_other, other.mean, to_own * own.mean) : __builtin_fmaf(to_own, own.mean, to_other * other.mean);
    const float m2 = __builtin_fmaf(delta * delta * other.count, to_own, own.m2 + other.m2);
    return {count > 0.0f ? mean : 0.0f, count > 0.0f ? m2 : 0.0f, count};
}
template <int kControl> __device__ __forceinline__ Part moved(const Part &p) { return {moved<kControl>(p.mean), moved<kControl>(p.m2), moved<kControl>(p.count)}; }
__device__ __forceinline__ float sixteen_up(float v) { return __uint_as_float(__builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false)[1]); }
__device__ __forceinline__ float half_up(float v) { return __uint_as_float(__builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false)[1]); }

// the parts of a wavefront of 64 threads, of which the first G have numbers, in the first of G lanes
template <int G> __device__ __forceinline__ Part joined_lanes(Part p)
{
    if constexpr (G >= 64) p = joined<true>(p, Part{half_up(p.mean), half_up(p.m2), half_up(p.count)});
    if constexpr (G >= 32) p = joined<true>(p, Part{sixteen_up(p.mean), sixteen_up(p.m2), sixteen_up(p.count)});
    // (of threads without numbers nothing joins but, where its square is infinite, the mean's distance from their 0)
    if constexpr (G < 64) p.m2 = __builtin_fmaf(p.mean * p.mean, 0.0f, p.m2);
    p = joined<true>(p, moved<0x108>(p));      // row_shl
    p = joined<true>(p, moved<0x104>(p));
    p = joined<true>(p, moved<0x102>(p));
    return joined<true>(p, moved<0x101>(p));
}
// the first lane's number in all G
template <int G> __device__ __forceinline__ float of_first(float v)
{
    if constexpr (G == 64) return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v)));
    v = moved<0x150>(v);                       // row_newbcast
    if constexpr (G == 32) v = __uint_as_float(__builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false)[0]);
    return v;
}

template <int G, int PARTS, bool kResidual>
__global__ __launch_bounds__(kLnThreads) void train_layernorm_kernel(const float *__restrict__ x, const __half *residual,
                                                                     const float *__restrict__ gamma, const float *__restrict__ beta, float eps,
                                                                     float *__restrict__ sum, __half *y, int64_t N, int C)
{
    const int lane = threadIdx.x % G;
    const int64_t row = (static_cast<int64_t>(blockIdx.x) * kLnThreads + threadIdx.x) / G;
    if (row >= N) return;   // whole groups leave together
    const int fours = C / 4;
    float4 v[PARTS], g[PARTS], b[PARTS];
    uint2 raw[PARTS];
#pragma unroll
    for (int i = 0; i < PARTS; ++i) {
        const int at = min(lane + i * G, fours - 1);
        v[i] = *reinterpret_cast<const float4 *>(x + row * C + 4 * at);
        if (kResidual) raw[i] = *reinterpret_cast<const uint2 *>(residual + row * C + 4 * at);
    }
#pragma unroll
    for (int i = 0; i < PARTS; ++i) {
        const int at = min(lane + i * G, fours - 1);
        g[i] = *reinterpret_cast<const float4 *>(gamma + 4 * at);
        b[i] = *reinterpret_cast<const float4 *>(beta + 4 * at);
    }
    float three = 3.0f;
    asm volatile("" : "+v"(three));            // (the compiler's reciprocal of a constant is the nearest one)
    const float thirds = __builtin_amdgcn_rcpf(three);
    Part part[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) part[i] = Part{0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < PARTS; ++i) {
        if (kResidual) {
            const float2 lo = __half22float2(*reinterpret_cast<const __half2 *>(&raw[i].x)), hi = __half22float2(*reinterpret_cast<const __half2 *>(&raw[i].y));
            v[i].x += lo.x; v[i].y += lo.y; v[i].z += hi.x; v[i].w += hi.y;
        }
        if (lane + i * G < fours) {
            part[i] = part_of(v[i], thirds);
            if (kResidual) *reinterpret_cast<float4 *>(sum + row * C + 4 * (lane + i * G)) = v[i];
        }
        part[i] = joined_lanes<G>(part[i]);
    }
    const Part all = joined<false>(joined<false>(part[0], part[2]), joined<false>(part[1], part[3]));
    const float mean = of_first<G>(all.mean), rstd = rsqrtf(of_first<G>(all.m2) / static_cast<float>(C) + eps);
#pragma unroll
    for (int i = 0; i < PARTS; ++i) {
        if (lane + i * G >= fours) continue;
        uint2 packed;
        *reinterpret_cast<__half2 *>(&packed.x) = __floats2half2_rn(fmaf(g[i].x, rstd * (v[i].x - mean), b[i].x), fmaf(g[i].y, rstd * (v[i].y - mean), b[i].y));
        *reinterpret_cast<__half2 *>(&packed.y) = __floats2half2_rn(fmaf(g[i].z, rstd * (v[i].z - mean), b[i].z), fmaf(g[i].w, rstd * (v[i].w - mean), b[i].w));
        *reinterpret_cast<uint2 *>(y + row * C + 4 * (lane + i * G)) = packed;
    }
}

template <int G, int PARTS>
void launch_train_layernorm(const float *x, const __half *residual, const float *gamma, const float *beta, float eps, float *sum, __half *y, int64_t N, int C,
                            hipStream_t stream)
{
    const dim3 grid(static_cast<unsigned>(ceil_div(N * G, kLnThreads)));
    auto kernel = residual ? train_layernorm_kernel<G, PARTS, true> : train_layernorm_kernel<G, PARTS, false>;
    hipLaunchKernelGGL(kernel, grid, dim3(kLnThreads), 0, stream, x, residual, gamma, beta, eps, sum, y, N, C);
}

}  // namespace
}  // namespace s3d

extern "C" __attribute__((visibility("default"))) int s3d_train_add_layernorm(const float *x, const void *residual, const float *gamma, const float *beta,
                                                                              float eps, float *sum, void *y, int64_t N, int32_t C, void *stream)
{
    using namespace s3d;
    if (N < 0 || C < 4 || C % 4 != 0 || C > 4 * kMaxChunks * 64)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_train_add_layernorm: N=%lld C=%d (C a multiple of 4, 4..%d)", (long long)N, C, 4 * kMaxChunks * 64);
    if (N == 0) return S3D_OK;
    if (!x || !gamma || !beta || !y || (residual && !sum)) return fail(S3D_ERR_NULL_POINTER, "s3d_train_add_layernorm: null device pointer");
    const int fours = C / 4;
    auto launch = fours <= 16 ? launch_train_layernorm<16, 1> : fours <= 32 ? launch_train_layernorm<32, 1> : fours <= 64 ? launch_train_layernorm<64, 1>
                  : fours <= 128 ? launch_train_layernorm<64, 2> : launch_train_layernorm<64, kMaxChunks>;
    launch(x, static_cast<const __half *>(residual), gamma, beta, eps, sum, static_cast<__half *>(y), N, C, static_cast<hipStream_t>(stream));
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

// The gradients of (sum, y) = (x + residual, LayerNorm(x + residual)):  with h = (sum - mean) rstd and g = dy gamma,
//   d = dsum + rstd (g - mean(g) - h mean(g h)),  dgamma = column sums of dy h,  dbeta = those of dy;
// d goes to x in fp32 and to the residual in its fp16.
//
// Memory bound: the rows of sum, dsum, dy once in, d (and its fp16 copy) once out.  Mean and deviation are taken again from
// the row, which is read anyway.  A lane keeps its channels' share of dgamma and dbeta in registers over all the rows that
// its group draws; the groups of a workgroup add theirs in LDS and leave a part per workgroup, in a fixed order.
// 199,327 rows of 48: 24 us (153 MB moved, 6.5 TB/s), 12,421 of 192: 12 us and the parts' sum 4.7 (linear_grad_sum_kernel); through torch the same
// three gradients took 300 us and 40, with two more passes for the sum with dsum and the fp16 copy.
namespace s3d {
namespace {

struct LnGradArgs {
    const float *sum, *dsum;
    const __half *dy;
    const float *gamma;
    float eps;
    float *dx;
    __half *dres;
    float *parts;      // [workgroups][2 C]
    int64_t N;
    int C;
};

__device__ __forceinline__ float4 load_half4(const __half *p)
{
    const uint2 raw = *reinterpret_cast<const uint2 *>(p);
    const float2 lo = __half22float2(*reinterpret_cast<const __half2 *>(&raw.x)), hi = __half22float2(*reinterpret_cast<const __half2 *>(&raw.y));
    return make_float4(lo.x, lo.y, hi.x, hi.y);
}

// G lanes a row, CH chunks of four channels a lane
template <int G, int CH> __global__ __launch_bounds__(kLnThreads) void layernorm_grad_kernel(LnGradArgs a)
{
    constexpr int kGroups = kLnThreads / G;
    __shared__ float shared[kGroups][G * CH * 4];
    const int lane = threadIdx.x % G, group = threadIdx.x / G, chunks = a.C / 4;
    const float over = 1.0f / static_cast<float>(a.C);
    float gamma[CH][4], dgamma[CH][4] = {}, dbeta[CH][4] = {};
    bool mine[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        mine[i] = lane + i * G < chunks;
        *reinterpret_cast<float4 *>(gamma[i]) = mine[i] ? *reinterpret_cast<const float4 *>(a.gamma + 4 * (lane + i * G)) : make_float4(0, 0, 0, 0);
    }
    const int64_t step = static_cast<int64_t>(gridDim.x) * kGroups;
    for (int64_t row = static_cast<int64_t>(blockIdx.x) * kGroups + group; row < a.N; row += step) {      // (a group stays together)
        float v[CH][4], dy[CH][4], ds[CH][4];
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const int64_t at = row * a.C + 4 * (lane + i * G);
            float4 x = make_float4(0, 0, 0, 0), y = x, s = x;
            if (mine[i]) {
                x = *reinterpret_cast<const float4 *>(a.sum + at);
                y = load_half4(a.dy + at);
                if (a.dsum) s = *reinterpret_cast<const float4 *>(a.dsum + at);
            }
            *reinterpret_cast<float4 *>(v[i]) = x;
            *reinterpret_cast<float4 *>(dy[i]) = y;
            *reinterpret_cast<float4 *>(ds[i]) = s;
            sum += (x.x + x.y) + (x.z + x.w);
        }
        const float mean = group_sum<G>(sum) * over;
        float sq = 0.0f, sum_g = 0.0f, sum_gh = 0.0f;
#pragma unroll
        for (int i = 0; i < CH; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[i][e] = mine[i] ? v[i][e] - mean : 0.0f;
                sq += v[i][e] * v[i][e];
                sum_g += dy[i][e] * gamma[i][e];
                sum_gh += dy[i][e] * gamma[i][e] * v[i][e];
            }
        const float rstd = rsqrtf(group_sum<G>(sq) * over + a.eps);
        const float mean_g = group_sum<G>(sum_g) * over, mean_gh = group_sum<G>(sum_gh) * rstd * over;
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            if (!mine[i]) continue;
            const int64_t at = row * a.C + 4 * (lane + i * G);
            float d[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float h = v[i][e] * rstd;
                dgamma[i][e] += dy[i][e] * h;
                dbeta[i][e] += dy[i][e];
                d[e] = ds[i][e] + rstd * (dy[i][e] * gamma[i][e] - mean_g - h * mean_gh);
            }
            if (a.dx) *reinterpret_cast<float4 *>(a.dx + at) = make_float4(d[0], d[1], d[2], d[3]);
            if (a.dres) {
                uint2 packed;
                *reinterpret_cast<__half2 *>(&packed.x) = __floats2half2_rn(d[0], d[1]);
                *reinterpret_cast<__half2 *>(&packed.y) = __floats2half2_rn(d[2], d[3]);
                *reinterpret_cast<uint2 *>(a.dres + at) = packed;
            }
        }
    }
    float *part = a.parts + static_cast<int64_t>(blockIdx.x) * 2 * a.C;
#pragma unroll
    for (int which = 0; which < 2; ++which) {
        if (which) __syncthreads();
#pragma unroll
        for (int i = 0; i < CH; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) shared[group][4 * (lane + i * G) + e] = which ? dbeta[i][e] : dgamma[i][e];
        __syncthreads();
        for (int c = threadIdx.x; c < a.C; c += kLnThreads) {
            float sum = 0.0f;
#pragma unroll
            for (int g = 0; g < kGroups; ++g) sum += shared[g][c];
            part[which * a.C + c] = sum;
        }
    }
}

// lanes a row: as few as hold it in two chunks each
int ln_lanes(int C) { return C <= 128 ? 16 : C <= 256 ? 32 : 64; }

// four rows a group at least, four workgroups a CU at most
int64_t ln_parts(int64_t N, int C)
{
    const int64_t wanted = ceil_div(N, 4 * (kLnThreads / ln_lanes(C)));
    return wanted < 1024 ? wanted : 1024;
}

bool ln_fits(int64_t N, int32_t C) { return N >= 1 && C >= 4 && C % 4 == 0 && C <= 4 * kMaxChunks * 64; }

}  // namespace

size_t layernorm_grad_bytes(int64_t N, int32_t C) { return ln_fits(N, C) ? static_cast<size_t>(ln_parts(N, C)) * 2 * C * sizeof(float) : 0; }

int launch_layernorm_grad(const float *sum, const float *dsum, const void *dy, const float *gamma, float eps, float *dx, void *dresidual, NormGrad *norm,
                          int64_t N, int32_t C, float *parts, hipStream_t stream)
{
    const LnGradArgs args{sum, dsum, static_cast<const __half *>(dy), gamma, eps, dx, static_cast<__half *>(dresidual), parts, N, C};
    norm->parts = parts;
    norm->count = static_cast<int>(ln_parts(N, C));
    norm->C = C;
    auto kernel = C <= 64 ? layernorm_grad_kernel<16, 1> : C <= 128 ? layernorm_grad_kernel<16, 2> : C <= 256 ? layernorm_grad_kernel<32, 2>
                  : C <= 512 ? layernorm_grad_kernel<64, 2> : layernorm_grad_kernel<64, 4>;
    hipLaunchKernelGGL(kernel, dim3(norm->count), dim3(kLnThreads), 0, stream, args);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

}  // namespace s3d

extern "C" __attribute__((visibility("default"))) size_t s3d_layernorm_grad_workspace_bytes(int64_t N, int32_t C)
{
    return s3d::layernorm_grad_bytes(N, C);
}

extern "C" __attribute__((visibility("default"))) int s3d_layernorm_grad(
    const float *sum, const float *dsum, const void *dy, const float *gamma, float eps, float *dx, void *dresidual, float *dgamma,
    float *dbeta, int64_t N, int32_t C, void *workspace, size_t workspace_bytes, void *stream)
{
    using namespace s3d;
    if (!ln_fits(N, C))
        return fail(S3D_ERR_BAD_SHAPE, "s3d_layernorm_grad: N=%lld C=%d (C a multiple of 4, 4..%d)", (long long)N, C, 4 * kMaxChunks * 64);
    if (!sum || !dy || !gamma || !dgamma || !dbeta) return fail(S3D_ERR_NULL_POINTER, "s3d_layernorm_grad: null device pointer");
    const size_t need = s3d_layernorm_grad_workspace_bytes(N, C);
    if (!workspace || workspace_bytes < need)
        return fail(S3D_ERR_WORKSPACE, "s3d_layernorm_grad: workspace %zu B < required %zu B", workspace ? workspace_bytes : size_t(0), need);
    hipStream_t s = static_cast<hipStream_t>(stream);
    NormGrad norm{nullptr, dgamma, dbeta};
    if (int rc = launch_layernorm_grad(sum, dsum, dy, gamma, eps, dx, dresidual, &norm, N, C, static_cast<float *>(workspace), s)) return rc;
    return launch_linear_grad_sums(nullptr, 0, &norm, S3D_DTYPE_F32, s);
}
