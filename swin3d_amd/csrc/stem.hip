// The stem at inference in one kernel (gfx950): 3x3x3 convolution over a voxel's lattice neighbours, BatchNorm with its running
// statistics, ReLU (MinkConvBNRelu, Swin3D/modules/mink_layers.py:50-80).  fp16 operands, fp32 accumulation, the convolution rounded
// to fp16 as under autocast, the rest in fp32.
//
// Layer by layer, 595,677 voxels of 9 channels were gathered into rows of 243 numbers (290 MB written and read), and the result went
// to memory four times, between the product, a cast, the norm and ReLU.  Here a voxel's channels are padded to sixteen, a step of a
// product, by a kernel before, so that a lane takes its operand from a neighbour's row as it lies in memory; what there is no
// neighbour for is a row of zeros.  The weights, 70 KB at 80 channels, stay in LDS.  us, the layers / so: 595,677 voxels to 80 channels
// 621 / 140 (360 MB, 77 us at a copy's rate), 199,327 to 48 182 / 39; 25,013 85 / 23,
// the host's share of eight launches and of two.  The error against 64 bits is the same, 9.4e-5.
#include "attn_kernels.h"
#include "dense.h"

namespace s3d {
namespace {

constexpr int kThreads = 256;
constexpr int kOffsets = 27, kWide = 16;                      // neighbours of a voxel (itself among them), channels of a padded row
constexpr int kPitch = kOffsets * kWide / 8 + 1;              // pieces of 16 bytes between the weights of two channels: odd, for the banks
constexpr int kOutPitch = 32 + 8;                             // of 32 finished rows of 32 channels, in fp16 numbers
constexpr int kWaveBytes = 32 * kOffsets * 4;                 // a wavefront's neighbours, then its finished rows
static_assert(32 * kOutPitch * 2 <= kWaveBytes && kWaveBytes % 16 == 0, "they share the room");
constexpr int kMostOut = 96;

struct StemArgs {
    const void *feats;                                        // [N,cin] fp32 or fp16
    const int64_t *neighbours;                                // [N,27]
    const float *weight, *mean, *var, *gamma, *beta;          // [27,cin,cout], [cout] each; gamma, beta or null
    float *out;                                               // [N,cout]
    _Float16 *rows, *weights;                                 // workspace: [N + 2][16], [cout][27][16]
    int64_t N;
    int cin, cout;
    float eps;
};

// The padded rows, one of zeros behind them and one of NaN (a row that is none, as a gather has it), and the weights in fp16, a
// piece of eight numbers a thread.
template <typename T> __global__ __launch_bounds__(kThreads) void stem_prepare_kernel(StemArgs a)
{
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x, pieces = (a.N + 2) * 2;
    half8 v;
    if (t < pieces) {
        const int64_t row = t / 2;
        const int first = static_cast<int>(t % 2) * 8;
        const T *from = static_cast<const T *>(a.feats) + row * a.cin + first;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            v[e] = static_cast<_Float16>(row == a.N + 1 ? __builtin_nanf("") : 0.0f);
            if (row < a.N && first + e < a.cin) v[e] = static_cast<_Float16>(from[e]);
        }
        reinterpret_cast<half8 *>(a.rows)[t] = v;
        return;
    }
    const int64_t w = t - pieces;
    if (w >= static_cast<int64_t>(a.cout) * kOffsets * 2) return;
    const int n = static_cast<int>(w / (kOffsets * 2)), offset = static_cast<int>(w / 2 % kOffsets), first = static_cast<int>(w % 2) * 8;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        v[e] = 0;
        if (first + e < a.cin) v[e] = static_cast<_Float16>(a.weight[static_cast<int64_t>(offset * a.cin + first + e) * a.cout + n]);
    }
    reinterpret_cast<half8 *>(a.weights)[w] = v;
}

// A wavefront takes 32 voxels at a time, TN tiles of 32 channels.
template <int TN> __global__ __launch_bounds__(1024) void stem_kernel(StemArgs a)
{
    extern __shared__ __align__(16) char smem[];
    half8 *weights = reinterpret_cast<half8 *>(smem);
    float *norm = reinterpret_cast<float *>(smem + a.cout * kPitch * 16);       // mean, scale, shift of a channel
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x / 64;
    char *own = reinterpret_cast<char *>(norm + 3 * kMostOut) + wave * kWaveBytes;
    const int r32 = lane & 31, half = lane >> 5;
    for (int p = tid; p < a.cout * kOffsets * 2; p += blockDim.x)
        weights[p / (kOffsets * 2) * kPitch + p % (kOffsets * 2)] = reinterpret_cast<const half8 *>(a.weights)[p];
    for (int c = tid; c < a.cout; c += blockDim.x) {
        norm[c] = a.mean[c];
        norm[kMostOut + c] = (a.gamma ? a.gamma[c] : 1.0f) / sqrtf(a.var[c] + a.eps);
        norm[2 * kMostOut + c] = a.beta ? a.beta[c] : 0.0f;
    }
    __syncthreads();
    const int64_t tiles = (a.N + 31) / 32, step = static_cast<int64_t>(gridDim.x) * waves;
    for (int64_t tile = static_cast<int64_t>(blockIdx.x) * waves + wave; tile < tiles; tile += step) {
        const int64_t first = tile * 32;
        const int here = static_cast<int>(min(int64_t(32), a.N - first));
        int32_t *row_of = reinterpret_cast<int32_t *>(own);
#pragma unroll
        for (int i = 0; i < (32 * kOffsets + 63) / 64; ++i) {
            const int at = i * 64 + lane;
            int64_t row = a.N;
            if (at < here * kOffsets) row = a.neighbours[first * kOffsets + at];
            if (row < 0) row += a.N + 1;       // (counted from behind the row of zeros, as an index is)
            if (at < 32 * kOffsets) row_of[at] = static_cast<int32_t>(row < 0 || row > a.N ? a.N + 1 : row);
        }
        wave_fence();
        f32x16 acc[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[j] = f32x16{};
        constexpr int kAhead = 9;
#pragma unroll
        for (int o0 = 0; o0 < kOffsets; o0 += kAhead) {
            half8 x[kAhead];
#pragma unroll
            for (int i = 0; i < kAhead; ++i)
                x[i] = *reinterpret_cast<const half8 *>(a.rows + static_cast<int64_t>(row_of[r32 * kOffsets + o0 + i]) * kWide + 8 * half);
#pragma unroll
            for (int i = 0; i < kAhead; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(weights[min(32 * j + r32, a.cout - 1) * kPitch + 2 * (o0 + i) + half], x[i], acc[j], 0, 0, 0);
        }
        wave_fence();
        // a lane has channels 8 g + 4 half .. + 3 of 32 of row r32; whole rows leave, a lane's channels the same for all of its rows
        _Float16 *rows = reinterpret_cast<_Float16 *>(own);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                half4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = static_cast<_Float16>(acc[j][4 * g + e]);
                *reinterpret_cast<half4 *>(rows + r32 * kOutPitch + 8 * g + 4 * half) = v;
            }
            wave_fence();
            const int c = 32 * j + lane % 8 * 4, c_in = min(c, a.cout - 4);
            const float4 mean = *reinterpret_cast<const float4 *>(norm + c_in), scale = *reinterpret_cast<const float4 *>(norm + kMostOut + c_in),
                         shift = *reinterpret_cast<const float4 *>(norm + 2 * kMostOut + c_in);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = i * 8 + lane / 8;
                const half4 v = *reinterpret_cast<const half4 *>(rows + r * kOutPitch + lane % 8 * 4);
                auto normed = [](_Float16 x, float m, float s, float b) {
                    const float z = fmaf(static_cast<float>(x) - m, s, b);
                    return z < 0.0f ? 0.0f : z;       // (NaN stays)
                };
                const float4 z = make_float4(normed(v[0], mean.x, scale.x, shift.x), normed(v[1], mean.y, scale.y, shift.y),
                                             normed(v[2], mean.z, scale.z, shift.z), normed(v[3], mean.w, scale.w, shift.w));
                if (r < here && c < a.cout) *reinterpret_cast<float4 *>(a.out + (first + r) * a.cout + c) = z;
            }
            wave_fence();
        }
    }
}

size_t rows_bytes(int64_t N) { return align_up(static_cast<size_t>(N + 2) * kWide * 2, 256); }

template <int TN> int launch(const StemArgs &a, hipStream_t stream)
{
    // As many wavefronts beside the weights as there are tiles for on all CUs, sixteen at most
    const int64_t tiles = ceil_div(a.N, 32), cus = device_cus();
    const int waves = tiles >= 16 * cus ? 16 : tiles >= 8 * cus ? 8 : 4;
    const size_t lds = static_cast<size_t>(a.cout) * kPitch * 16 + 3 * kMostOut * sizeof(float) + static_cast<size_t>(waves) * kWaveBytes;
    S3D_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(stem_kernel<TN>), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    const int64_t groups = ceil_div(tiles, waves);
    hipLaunchKernelGGL(stem_kernel<TN>, dim3(static_cast<unsigned>(groups < cus ? groups : cus)), dim3(64 * waves), lds, stream, a);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

}  // namespace
}  // namespace s3d

extern "C" __attribute__((visibility("default"))) size_t s3d_stem_workspace_bytes(int64_t N, int32_t cout)
{
    return N < 0 || cout < 0 ? 0 : s3d::rows_bytes(N) + static_cast<size_t>(cout) * s3d::kOffsets * s3d::kWide * 2;
}

extern "C" __attribute__((visibility("default"))) int s3d_stem(const void *feats, int32_t dtype, int64_t N, int32_t cin, const int64_t *neighbours,
                                                               const float *weight, int32_t cout, const float *mean, const float *var,
                                                               const float *gamma, const float *beta, float eps, float *out, void *workspace,
                                                               size_t workspace_bytes, void *stream)
{
    using namespace s3d;
    if (N < 0 || N > 0x7ffffff0 || cin < 1 || cin > kWide || cout < 16 || cout % 16 || cout > kMostOut)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_stem: N=%lld, %d to %d channels (1..%d to a multiple of 16 up to %d)", (long long)N, cin, cout, kWide, kMostOut);
    if (dtype != S3D_DTYPE_F32 && dtype != S3D_DTYPE_F16) return fail(S3D_ERR_BAD_DTYPE, "s3d_stem: dtype %d (0 = fp32, 1 = fp16)", dtype);
    if (N == 0) return S3D_OK;
    if (!feats || !neighbours || !weight || !mean || !var || !out || !workspace) return fail(S3D_ERR_NULL_POINTER, "s3d_stem: null device pointer");
    const size_t need = s3d_stem_workspace_bytes(N, cout);
    if (workspace_bytes < need) return fail(S3D_ERR_WORKSPACE, "s3d_stem: workspace %zu B < required %zu B", workspace_bytes, need);
    hipStream_t s = static_cast<hipStream_t>(stream);
    StemArgs a{feats, neighbours, weight, mean, var, gamma, beta, out, static_cast<_Float16 *>(workspace),
               reinterpret_cast<_Float16 *>(static_cast<char *>(workspace) + rows_bytes(N)), N, cin, cout, eps};
    const int64_t pieces = (N + 2) * 2 + static_cast<int64_t>(cout) * kOffsets * 2;
    const dim3 grid(static_cast<unsigned>(ceil_div(pieces, kThreads)));
    if (dtype == S3D_DTYPE_F32) hipLaunchKernelGGL(stem_prepare_kernel<float>, grid, dim3(kThreads), 0, s, a);
    else hipLaunchKernelGGL(stem_prepare_kernel<_Float16>, grid, dim3(kThreads), 0, s, a);
    S3D_HIP_CHECK(hipGetLastError());
    return cout <= 32 ? launch<1>(a, s) : cout <= 64 ? launch<2>(a, s) : launch<3>(a, s);
}
