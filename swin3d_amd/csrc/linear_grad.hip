// The gradients of a dense layer's weight and bias: dW = dY^T X, db = the column sums of dY; fp16 operands, fp32
// accumulation, results in the parameters' type (gfx950).  The projections of a Swin block in training
// (Swin3D/modules/swin3d_layers.py:153-176, 382-560): dW is N x K, a few dozen to a few hundred each, and the sum runs
// over the voxels.
//
// What it cannot do without is reading both operands once.  A product that gives a workgroup a tile of dW and all rows
// has a handful of workgroups at the first levels (7 for 48 x 96: 500 us for 199,327 rows); here the rows are split as
// well, so that the chip has two workgroups a CU, and the parts are added by a second kernel: no atomics, the same bits
// on every call.
//
// The matrix instruction wants eight numbers along the sum per lane, but the operands lie across it.  A thread loads
// eight rows of eight columns (16 bytes of a row at a time), turns them in registers (24 byte permutes) and leaves eight
// columns of eight rows in LDS; the next 64 rows are on their way meanwhile.
//
// Both kernels with their launches, against dY^T X and the column sums as two library calls: 199,327 rows, 192 x 48, 30 us
// (3.2 TB/s of operands) against 499; 48 x 48, 19 against 191; 12,421 rows, 768 x 192, 24 against 100; 811 rows, 384 x 384,
// 14 (the host's share of the call) against 28.
#include "linear.h"

namespace s3d {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kRows = 64;            // voxels staged at a time
constexpr int kOctets = kRows / 8;   // 16-byte pieces of a column in LDS

// The place of piece p of column c: the pieces p of 16 neighbouring columns (a read) and those of every eighth column (a
// write) lie in different banks.
__device__ __forceinline__ int placed(int c, int p) { return c * kOctets + (p ^ (((c >> 1) ^ (c >> 4)) & (kOctets - 1))); }

struct GradArgs {
    const _Float16 *dy, *x;   // [M,N], [M,K]
    float *parts;             // [splits][N K + N]
    int64_t M, rows;          // rows of a split: a multiple of kRows
    int N, K, tiles_k;
};

// 2 x 2 wavefronts of UN x UK products of 16 x 16: a tile of 32 UN columns of dY by 32 UK columns of X
template <int UN, int UK>
__global__ __launch_bounds__(kThreads, 2) void linear_grad_kernel(GradArgs a)
{
    constexpr int kN = 32 * UN, kK = 32 * UK;
    static_assert(kN + kK <= kThreads, "a thread turns one block of a chunk");
    __shared__ uint4 staged[2][(kN + kK) * kOctets];
    const int n0 = static_cast<int>(blockIdx.x) / a.tiles_k * kN, k0 = static_cast<int>(blockIdx.x) % a.tiles_k * kK;
    const int64_t begin = static_cast<int64_t>(blockIdx.y) * a.rows, end = min(begin + a.rows, a.M);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_n = wave % 2 * (16 * UN), wave_k = wave / 2 * (16 * UK);

    // this thread's block of a chunk: eight rows of eight columns of [dY columns, X columns]
    constexpr int kAcross = (kN + kK) / 8;
    const bool working = tid < kAcross * kOctets;
    const int octet = tid / kAcross, column = tid % kAcross * 8;
    const bool of_x = column >= kN;
    const int width = of_x ? a.K : a.N, at = of_x ? k0 + column - kN : n0 + column;
    const bool inside = working && at < width;
    const _Float16 *from = (of_x ? a.x : a.dy) + at;
    uint4 held[8];
    auto fetch = [&](int64_t row) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int64_t r = row + octet * 8 + i;
            held[i] = inside && r < end ? *reinterpret_cast<const uint4 *>(from + r * width) : make_uint4(0, 0, 0, 0);
        }
    };
    auto put = [&](uint4 *to) {
        if (!working) return;
        // columns 2 w and 2 w + 1 are the halves of word w of every row
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            uint32_t even[4], odd[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t first = reinterpret_cast<const uint32_t *>(&held[2 * i])[w], second = reinterpret_cast<const uint32_t *>(&held[2 * i + 1])[w];
                even[i] = __builtin_amdgcn_perm(second, first, 0x05040100u);
                odd[i] = __builtin_amdgcn_perm(second, first, 0x07060302u);
            }
            to[placed(column + 2 * w, octet)] = make_uint4(even[0], even[1], even[2], even[3]);
            to[placed(column + 2 * w + 1, octet)] = make_uint4(odd[0], odd[1], odd[2], odd[3]);
        }
    };
    f32x4 acc[UN][UK] = {}, sums[UN] = {};
    const bool sum_dy = k0 == 0 && wave_k == 0;
    half8 ones;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = static_cast<_Float16>(1.0f);
    const int r16 = lane & 15, quarter = lane >> 4;
    auto multiply = [&](const uint4 *buffer) {
        const half8 *from_lds = reinterpret_cast<const half8 *>(buffer);
#pragma unroll
        for (int s = 0; s < kRows / 32; ++s) {
            half8 n[UN], k[UK];
#pragma unroll
            for (int i = 0; i < UN; ++i) n[i] = from_lds[placed(wave_n + 16 * i + r16, 4 * s + quarter)];
#pragma unroll
            for (int j = 0; j < UK; ++j) k[j] = from_lds[placed(kN + wave_k + 16 * j + r16, 4 * s + quarter)];
            // X as the first operand: a lane ends up with four neighbours of a row of dW
#pragma unroll
            for (int i = 0; i < UN; ++i)
#pragma unroll
                for (int j = 0; j < UK; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k[j], n[i], acc[i][j], 0, 0, 0);
            if (sum_dy) {
#pragma unroll
                for (int i = 0; i < UN; ++i) sums[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, n[i], sums[i], 0, 0, 0);
            }
        }
    };
    fetch(begin);
    put(staged[0]);
    __syncthreads();
    int buffer = 0;
    for (int64_t row = begin; row < end; row += kRows, buffer ^= 1) {
        const bool more = row + kRows < end;      // (the same for the whole workgroup)
        if (more) fetch(row + kRows);
        multiply(staged[buffer]);
        if (more) put(staged[buffer ^ 1]);
        __syncthreads();
    }
    float *part = a.parts + static_cast<int64_t>(blockIdx.y) * (static_cast<int64_t>(a.N) * a.K + a.N);
#pragma unroll
    for (int i = 0; i < UN; ++i) {
        const int n = n0 + wave_n + 16 * i + r16;
        if (n >= a.N) continue;
#pragma unroll
        for (int j = 0; j < UK; ++j) {
            const int k = k0 + wave_k + 16 * j + 4 * quarter;
            if (k < a.K) *reinterpret_cast<f32x4 *>(part + static_cast<int64_t>(n) * a.K + k) = acc[i][j];
        }
        if (sum_dy && quarter == 0) part[static_cast<int64_t>(a.N) * a.K + n] = sums[i][0];
    }
}

struct GradSums {
    const float *parts[kMostLinearGrads];
    void *dw[kMostLinearGrads], *db[kMostLinearGrads];
    int64_t products[kMostLinearGrads];
    int n[kMostLinearGrads], k[kMostLinearGrads], splits[kMostLinearGrads], scaled[kMostLinearGrads];
    int first[kMostLinearGrads];      // the first workgroup of each
    float scale[kMostLinearGrads];
};

// The sum of the parts: 64 numbers a workgroup, its four wavefronts share the parts.  Several layers share a launch: the sums
// of a Swin block's four are 5 us each by themselves, for some 20 MB of parts.
template <typename T>
__global__ __launch_bounds__(kThreads) void linear_grad_sum_kernel(GradSums a)
{
    __shared__ float shared[kThreads];
    int at = 0;
#pragma unroll
    for (int i = 1; i < kMostLinearGrads; ++i) at = static_cast<int>(blockIdx.x) >= a.first[i] ? i : at;
    const float *parts = a.parts[0];
    T *dw = static_cast<T *>(a.dw[0]), *db = static_cast<T *>(a.db[0]);
    int64_t products = a.products[0];
    int n = a.n[0], k = a.k[0], splits = a.splits[0], scaled = a.scaled[0], first = a.first[0];
    float scale = a.scale[0];
#pragma unroll
    for (int i = 1; i < kMostLinearGrads; ++i) {
        if (at != i) continue;
        parts = a.parts[i]; dw = static_cast<T *>(a.dw[i]); db = static_cast<T *>(a.db[i]); products = a.products[i];
        n = a.n[i]; k = a.k[i]; splits = a.splits[i]; scaled = a.scaled[i]; first = a.first[i]; scale = a.scale[i];
    }
    const int64_t total = products + n;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t e = (static_cast<int64_t>(blockIdx.x) - first) * 64 + lane, from = min(e, total - 1);
    float sum = 0.0f;
#pragma unroll 8
    for (int s = wave; s < splits; s += 4) sum += parts[s * total + from];
    shared[threadIdx.x] = sum;
    __syncthreads();
    if (wave > 0 || e >= total) return;
    sum = (shared[lane] + shared[lane + 64]) + (shared[lane + 128] + shared[lane + 192]);
    if (e < products) {
        if (e < static_cast<int64_t>(scaled) * k) sum *= scale;
        if (dw) dw[e] = static_cast<T>(sum);
    } else if (db) {
        if (e - products < scaled) sum *= scale;
        db[e - products] = static_cast<T>(sum);
    }
}

struct Split {
    int un, uk, tiles, tiles_k, count;
    int64_t rows;
};

// Per side the tile of 64 or 96 columns that pads least (96 for equals: fewer reads of the other side), and as many parts
// of the rows as give every CU two workgroups, but none of fewer than 256 rows: a part is written and read in fp32, which
// for a tile of 96 x 96 is as much traffic as 192 rows of its operands.
Split split_of(int64_t M, int N, int K)
{
    auto units = [](int width) { return (width + 95) / 96 * 96 <= (width + 63) / 64 * 64 ? 3 : 2; };
    Split s{units(N), units(K), 0, 0, 0, 0};
    s.tiles_k = (K + 32 * s.uk - 1) / (32 * s.uk);
    s.tiles = (N + 32 * s.un - 1) / (32 * s.un) * s.tiles_k;
    const int64_t most = ceil_div(M, 256), wanted = ceil_div(512, s.tiles);
    s.rows = ceil_div(ceil_div(M, most < wanted ? most : wanted), kRows) * kRows;
    s.count = static_cast<int>(ceil_div(M, s.rows));
    return s;
}

bool fits(int64_t M, int32_t N, int32_t K) { return M > 0 && M <= 0x7fffffff && N >= 8 && N % 8 == 0 && K >= 8 && K % 8 == 0 && N <= 16384 && K <= 16384; }

}  // namespace

size_t linear_grad_part_count(const LinearGrad &g) { return static_cast<size_t>(split_of(g.M, g.N, g.K).count) * (static_cast<size_t>(g.N) * g.K + g.N); }

size_t linear_grads_bytes(const LinearGrad *grads, int num)
{
    size_t count = 0;
    for (int i = 0; i < num; ++i) count += linear_grad_part_count(grads[i]);
    return count * sizeof(float);
}

int launch_linear_grad_parts(const LinearGrad &g, float *parts, hipStream_t stream)
{
    if (!fits(g.M, g.N, g.K))
        return fail(S3D_ERR_BAD_SHAPE, "s3d_linear_grad: M=%lld N=%d K=%d (N and K multiples of 8, at most 16384)", (long long)g.M, g.N, g.K);
    const Split split = split_of(g.M, g.N, g.K);
    const GradArgs args{static_cast<const _Float16 *>(g.dy), static_cast<const _Float16 *>(g.x), parts, g.M, split.rows, g.N, g.K, split.tiles_k};
    auto kernel = split.un == 3 ? (split.uk == 3 ? linear_grad_kernel<3, 3> : linear_grad_kernel<3, 2>)
                                : (split.uk == 3 ? linear_grad_kernel<2, 3> : linear_grad_kernel<2, 2>);
    hipLaunchKernelGGL(kernel, dim3(split.tiles, split.count), dim3(kThreads), 0, stream, args);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

int launch_linear_grad_sums(const LinearGrad *grads, int num, float *parts, int32_t grad_dtype, hipStream_t stream)
{
    GradSums a{};
    int64_t blocks = 0;
    for (int i = 0; i < kMostLinearGrads; ++i) {
        a.first[i] = 0x7fffffff;
        if (i >= num) continue;
        const LinearGrad &g = grads[i];
        a.parts[i] = parts;
        a.dw[i] = g.dw;
        a.db[i] = g.db;
        a.products[i] = static_cast<int64_t>(g.N) * g.K;
        a.n[i] = g.N;
        a.k[i] = g.K;
        a.splits[i] = split_of(g.M, g.N, g.K).count;
        a.scaled[i] = g.scaled;
        a.scale[i] = g.scale;
        a.first[i] = static_cast<int>(blocks);
        blocks += ceil_div(a.products[i] + g.N, 64);      // (at most 2^22 + 256 a layer)
        parts += linear_grad_part_count(g);
    }
    if (grad_dtype == S3D_DTYPE_F32)
        hipLaunchKernelGGL(linear_grad_sum_kernel<float>, dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 0, stream, a);
    else
        hipLaunchKernelGGL(linear_grad_sum_kernel<_Float16>, dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 0, stream, a);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

}  // namespace s3d

extern "C" __attribute__((visibility("default"))) size_t s3d_linear_grad_workspace_bytes(int64_t M, int32_t N, int32_t K)
{
    using namespace s3d;
    if (!fits(M, N, K)) return 0;
    return static_cast<size_t>(split_of(M, N, K).count) * (static_cast<size_t>(N) * K + N) * sizeof(float);
}

extern "C" __attribute__((visibility("default"))) int s3d_linear_grad(
    const void *dy, const void *x, void *dw, void *db, int32_t grad_dtype, int64_t M, int32_t N, int32_t K, void *workspace,
    size_t workspace_bytes, void *stream)
{
    using namespace s3d;
    if (!fits(M, N, K))
        return fail(S3D_ERR_BAD_SHAPE, "s3d_linear_grad: M=%lld N=%d K=%d (N and K multiples of 8, at most 16384)", (long long)M, N, K);
    if (grad_dtype != S3D_DTYPE_F32 && grad_dtype != S3D_DTYPE_F16)
        return fail(S3D_ERR_BAD_DTYPE, "s3d_linear_grad: grad_dtype %d (0 = fp32, 1 = fp16)", grad_dtype);
    if (!dy || !x || !(dw || db)) return fail(S3D_ERR_NULL_POINTER, "s3d_linear_grad: null device pointer");
    const size_t need = s3d_linear_grad_workspace_bytes(M, N, K);
    if (!workspace || workspace_bytes < need)
        return fail(S3D_ERR_WORKSPACE, "s3d_linear_grad: workspace %zu B < required %zu B", workspace ? workspace_bytes : size_t(0), need);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const LinearGrad g{dy, x, dw, db, M, N, K, 0, 1.0f};
    float *parts = static_cast<float *>(workspace);
    if (int rc = launch_linear_grad_parts(g, parts, s)) return rc;
    return launch_linear_grad_sums(&g, 1, parts, grad_dtype, s);
}
