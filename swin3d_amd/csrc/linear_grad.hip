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
    int64_t M, rows, chain;   // rows of a split, and of a chain of additions in it: multiples of kRows
    int N, K, tiles_k;
};

// Layers of as many rows and the same tiles share a launch
struct GradGroup {
    GradArgs of[kMostLinearGrads];
    int first[kMostLinearGrads];      // the first tile of each
};

// 2 x 2 wavefronts of UN x UK products of 16 x 16: a tile of 32 UN columns of dY by 32 UK columns of X.  kChains: the sum over
// the rows is one of chains, as long as the parts of the layer by itself (one chain for twice the rows has 1.2 to 1.4 times the
// error against 64 bits).
template <int UN, int UK, bool kChains>
__global__ __launch_bounds__(kThreads, 2) void linear_grad_kernel(GradGroup group)
{
    GradArgs a = group.of[0];
    int first = 0;
#pragma unroll
    for (int i = 1; i < kMostLinearGrads; ++i) {
        if (static_cast<int>(blockIdx.x) < group.first[i]) continue;
        a = group.of[i];
        first = group.first[i];
    }
    constexpr int kN = 32 * UN, kK = 32 * UK;
    static_assert(kN + kK <= kThreads, "a thread turns one block of a chunk");
    __shared__ uint4 staged[2][(kN + kK) * kOctets];
    const int tile = static_cast<int>(blockIdx.x) - first, n0 = tile / a.tiles_k * kN, k0 = tile % a.tiles_k * kK;
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
    f32x4 acc[UN][UK] = {}, sums[UN] = {}, total[UN][UK] = {}, total_sums[UN] = {};
    auto end_chain = [&]() {
#pragma unroll
        for (int i = 0; i < UN; ++i) {
#pragma unroll
            for (int j = 0; j < UK; ++j) {
                total[i][j] += acc[i][j];
                acc[i][j] = f32x4{};
            }
            total_sums[i] += sums[i];
            sums[i] = f32x4{};
        }
    };
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
    int64_t next_chain = begin + a.chain;
    for (int64_t row = begin; row < end; row += kRows, buffer ^= 1) {
        if (kChains && row == next_chain) {
            end_chain();
            next_chain += a.chain;
        }
        const bool more = row + kRows < end;      // (the same for the whole workgroup)
        if (more) fetch(row + kRows);
        multiply(staged[buffer]);
        if (more) put(staged[buffer ^ 1]);
        __syncthreads();
    }
    if (kChains) end_chain();
    float *part = a.parts + static_cast<int64_t>(blockIdx.y) * (static_cast<int64_t>(a.N) * a.K + a.N);
#pragma unroll
    for (int i = 0; i < UN; ++i) {
        const int n = n0 + wave_n + 16 * i + r16;
        if (n >= a.N) continue;
#pragma unroll
        for (int j = 0; j < UK; ++j) {
            const int k = k0 + wave_k + 16 * j + 4 * quarter;
            if (k < a.K) *reinterpret_cast<f32x4 *>(part + static_cast<int64_t>(n) * a.K + k) = kChains ? total[i][j] : acc[i][j];
        }
        if (sum_dy && quarter == 0) part[static_cast<int64_t>(a.N) * a.K + n] = kChains ? total_sums[i][0] : sums[i][0];
    }
}

struct GradSums {
    const float *parts[kMostLinearGrads];
    void *dw[kMostLinearGrads], *db[kMostLinearGrads];
    int64_t products[kMostLinearGrads];
    int n[kMostLinearGrads], k[kMostLinearGrads], splits[kMostLinearGrads], scaled[kMostLinearGrads];
    int first[kMostLinearGrads];      // the first workgroup of each
    float scale[kMostLinearGrads];
    NormGrad norm;
    int first_norm;
};

// Four results to where they fit in one piece, which a gradient inside a larger buffer may not
template <typename T> __device__ __forceinline__ void store_four(T *to, const f32x4 &v)
{
    typedef T four __attribute__((ext_vector_type(4)));
    if (reinterpret_cast<uintptr_t>(to) % sizeof(four) == 0) {
        *reinterpret_cast<four *>(to) = four{static_cast<T>(v[0]), static_cast<T>(v[1]), static_cast<T>(v[2]), static_cast<T>(v[3])};
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) to[i] = static_cast<T>(v[i]);
    }
}

// The sum of the parts: 256 numbers a workgroup, its four wavefronts share the parts.  Several layers share a launch: the sums
// of a Swin block's four are 5 us each by themselves, for some 20 MB of parts.
// With 16-byte loads, where they were 4 bytes, and half the parts (launch_linear_grad_parts), us a block: 96 channels, 50,000 rows, 15 / 10; 192,
// 12,400, 16 / 8; 384, 3,000, 21 / 9; 384, 811, 17.5 / 7.5 (35 MB).
// The parts of a norm, up to 1024 of 2 C numbers, are summed beside them, 16 numbers a workgroup and 64 shares of the parts (sixteen
// were a chain of eight trips to memory).  In a launch of its own behind every block that was 4.5 us
// and the gap before it; 24 blocks, 200,000 voxels: the sums 619 us a pass -> 522, the pass 29.5 ms -> 29.2.
template <typename T>
__global__ __launch_bounds__(kThreads) void linear_grad_sum_kernel(GradSums a)
{
    __shared__ f32x4 shared[kThreads];
    if (static_cast<int>(blockIdx.x) >= a.first_norm) {
        typedef float four __attribute__((ext_vector_type(4), aligned(4)));      // (the caller's scratch memory, as it is)
        constexpr int kShares = kThreads / 4;
        const int share = threadIdx.x / 4, c = (static_cast<int>(blockIdx.x) - a.first_norm) * 16 + threadIdx.x % 4 * 4, width = 2 * a.norm.C;
        const float *from = a.norm.parts + min(c, width - 4);
        f32x4 sum = {};
#pragma unroll 8
        for (int p = share; p < a.norm.count; p += kShares) sum += *reinterpret_cast<const four *>(from + static_cast<int64_t>(p) * width);
        shared[threadIdx.x] = sum;
#pragma unroll
        for (int half = kShares / 2; half > 0; half /= 2) {
            __syncthreads();
            if (share < half) shared[threadIdx.x] = sum += shared[threadIdx.x + 4 * half];
        }
        if (share == 0 && c < width) store_four(c < a.norm.C ? a.norm.dgamma + c : a.norm.dbeta + (c - a.norm.C), sum);
        return;
    }
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
    // (N and K are multiples of 8: four numbers are of one row, and of the weight or of the bias)
    const int64_t e = (static_cast<int64_t>(blockIdx.x) - first) * 256 + 4 * lane, from = min(e, total - 4);
    f32x4 sum = {};
#pragma unroll 8
    for (int s = wave; s < splits; s += 4) sum += *reinterpret_cast<const f32x4 *>(parts + s * total + from);
    shared[threadIdx.x] = sum;
    __syncthreads();
    if (wave > 0 || e >= total) return;
    sum = (shared[lane] + shared[lane + 64]) + (shared[lane + 128] + shared[lane + 192]);
    if (e < products) {
        if (e < static_cast<int64_t>(scaled) * k) sum *= scale;
        if (dw) store_four(dw + e, sum);
    } else if (db) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (e - products + i < scaled) sum[i] *= scale;
        store_four(db + (e - products), sum);
    }
}

// Per side the tile of 64 or 96 columns that pads least (96 for equals: fewer reads of the other side).
struct Tiles {
    int un, uk, count, along_k;
};

Tiles tiles_of(int N, int K)
{
    auto units = [](int width) { return (width + 95) / 96 * 96 <= (width + 63) / 64 * 64 ? 3 : 2; };
    Tiles t{units(N), units(K), 0, 0};
    t.along_k = (K + 32 * t.uk - 1) / (32 * t.uk);
    t.count = (N + 32 * t.un - 1) / (32 * t.un) * t.along_k;
    return t;
}

// As many parts of the rows as give every CU two workgroups, but none of fewer than 256 rows: a part is written and read in
// fp32, which for a tile of 96 x 96 is as much traffic as 192 rows of its operands.  More tiles never make more parts.
struct Split {
    int64_t rows;
    int count;
};

Split split_of(int64_t M, int tiles)
{
    const int64_t most = ceil_div(M, 256), wanted = ceil_div(512, tiles);
    const int64_t rows = ceil_div(ceil_div(M, most < wanted ? most : wanted), kRows) * kRows;
    return {rows, static_cast<int>(ceil_div(M, rows))};
}

bool fits(int64_t M, int32_t N, int32_t K) { return M > 0 && M <= 0x7fffffff && N >= 8 && N % 8 == 0 && K >= 8 && K % 8 == 0 && N <= 16384 && K <= 16384; }

}  // namespace

size_t linear_grads_bytes(const LinearGrad *grads, int num)
{
    size_t count = 0;
    for (int i = 0; i < num; ++i)
        count += static_cast<size_t>(split_of(grads[i].M, tiles_of(grads[i].N, grads[i].K).count).count) *
                 (static_cast<size_t>(grads[i].N) * grads[i].K + grads[i].N);
    return count * sizeof(float);
}

namespace {

template <int UN, int UK> int launch_group(const GradGroup &group, int tiles, int splits, bool chains, hipStream_t stream)
{
    if (chains)
        hipLaunchKernelGGL((linear_grad_kernel<UN, UK, true>), dim3(tiles, splits), dim3(kThreads), 0, stream, group);
    else
        hipLaunchKernelGGL((linear_grad_kernel<UN, UK, false>), dim3(tiles, splits), dim3(kThreads), 0, stream, group);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

// the layers of `which` (bits), whose tiles are the same, in one launch
int launch_some(LinearGrad *grads, int num, unsigned which, float **parts, hipStream_t stream)
{
    int tiles = 0, at = 0;
    for (int i = 0; i < num; ++i)
        if (which >> i & 1) tiles += tiles_of(grads[i].N, grads[i].K).count;
    const Split split = split_of(grads[0].M, tiles);
    GradGroup group{};
    Tiles t{};
    bool chains = false;
    for (int i = 0, first = 0; i < num; ++i) {
        if (!(which >> i & 1)) continue;
        LinearGrad &g = grads[i];
        t = tiles_of(g.N, g.K);
        const int64_t chain = split_of(g.M, t.count).rows;
        chains = chains || chain < split.rows;
        group.of[at] = {static_cast<const _Float16 *>(g.dy), static_cast<const _Float16 *>(g.x), *parts, g.M, split.rows, chain, g.N, g.K, t.along_k};
        group.first[at++] = first;
        first += t.count;
        g.parts = *parts;
        g.splits = split.count;
        *parts += static_cast<size_t>(split.count) * (static_cast<size_t>(g.N) * g.K + g.N);
    }
    for (; at < kMostLinearGrads; ++at) group.first[at] = 0x7fffffff;
    return t.un == 3 ? (t.uk == 3 ? launch_group<3, 3>(group, tiles, split.count, chains, stream) : launch_group<3, 2>(group, tiles, split.count, chains, stream))
                     : (t.uk == 3 ? launch_group<2, 3>(group, tiles, split.count, chains, stream) : launch_group<2, 2>(group, tiles, split.count, chains, stream));
}

}  // namespace

// Layers with the same tiles share a launch as long as that leaves each a part: two have half the parts each, and one beginning
// and one end.  (Beyond, they have one part or two by themselves, and the registers of chains cost a workgroup a CU: 640 -> 2560
// and back, 2,300 rows, together 1.3 times as slow.)  The four layers of a Swin block, us for the parts, alone / in pairs: 96
// channels, 50,000 rows, 62 / 50; 192, 12,400, 59 / 47; 384, 3,000, 51 / 39; 384, 811, 34 / 21.
int launch_linear_grad_parts(LinearGrad *grads, int num, float **parts, hipStream_t stream)
{
    unsigned left = 0;
    for (int i = 0; i < num; ++i) {
        if (!fits(grads[i].M, grads[i].N, grads[i].K) || grads[i].M != grads[0].M)
            return fail(S3D_ERR_BAD_SHAPE, "s3d_linear_grad: M=%lld N=%d K=%d (N and K multiples of 8, at most 16384)", (long long)grads[i].M,
                        grads[i].N, grads[i].K);
        left |= 1u << i;
    }
    for (int i = 0; i < num; ++i) {
        if (!(left >> i & 1)) continue;
        const Tiles t = tiles_of(grads[i].N, grads[i].K);
        unsigned which = 1u << i;
        int tiles = t.count;
        for (int j = i + 1; j < num; ++j) {
            const Tiles other = tiles_of(grads[j].N, grads[j].K);
            if (other.un != t.un || other.uk != t.uk || tiles + other.count > 512) continue;
            which |= 1u << j;
            tiles += other.count;
        }
        left &= ~which;
        if (int rc = launch_some(grads, num, which, parts, stream)) return rc;
    }
    return S3D_OK;
}

int launch_linear_grad_sums(const LinearGrad *grads, int num, const NormGrad *norm, int32_t grad_dtype, hipStream_t stream)
{
    GradSums a{};
    int64_t blocks = 0;
    for (int i = 0; i < kMostLinearGrads; ++i) {
        a.first[i] = 0x7fffffff;
        if (i >= num) continue;
        const LinearGrad &g = grads[i];
        a.parts[i] = g.parts;
        a.dw[i] = g.dw;
        a.db[i] = g.db;
        a.products[i] = static_cast<int64_t>(g.N) * g.K;
        a.n[i] = g.N;
        a.k[i] = g.K;
        a.splits[i] = g.splits;
        a.scaled[i] = g.scaled;
        a.scale[i] = g.scale;
        a.first[i] = static_cast<int>(blocks);
        blocks += ceil_div(a.products[i] + g.N, 256);      // (at most 2^20 + 64 a layer)
    }
    a.first_norm = static_cast<int>(blocks);
    if (norm) {
        a.norm = *norm;
        blocks += ceil_div(2 * norm->C, 16);
    }
    if (blocks == 0) return S3D_OK;
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
    const LinearGrad g{nullptr, nullptr, nullptr, nullptr, M, N, K, 0, 1.0f};
    return linear_grads_bytes(&g, 1);
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
    LinearGrad g{dy, x, dw, db, M, N, K, 0, 1.0f};
    float *parts = static_cast<float *>(workspace);
    if (int rc = launch_linear_grad_parts(&g, 1, &parts, s)) return rc;
    return launch_linear_grad_sums(&g, 1, nullptr, grad_dtype, s);
}
