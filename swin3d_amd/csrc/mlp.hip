// Y = fc2(GELU(fc1(X))) in one kernel (gfx950): the MLP of a Swin block at inference (Swin3D/modules/swin3d_layers.py:153-176),
// fp16 operands, fp32 accumulation, bias and GELU, the hidden layer and the result rounded to fp16 once, with the bits of the two
// layers apart (linear.hip).
//
// Apart, the hidden layer, four times the rows' channels, went to memory and back: 600,000 rows of 80 channels are 96 MB, their
// hidden layer 381.  Here a wavefront takes 32 rows through both layers, 32 hidden channels at a time: a product's result has a row's
// numbers in the two lanes that the next product wants them in, but for the halves of each sixteen, which change places
// (v_permlane32_swap).  So the hidden layer stays in registers, as do the rows and the result; the weights come through LDS, 32
// hidden channels of both layers at a time, the next ones on their way meanwhile.  us, the layers apart / so: 595,677 rows of 80 279 / 126,
// 149,993 of 160 154 / 97, 199,327 of 48 46 / 26, 49,682 of 96 32 / 20.  Bound by VALU issue, some twenty instructions of GELU a hidden
// number (97 of the 126 us), so these stand between the products: 133, 103, 29 and 23 us with products and GELU one after the other.
#include "dense.h"
#include "linear.h"

namespace s3d {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256, kRows = kThreads / 64 * 32;      // rows of a workgroup
constexpr int kHidden = 32, kMostHidden = 1024;                // hidden channels at a time, and of a layer

template <int C> struct Mlp {
    static_assert(C % 16 == 0, "steps of 16");
    static constexpr int kSteps = C / 16, kTiles = (C + 31) / 32;
    // LDS, in pieces of 16 bytes: rows of both weights an odd number of pieces apart, so that sixteen rows' pieces lie in all banks
    static constexpr int kPitch1 = C / 8 | 1, kPitch2 = kHidden / 8 + 1;
    static constexpr int kPieces = 8 * C, kLoads = (kPieces + kThreads - 1) / kThreads;
    static constexpr int kBuffer = kHidden * kPitch1 + C * kPitch2;
    static constexpr int kOutPitch = 32 + 8;                   // of 32 finished rows of 32 channels of a wavefront, in numbers
    static constexpr int kOut = kThreads / 64 * 32 * kOutPitch / 8;
    static constexpr int kLds = 2 * kBuffer > kOut ? 2 * kBuffer : kOut;
};

template <int C>
__global__ __launch_bounds__(kThreads, 2) void mlp_kernel(const _Float16 *__restrict__ x, const _Float16 *__restrict__ w1,
                                                          const _Float16 *__restrict__ b1, const _Float16 *__restrict__ w2,
                                                          const _Float16 *__restrict__ b2, _Float16 *__restrict__ y, int M, int hidden)
{
    using L = Mlp<C>;
    __shared__ __align__(16) half8 weights_s[L::kLds];
    __shared__ __align__(16) float bias_s[kMostHidden];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r32 = lane & 31, half = lane >> 5;
    const int m0 = static_cast<int>(blockIdx.x) * kRows + wave * 32;

    // this thread's pieces of the weights: of 32 rows of fc1's, which lie one after the other, and of 32 columns of fc2's
    const _Float16 *from[L::kLoads];
    int to[L::kLoads], ahead[L::kLoads];
#pragma unroll
    for (int i = 0; i < L::kLoads; ++i) {
        const int p = min(tid + i * kThreads, L::kPieces - 1), q = p - 4 * C;
        const bool first = q < 0;
        from[i] = first ? w1 + p * 8 : w2 + static_cast<int64_t>(q >> 2) * hidden + (q & 3) * 8;
        ahead[i] = first ? kHidden * C : kHidden;
        to[i] = first ? p / (C / 8) * L::kPitch1 + p % (C / 8) : kHidden * L::kPitch1 + (q >> 2) * L::kPitch2 + (q & 3);
    }
    // A stage is fc1's weights of 32 hidden channels and fc2's of those before them.  (No load behind a branch, where it would be
    // waited for at once: what there is none of comes again, and a thread without a piece has the last one.)
    half8 held[L::kLoads];
    const int chunks = hidden / kHidden;
    auto fetch = [&](int stage) {
#pragma unroll
        for (int i = 0; i < L::kLoads; ++i) {
            held[i] = *reinterpret_cast<const half8 *>(from[i]);
            from[i] += ahead[i] == kHidden ? (stage > 0 ? kHidden : 0) : (stage + 1 < chunks ? kHidden * C : 0);
        }
    };
    auto put = [&](int buffer) {
#pragma unroll
        for (int i = 0; i < L::kLoads; ++i) weights_s[buffer * L::kBuffer + to[i]] = held[i];
    };
    fetch(0);
    half8 rows[L::kSteps];
    {
        const _Float16 *row = x + static_cast<int64_t>(min(m0 + r32, M - 1)) * C + 8 * half;
#pragma unroll
        for (int s = 0; s < L::kSteps; ++s) rows[s] = *reinterpret_cast<const half8 *>(row + 16 * s);
    }
    put(0);
    for (int t = tid; t < hidden; t += kThreads) bias_s[t] = b1 ? static_cast<float>(b1[t]) : 0.0f;
    f32x16 acc[L::kTiles];
#pragma unroll
    for (int j = 0; j < L::kTiles; ++j) acc[j] = f32x16{};
    // (the rows are there: a wait for them inside the loop would also be one for its own loads)
#pragma unroll
    for (int r = 0; r < L::kSteps; ++r) asm volatile("" : "+v"(rows[r]));
    __syncthreads();
    // fc1 of 32 hidden channels: 8 g + 4 half .. + 3 of row r32 are numbers 4 g .. of its sum
    auto first_layer = [&](f32x16 &sum, int buffer, int begin, int end) {
        const half8 *at = weights_s + buffer * L::kBuffer + r32 * L::kPitch1 + half;
#pragma unroll
        for (int s = begin; s < end; ++s) sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(at[2 * s], rows[s], sum, 0, 0, 0);
    };
    uint2 h[4];
    auto activate = [&](const f32x16 &sum, int chunk, int g) {
        const f32x4 b = *reinterpret_cast<const f32x4 *>(bias_s + chunk * kHidden + 8 * g + 4 * half);
        half4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = static_cast<_Float16>(gelu(sum[4 * g + e] + b[e]));
        h[g] = __builtin_bit_cast(uint2, o);
    };
    // hidden channels 16 s + 8 half .. + 7
    auto terms_of = [&](int s) {
        const auto lo = __builtin_amdgcn_permlane32_swap(h[2 * s].x, h[2 * s + 1].x, false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(h[2 * s].y, h[2 * s + 1].y, false, false);
        return __builtin_bit_cast(half8, make_uint4(lo[0], hi[0], lo[1], hi[1]));
    };
    auto second_layer = [&](const half8 &terms, int s, int buffer, int begin, int end) {
        const half8 *at = weights_s + buffer * L::kBuffer + kHidden * L::kPitch1 + half;
#pragma unroll
        for (int j = begin; j < end; ++j) {
            const int r = 32 * j + 32 <= C ? 32 * j + r32 : min(32 * j + r32, C - 1);
            acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(at[r * L::kPitch2 + 2 * s], terms, acc[j], 0, 0, 0);
        }
    };
    fetch(1);
    f32x16 sum = {};
    first_layer(sum, 0, 0, L::kSteps);
    put(1);
    __syncthreads();
    for (int t = 1; t < chunks; ++t) {
        const int buffer = t & 1;
        fetch(t + 1);
        f32x16 next = {};
        half8 terms;
        // GELU's instructions between the products of the next hidden channels, then those of fc2 with the first half of these
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            __builtin_amdgcn_sched_barrier(0);
            constexpr int kHalf = L::kSteps / 2, kSome = L::kTiles / 2;
            if (g == 2) terms = terms_of(0);
            if (g < 2) first_layer(next, buffer, g == 0 ? 0 : kHalf, g == 0 ? kHalf : L::kSteps);
            else second_layer(terms, 0, buffer, g == 2 ? 0 : kSome, g == 2 ? kSome : L::kTiles);
            activate(sum, t - 1, g);
        }
        __builtin_amdgcn_sched_barrier(0);
        second_layer(terms_of(1), 1, buffer, 0, L::kTiles);
        sum = next;
        put(buffer ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) activate(sum, chunks - 1, g);
    second_layer(terms_of(0), 0, chunks & 1, 0, L::kTiles);
    second_layer(terms_of(1), 1, chunks & 1, 0, L::kTiles);
    __syncthreads();
    // the result leaves as rows, 32 channels at a time through the wavefront's own part of LDS (no barrier)
    _Float16 *out = reinterpret_cast<_Float16 *>(weights_s) + wave * (32 * L::kOutPitch);
#pragma unroll
    for (int j = 0; j < L::kTiles; ++j) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            half4 o, b = {0, 0, 0, 0};
            if (b2) b = *reinterpret_cast<const half4 *>(b2 + min(32 * j + 8 * g + 4 * half, C - 4));
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = static_cast<_Float16>(acc[j][4 * g + e] + static_cast<float>(b[e]));
            *reinterpret_cast<half4 *>(out + r32 * L::kOutPitch + 8 * g + 4 * half) = o;
        }
        wave_fence();
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int r = t * 16 + lane / 4, n = lane % 4 * 8;
            const half8 v = *reinterpret_cast<const half8 *>(out + r * L::kOutPitch + n);
            if (m0 + r < M && (32 * j + 32 <= C || 32 * j + n < C)) *reinterpret_cast<half8 *>(y + static_cast<int64_t>(m0 + r) * C + 32 * j + n) = v;
        }
        wave_fence();
    }
}

template <int C> int launch(const MlpArgs &a, hipStream_t stream)
{
    hipLaunchKernelGGL(mlp_kernel<C>, dim3(static_cast<unsigned>(ceil_div(a.M, kRows))), dim3(kThreads), 0, stream, static_cast<const _Float16 *>(a.x),
                       static_cast<const _Float16 *>(a.w1), static_cast<const _Float16 *>(a.b1), static_cast<const _Float16 *>(a.w2),
                       static_cast<const _Float16 *>(a.b2), static_cast<_Float16 *>(a.y), static_cast<int>(a.M), a.hidden);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

}  // namespace

bool mlp_takes(int64_t M, int32_t C, int32_t hidden)
{
    const bool width = C == 48 || C == 64 || C == 80 || C == 96 || C == 128 || C == 160 || C == 192;
    return width && hidden >= kHidden && hidden % kHidden == 0 && hidden <= kMostHidden && M <= (1 << 30);
}

// A workgroup has 128 rows and goes through all hidden channels, so that few rows leave most of the chip idle, the longer the more
// channels there are.  Both layers in one over the layers apart, hidden = 4 C: 1.06 to 1.17 at 12,000 to 15,000 rows of 64 to 96
// channels, 0.92 to 0.97 at 9,000 to 16,000 of 48; at the line 0.92 (48), 0.95 (64), 1.0 (80, 96, 128), 0.76 (160), 1.03 (192); 0.61
// to 0.83 at twice the line's rows, 0.46 at 600,000 of 80.  256 and 320 channels, whose sums leave one wavefront a SIMD: 1.3 at 20,000
// rows, 1.6 at 37,500.
bool mlp_pays(int64_t M, int32_t C, int32_t hidden) { return mlp_takes(M, C, hidden) && M >= 16384 && M >= 192 * C; }

int launch_mlp(const MlpArgs &a, hipStream_t stream)
{
    if (a.M < 0 || !mlp_takes(a.M, a.C, a.hidden)) return fail(S3D_ERR_BAD_SHAPE, "s3d_mlp: M=%lld C=%d hidden=%d", (long long)a.M, a.C, a.hidden);
    if (a.M == 0) return S3D_OK;
    if (!a.x || !a.w1 || !a.w2 || !a.y) return fail(S3D_ERR_NULL_POINTER, "s3d_mlp: null device pointer");
    switch (a.C) {
#define S3D_CASE(C) case C: return launch<C>(a, stream);
        S3D_CASE(48) S3D_CASE(64) S3D_CASE(80) S3D_CASE(96) S3D_CASE(128) S3D_CASE(160) S3D_CASE(192)
#undef S3D_CASE
    }
    return fail(S3D_ERR_BAD_SHAPE, "s3d_mlp: C=%d", a.C);
}

}  // namespace s3d

extern "C" __attribute__((visibility("default"))) int s3d_mlp(const void *x, const void *w1, const void *b1, const void *w2, const void *b2, void *y,
                                                              int64_t M, int32_t C, int32_t hidden, void *stream)
{
    return s3d::launch_mlp(s3d::MlpArgs{x, w1, b1, w2, b2, y, M, C, hidden}, static_cast<hipStream_t>(stream));
}
