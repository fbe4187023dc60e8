// Y = X W^T + b, with GELU on request: fp16 operands, fp32 accumulation and fp32 bias and GELU, one rounding to fp16
// (gfx950).  The projections of a Swin block at inference (Swin3D/modules/swin3d_layers.py:153-176, 382-560): tall X
// (rows = voxels), K and N a few dozen to a few thousand.
//
// Both operands are contiguous along K, which is how a lane of v_mfma_f32_32x32x16 wants them: eight consecutive numbers
// of a row.  A workgroup stages 64 numbers of K of its rows of X and W in LDS (the next 64 on their way into a second buffer
// meanwhile) with the 16-byte pieces of a row in an order that depends on the row, so that the lanes' reads of 32 rows
// spread over all banks; W goes in as the first operand, so that a lane ends up with four neighbouring outputs of one
// row, and the tile leaves through LDS as whole rows.
//
// At the first levels the layers are bound by memory (K and N below 400): 600,000 rows, 80 -> 320 with GELU, 165 us against
// 416 us as product and GELU apart; 80 -> 240, 96 us against 207, at 4.0 of the 4.7 TB/s that a copy reaches.  At the
// deepest the tiles are few and a tile's chain of chunks is what counts (linear_thin_kernel): 390 rows, 384 -> 384, 3.4 us against 18
// through torch, whose launch alone takes the host that long.
#include "attn_kernels.h"
#include "dense.h"
#include "linear.h"

#include <type_traits>

namespace s3d {
namespace {

constexpr int kThreads = 256;
constexpr int kChunk = 64;        // numbers of K staged at a time
constexpr int kPieces = kChunk / 8;

// The derivative of x Phi(x): Phi(x) + x phi(x), in fp32.  With Phi(-u) = phi(u) M(u), M the ratio of Mills, that is
// phi(u) (u - M(u)) with the sign of x, and 1 more for x above 0, u = |x|: u - M(u) by the polynomial of degree 12 that fits
// phi(u) (u - M(u)) best over [0, 5.8], 8.7e-9 off at most, up to 5, where phi is still large enough to hold its relative error, and by
// a line from there on, where u - M(u) is close to one.  Over all fp16 numbers the error is the rounding of fp32, 9.2e-8 at most
// (1.47e-7 with erff and the exponential apart).  Where the derivative is small and negative it is a relative 1.4e-4 at most from -3 to
// -5, 1.0e-3 to -8 and 6.5e-3 to -13 (1.7e-3, 3.3e-2 and 2.1e-2, since 1 + erf cancels there; with the polynomial alone 3e-2 at -5.8, and beyond -6.8
// the other sign).  Infinities and NaN as the sum of
// the two terms has them: NaN.  A third of the instructions less: 199,327 rows of 48 to 192, us, 52.6 -> 41.5, 49,682 of 96 to 384
// 33.4 -> 27.0, 12,421 of 192 to 768 24.2 -> 19.0, with their rows alone 18, 15 and 12.
__device__ __forceinline__ float gelu_slope(float x)
{
    const float u = fabsf(x), c = fminf(u, 5.0f), phi = __builtin_amdgcn_exp2f(fmaf(u * u, -0.7213475204f, -1.325748064f));
    float q = fmaf(-1.467262933e-07f, c, 4.019878816e-06f);
    q = fmaf(q, c, -4.986505519e-05f);
    q = fmaf(q, c, 3.754729696e-04f);
    q = fmaf(q, c, -1.954356674e-03f);
    q = fmaf(q, c, 7.658625022e-03f);
    q = fmaf(q, c, -2.421350777e-02f);
    q = fmaf(q, c, 6.534569710e-02f);
    q = fmaf(q, c, -1.560686380e-01f);
    q = fmaf(q, c, 3.331732452e-01f);
    q = fmaf(q, c, -6.266347766e-01f);
    q = fmaf(q, c, 1.999998808e+00f);
    q = fmaf(q, c, -1.253314137e+00f);
    q = fmaf(u - c, 1.025f, q);
    return fmaf(__builtin_copysignf(phi, x), q, 0.5f + __builtin_copysignf(0.5f, x));
}

// x Phi(x) of a training forward, as torch has it: by the math library's erff, in this order of operations
__device__ __forceinline__ float gelu_erf(float x) { return (x * 0.5f) * (1.0f + erff(x * 0.70710678f)); }

enum class Behind { kNothing, kGelu, kGeluGrad, kGeluBeside };

// The place of 16-byte piece p of row r: sixteen consecutive rows' pieces p lie in 64 different banks.
__device__ __forceinline__ int placed(int r, int p) { return r * kPieces + (p ^ ((r >> 1) & (kPieces - 1))); }

// Sixteen bytes a lane from `from` to the wavefront's 1024 at `to` in LDS.  The compiler knows nothing of them: who reads them
// has waited for them (loads and stores end in the order of their issue) and met the other wavefronts at a barrier.  (m0 is reserved,
// of which it warns; named, it is a definition of m0, which the compiler's own uses of it have to respect.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load_to_lds(uint32_t to, const void *from)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(to), "v"(from) : "m0", "memory");
}
#pragma clang diagnostic pop
// ... all but the kBehind instructions issued last
template <int kBehind> __device__ __forceinline__ void loads_done() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kBehind) : "memory"); }
__device__ __forceinline__ void workgroup_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// WM x WN wavefronts of TM x TN products of 32 x 32
template <int WM, int WN, int TM, int TN> struct Tile {
    static_assert(WM * WN == kThreads / 64, "four wavefronts");
    static constexpr int kWM = WM, kTM = TM, kTN = TN;
    static constexpr int kM = 32 * WM * TM, kN = 32 * WN * TN;
    static constexpr int kStage = (kM + kN) * kChunk * 2;             // bytes of one staged chunk
    static constexpr int kPitch = 32 * TN + 8;                        // of 32 finished rows of a wavefront
    static_assert(kThreads / 64 * 32 * kPitch * 2 <= kStage, "they fit a buffer");
    static constexpr int kLds = 2 * kStage;
    static constexpr int kLoads = (kM + kN) * kPieces / kThreads;     // pieces per thread and chunk
};

// A workgroup works on tile after tile: the first chunk of the next one is on its way while the last chunk is
// multiplied and the finished rows leave, each wavefront's through its own part of the buffer that has just been multiplied (no
// barrier); where they all are rows of the result, the wait for that chunk leaves their stores under way.  With a workgroup a tile,
// a tile's first load waited for all that.
//
// Chunks go from memory to LDS without a register between.  Through registers a chunk was held by every thread until it was needed,
// stored (a quarter of LDS's time and of the instructions), and two barriers met per tile's end.  us, through registers / so: 9,400
// rows, 2560 -> 640 49.5 / 43.7, 640 -> 1920 33.7 / 30.4; 37,500, 1280 -> 320 51.3 / 45.2, 320 -> 960 38.7 / 34.8; 595,677, 80 -> 240 106 / 96;
// 12,421, 768 -> 192 11.1 / 9.7; 3,105, 1536 -> 384 13.6 / 11.1; 776 and 390 rows of it 9.8 / 8.3; 199,327, 48 -> 48, bound by its rows, 8.7 / 8.4.
// The matrix pipe is busy for a third of the time: a chunk of 128 x 128 is 512 clocks of it and 768 of LDS, and each waits for the
// chunk before.  A third, fourth and fifth buffer, which leave fewer workgroups a CU, were 2 to 15 % slower; operands of the
// next step read ahead 10 to 20 % (spread over the buffers by sched_barriers); 256 x 128 by eight wavefronts the same, 256 x 256 up
// to 1.5 times as long where the last round is nearly empty.
template <typename L, Behind kBehind>
__global__ __launch_bounds__(kThreads, 2) void linear_kernel(const _Float16 *__restrict__ x, const _Float16 *__restrict__ w,
                                                             const _Float16 *__restrict__ bias, _Float16 *__restrict__ y,
                                                             const _Float16 *__restrict__ gelu_at, _Float16 *__restrict__ gelu_out, int M,
                                                             int N, int K, int tiles_n, int tiles)
{
    constexpr int TM = L::kTM, TN = L::kTN;
    __shared__ __align__(16) char smem[L::kLds];
    // workgroups b, b + 8, .. run on one XCD: they get neighbouring tiles, which share rows of X
    const int share = (tiles + 7) / 8, begin = static_cast<int>(blockIdx.x) % 8 * share, end = min(begin + share, tiles);
    const int step = static_cast<int>(gridDim.x) / 8;
    int tile = begin + static_cast<int>(blockIdx.x) / 8;
    if (tile >= end) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_m = wave % L::kWM * (32 * TM), wave_n = wave / L::kWM * (32 * TN);
    const int r32 = lane & 31, half = lane >> 5;
    const int whole = (K - 1) / kChunk;      // chunks before the last one

    // This thread's pieces of a chunk: row (tid / 8 + 32 i) of [X rows, W rows], and of it the piece whose place is lane % 8, as
    // sixteen bytes a lane go to consecutive places.  Where the last chunk has no such piece the lane loads its first one.
    const int row = tid / kPieces, piece = (lane ^ (row >> 1)) & (kPieces - 1);
    const _Float16 *from[L::kLoads];
    const uint32_t lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char *)smem));
    auto aim = [&](int m0, int n0) {
#pragma unroll
        for (int i = 0; i < L::kLoads; ++i) {
            const int r = row + i * (kThreads / kPieces);
            from[i] = r < L::kM ? x + static_cast<int64_t>(min(m0 + r, M - 1)) * K : w + static_cast<int64_t>(min(n0 + r - L::kM, N - 1)) * K;
        }
    };
    auto fetch = [&](int buffer, int k0) {
        const int k = k0 + (k0 + piece * 8 < K ? piece * 8 : 0);
#pragma unroll
        for (int i = 0; i < L::kLoads; ++i) load_to_lds(lds + buffer * L::kStage + i * (kThreads * 16) + wave * 1024, from[i] + k);
    };
    f32x16 acc[TM][TN];
    auto multiply = [&](int buffer, int steps) {
        const half8 *at = reinterpret_cast<const half8 *>(smem + buffer * L::kStage);
#pragma unroll
        for (int s = 0; s < kChunk / 16; ++s) {
            if (s >= steps) break;
            half8 a[TM], b[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) a[i] = at[placed(wave_m + i * 32 + r32, 2 * s + half)];
#pragma unroll
            for (int j = 0; j < TN; ++j) b[j] = at[placed(L::kM + wave_n + j * 32 + r32, 2 * s + half)];
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(b[j], a[i], acc[i][j], 0, 0, 0);
        }
    };
    int buffer = 0;
    bool inside = false;      // the tile before left all its rows and columns: as many stores behind the loads under way
    aim(tile / tiles_n * L::kM, tile % tiles_n * L::kN);
    fetch(0, 0);
    for (; tile < end; tile += step) {
        const int m0 = tile / tiles_n * L::kM, n0 = tile % tiles_n * L::kN;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = f32x16{};
        // the chunk is there, and nobody reads the other buffer any more
        auto meet = [&]() {
            if (inside) loads_done<TM * 2 * TN * (kBehind == Behind::kGeluBeside ? 2 : 1)>();
            else loads_done<0>();
            inside = false;
            workgroup_barrier();
        };
        for (int c = 0; c < whole; ++c) {
            meet();
            fetch(buffer ^ 1, (c + 1) * kChunk);
            multiply(buffer, kChunk / 16);
            buffer ^= 1;
        }
        meet();
        // what the end of the tile reads, before the next tile's first chunk: loads return in order
        half4 b[TN][4];
        half8 at[TM][2 * TN];
        constexpr int kRowPieces = TN * 4;
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                b[j][g] = half4{0, 0, 0, 0};
                if (bias) b[j][g] = *reinterpret_cast<const half4 *>(bias + min(n0 + wave_n + j * 32 + 8 * g + 4 * half, N - 4));
            }
        if constexpr (kBehind == Behind::kGeluGrad) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int t = 0; t < 2 * TN; ++t) {
                    const int e = t * 64 + lane, r = min(m0 + wave_m + i * 32 + e / kRowPieces, M - 1);
                    at[i][t] = *reinterpret_cast<const half8 *>(gelu_at + static_cast<int64_t>(r) * N + min(n0 + wave_n + e % kRowPieces * 8, N - 8));
                }
        }
        const int next = tile + step;
        if (next < end) {
            aim(next / tiles_n * L::kM, next % tiles_n * L::kN);
            fetch(buffer ^ 1, 0);
        }
        multiply(buffer, (K - whole * kChunk) / 16);
        workgroup_barrier();
        inside = m0 + L::kM <= M && n0 + L::kN <= N;
        // a lane's outputs: row r32 of X, columns 8 g + 4 half .. + 3 of W's 32.  They become rows in the wavefront's own part of
        // the buffer that is free now.
        _Float16 *out = reinterpret_cast<_Float16 *>(smem + buffer * L::kStage) + wave * (32 * L::kPitch);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    half4 o;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float v = acc[i][j][4 * g + e] + static_cast<float>(b[j][g][e]);
                        o[e] = static_cast<_Float16>(kBehind == Behind::kGelu ? gelu(v) : v);
                    }
                    *reinterpret_cast<half4 *>(out + r32 * L::kPitch + j * 32 + 8 * g + 4 * half) = o;
                }
#pragma unroll
            for (int t = 0; t < 2 * TN; ++t) {
                const int e = t * 64 + lane, r = e / kRowPieces, n = e % kRowPieces * 8;
                half8 v = *reinterpret_cast<const half8 *>(out + r * L::kPitch + n);
                if constexpr (kBehind == Behind::kGeluGrad) {
#pragma unroll
                    for (int k = 0; k < 8; ++k) v[k] = static_cast<_Float16>(static_cast<float>(v[k]) * gelu_slope(static_cast<float>(at[i][t][k])));
                }
                const int64_t to = static_cast<int64_t>(m0 + wave_m + i * 32 + r) * N + n0 + wave_n + n;
                const bool there = inside || (m0 + wave_m + i * 32 + r < M && n0 + wave_n + n < N);
                if (there) *reinterpret_cast<half8 *>(y + to) = v;
                if constexpr (kBehind == Behind::kGeluBeside) {
#pragma unroll
                    for (int k = 0; k < 8; ++k) v[k] = static_cast<_Float16>(gelu_erf(static_cast<float>(v[k])));
                    if (there) *reinterpret_cast<half8 *>(gelu_out + to) = v;
                }
            }
        }
        buffer ^= 1;
    }
}

template <typename L>
int launch(const LinearArgs &a, hipStream_t stream)
{
    const int tiles_n = (a.N + L::kN - 1) / L::kN;
    const int64_t tiles = ceil_div(a.M, L::kM) * tiles_n;
    if (tiles > (1 << 30)) return fail(S3D_ERR_BAD_SHAPE, "s3d_linear: M = %lld rows", (long long)a.M);
    auto kernel = a.gelu ? linear_kernel<L, Behind::kGelu> : linear_kernel<L, Behind::kNothing>;
    if constexpr (L::kTN < 3) kernel = a.gelu_at ? linear_kernel<L, Behind::kGeluGrad> : kernel;
    if constexpr (L::kTM == 1 && L::kTN == 1) kernel = a.gelu_out ? linear_kernel<L, Behind::kGeluBeside> : kernel;
    // as many workgroups as fit the chip (by LDS), or one a tile
    constexpr int kPerCu = 160 * 1024 / L::kLds < 2 ? 1 : 160 * 1024 / L::kLds < 4 ? 160 * 1024 / L::kLds : 4;
    const int64_t slots = static_cast<int64_t>(kPerCu) * device_cus();
    const dim3 grid(static_cast<unsigned>(ceil_div(tiles < slots ? tiles : slots, 8) * 8));
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, stream, static_cast<const _Float16 *>(a.x), static_cast<const _Float16 *>(a.w),
                       static_cast<const _Float16 *>(a.bias), static_cast<_Float16 *>(a.y), static_cast<const _Float16 *>(a.gelu_at),
                       static_cast<_Float16 *>(a.gelu_out), static_cast<int>(a.M), a.N, a.K, tiles_n, static_cast<int>(tiles));
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

// A tile of 32 x 32 whose chunks are shared by eight wavefronts, wavefront s taking chunks s, s + 8, .. through an LDS buffer of its
// own (no barrier), two chunks ahead in registers.  The sums meet in LDS.
//
// Where tiles of 64 x 64 leave most CUs idle, a launch takes as long as one tile's chain of chunks, 720 clocks each: LDS reads and
// writes of 48 KB, a barrier, a memory round trip in front of it.  (Four groups of wavefronts on that tile's chunks were 14 % faster
// at K = 1536: the LDS traffic is the same.)  Here four times as many CUs have a quarter of it each, and a wavefront all its
// loads under way.  us, tiles of 64 x 64 / so: 390 rows, 1536 -> 384, 10.0 / 5.2; 384 -> 384, 4.5 / 3.4; 390, 2560 -> 640, 22.0 / 9.9;
// 100, 384 -> 1536 with GELU 4.9 / 3.8; 1,563, 192 -> 192, 3.7 / 3.6.
constexpr int kShares = 8;

template <Behind kBehind>
__global__ __launch_bounds__(64 * kShares) void linear_thin_kernel(const _Float16 *__restrict__ x, const _Float16 *__restrict__ w,
                                                                   const _Float16 *__restrict__ bias, _Float16 *__restrict__ y, int M, int N,
                                                                   int K, int tiles_n, int tiles)
{
    constexpr int kOwn = 2 * 32 * kChunk * 2, kPitch = 32 + 4;
    static_assert(32 * kPitch * 4 <= kOwn, "a wavefront's sums fit its buffer");
    __shared__ __align__(16) char smem[kShares * kOwn];
    // workgroups b, b + 8, .. run on one XCD: they get neighbouring tiles, which share rows of X
    const int share = (tiles + 7) / 8, tile = static_cast<int>(blockIdx.x) % 8 * share + static_cast<int>(blockIdx.x) / 8;
    if (tile >= tiles) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r32 = lane & 31, half = lane >> 5;
    const int m0 = tile / tiles_n * 32, n0 = tile % tiles_n * 32, chunks = (K + kChunk - 1) / kChunk;
    char *own = smem + wave * kOwn;

    const int piece = lane % kPieces, row = lane / kPieces;      // rows row + 8 i: of X, then of W
    const _Float16 *from[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int r = row + 8 * (i % 4);
        from[i] = (i < 4 ? x + static_cast<int64_t>(min(m0 + r, M - 1)) * K : w + static_cast<int64_t>(min(n0 + r, N - 1)) * K) + piece * 8;
    }
    f32x16 acc = {};
    auto fetch = [&](uint4 (&held)[8], int chunk) {
        if (chunk * kChunk + piece * 8 < K) {
#pragma unroll
            for (int i = 0; i < 8; ++i) held[i] = *reinterpret_cast<const uint4 *>(from[i] + chunk * kChunk);
        }
    };
    auto multiply = [&](uint4 (&held)[8], int chunk) {
        uint4 *to = reinterpret_cast<uint4 *>(own);
#pragma unroll
        for (int i = 0; i < 8; ++i) to[placed(row + 8 * i, piece)] = held[i];
        fetch(held, chunk + 2 * kShares);
        wave_fence();
        const half8 *at = reinterpret_cast<const half8 *>(own);
        const int steps = min(K - chunk * kChunk, kChunk) / 16;
#pragma unroll
        for (int s = 0; s < kChunk / 16; ++s) {
            if (s >= steps) break;
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(at[placed(32 + r32, 2 * s + half)], at[placed(r32, 2 * s + half)], acc, 0, 0, 0);
        }
        wave_fence();
    };
    uint4 first[8], second[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) first[i] = second[i] = make_uint4(0, 0, 0, 0);
    fetch(first, wave);
    fetch(second, wave + kShares);
    const int n = n0 + threadIdx.x % 16 * 2;
    half2 b = {0, 0};
    if (bias) b = *reinterpret_cast<const half2 *>(bias + min(n, N - 2));
    for (int chunk = wave; chunk < chunks; chunk += 2 * kShares) {
        multiply(first, chunk);
        if (chunk + kShares < chunks) multiply(second, chunk + kShares);
    }
    float *sums = reinterpret_cast<float *>(own);
#pragma unroll
    for (int g = 0; g < 4; ++g)
        *reinterpret_cast<float4 *>(sums + r32 * kPitch + 8 * g + 4 * half) = make_float4(acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]);
    __syncthreads();
#pragma unroll
    for (int r = threadIdx.x / 16; r < 32; r += 4 * kShares) {
        float v[2] = {0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < kShares; ++i) {
            const float2 part = *reinterpret_cast<const float2 *>(smem + i * kOwn + (r * kPitch + threadIdx.x % 16 * 2) * 4);
            v[0] += part.x;
            v[1] += part.y;
        }
        half2 o;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float z = v[e] + static_cast<float>(b[e]);
            o[e] = static_cast<_Float16>(kBehind == Behind::kGelu ? gelu(z) : z);
        }
        if (m0 + r < M && n < N) *reinterpret_cast<half2 *>(y + static_cast<int64_t>(m0 + r) * N + n) = o;
    }
}

int launch_thin(const LinearArgs &a, hipStream_t stream)
{
    const int tiles_n = (a.N + 31) / 32, tiles = static_cast<int>(ceil_div(a.M, 32)) * tiles_n;
    auto kernel = a.gelu ? linear_thin_kernel<Behind::kGelu> : linear_thin_kernel<Behind::kNothing>;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(ceil_div(tiles, 8) * 8)), dim3(64 * kShares), 0, stream, static_cast<const _Float16 *>(a.x),
                       static_cast<const _Float16 *>(a.w), static_cast<const _Float16 *>(a.bias), static_cast<_Float16 *>(a.y), static_cast<int>(a.M), a.N,
                       a.K, tiles_n, tiles);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

}  // namespace

int launch_linear(const LinearArgs &a, hipStream_t stream)
{
    if (a.M < 0 || a.M > 0x7fffffff || a.N < 8 || a.N % 8 || a.K < 16 || a.K % 16)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_linear: M=%lld N=%d K=%d (N a multiple of 8, K of 16)", (long long)a.M, a.N, a.K);
    if (a.M == 0) return S3D_OK;
    if (!a.x || !a.w || !a.y) return fail(S3D_ERR_NULL_POINTER, "s3d_linear: null device pointer");
    // Tiles of 32 x 32 with K shared as long as each has a CU, or half of one with enough chunks to share, or long chains.  us, 64 x 64 /
    // so, by tiles of 32 x 32: up to 260, all K, 0.45 to 0.97 of the time; 282 at K = 96 3.3 / 3.6, 441 3.4 / 3.6; 294 to 490 at K = 192 to
    // 640 0.86 to 1.00; 520 at K = 320 4.8 / 5.8, at 640 5.9 / 6.2, at 2560 23.0 / 13.9; 588 at K = 1536 10.4 / 10.0; 980 at 2560 23.7 / 19.4,
    // at 640 6.3 / 8.0; 1880 at 2560 27.0 / 35.4.
    const int64_t thin = ceil_div(a.M, 32) * ((a.N + 31) / 32);
    if (!a.gelu_at && !a.in_order && (thin <= 256 || (thin <= 512 && a.K >= 192) || (thin <= 1024 && a.K >= 2048))) return launch_thin(a, stream);
    // Tiles of 64 x 64 as long as larger ones would leave CUs without work: up to 576 of them, with GELU or its derivative, whose
    // instructions more wavefronts hide, up to 1024 (768 and 576 to 192, 64 x 64 / 128 x 64, us, by number: 288 6.7 / 7.0, 576 8.8 / 8.5,
    // 720 9.4 / 9.1, 864 11.8 / 9.6; with GELU 585 9.6 / 10.6).  With GELU's derivative and up to 384 channels until there
    // are 6144 of them (0.87 to 0.98 of the time at 1100 to 1700 and 2300 to 6000
    // tiles, 62,000 rows of 96 34.0 -> 29.7 us, 12,421 of 192 18.6 -> 15.8; 1.01 to 1.08 at some 1900 and at 3000; 1.02 to 1.12
    // beyond, and 1.12 to 1.22 at 640 channels); then 128 rows by the width that pads N least,
    // the widest of those that still fill the chip: of 128 columns two are on a CU, so between 384 and 512 they end in one round and
    // from 640 on the second is full enough (640 -> 640, 128 x 128 / 128 x 64, us, by number: 355 13.2 / 12.8, 385 13.8 / 15.7, 450
    // 14.7 / 16.8, 515 21.0 / 18.3, 560 20.6 / 19.5; 1536 -> 384: 354 25.7 / 26.1, 450 28.3 / 35.7, 561 41.8 / 38.9, 642 41.6 / 49.7; with
    // GELU the first is from 448 on).  Over nineteen layers of 96 to 2560 and 96 to 1400 such tiles the choice is 0.8 % behind
    // the best of the three in the mean.  192 columns take all of a wavefront's registers: with GELU only
    // where the tile is the whole row, with its derivative not at all (6 would spill).
    // So, too, with erff's GELU beside the rows, whose fifty instructions a number overlap with other tiles' loads only where
    // several tiles share a SIMD.  us, torch's GELU behind the layer / larger tiles / so: 199,327 rows of 48 to 192 47.0 / 50.9 / 45.0,
    // 49,682 of 96 to 384 30.8 / 34.9 / 26.5, 12,421 of 192 to 768 25.8 / 23.3 / 17.1, 3,105 of 384 to 1536 19.9 / 14.9 / 12.6;
    // 6,250 of 96 11.2 / 7.4.
    const int64_t small = ceil_div(a.M, 64) * ((a.N + 63) / 64);
    const bool heavy = a.gelu || a.gelu_at;
    if (a.gelu_out || small < (heavy ? 1024 : 576) || (a.gelu_at && a.K <= 384 && small <= 6144)) return launch<Tile<2, 2, 1, 1>>(a, stream);
    auto padded = [&](int width) { return (a.N + width - 1) / width * width; };
    auto count = [&](int width) { return ceil_div(a.M, 128) * (padded(width) / width); };
    const int least = padded(64);
    if (padded(192) == least && count(192) >= 512 && !a.gelu_at && (!a.gelu || a.N <= 192)) return launch<Tile<2, 2, 2, 3>>(a, stream);
    if (padded(128) == least && ((count(128) >= (heavy ? 448 : 384) && count(128) <= 512) || count(128) >= 640)) return launch<Tile<2, 2, 2, 2>>(a, stream);
    return launch<Tile<2, 2, 2, 1>>(a, stream);
}

}  // namespace s3d

extern "C" __attribute__((visibility("default"))) int s3d_linear(
    const void *x, const void *w, const void *bias, void *y, int64_t M, int32_t N, int32_t K, int32_t gelu, void *stream)
{
    return s3d::launch_linear(s3d::LinearArgs{x, w, bias, y, M, N, K, gelu != 0}, static_cast<hipStream_t>(stream));
}

extern "C" __attribute__((visibility("default"))) int s3d_linear_in_order(const void *x, const void *w, const void *bias, void *y, void *gelu, int64_t M,
                                                                          int32_t N, int32_t K, void *stream)
{
    s3d::LinearArgs a{x, w, bias, y, M, N, K, false};
    a.in_order = true;
    a.gelu_out = gelu;
    return s3d::launch_linear(a, static_cast<hipStream_t>(stream));
}
