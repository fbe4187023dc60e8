// Pieces shared by the tile kernels of the attention forward and backward (gfx950): the unit list, matrix operands in
// fp16 or split fp32, LDS cells.
#pragma once

#include "attn_kernels.h"
#include "sweep_common.h"

namespace s3d {
namespace tile {

using namespace sweep;

constexpr int kThreads = 512;            // eight wavefronts; two workgroups share a CU (LDS, 128 registers)
constexpr int kWaves = kThreads / 64;
constexpr int kCols = 64;                // voxels on either side of a tile
constexpr int kSteps = 8;                // pairs of a thread at most: kCols * kCols / kThreads
// Words between rows of a [row][column] array in LDS.  Lanes of a wavefront hold consecutive columns: gathers and atomic
// adds of different rows then meet in a bank only where 8 (r - r') = c' - c mod 64, the two half-wavefronts of a 32x32
// matrix result (four rows apart) write to different halves of the banks, and so do the four lane groups of a 16x16x32
// operand when they take rows two apart (permuted_row).
constexpr int kStride = 72;
// a key's row: its coordinates, then its products with the rows of a stage.  8 mod 16 words for the same reason
constexpr int kCoordWords = 12, kKeyStride = 88;

// The axes are worked off in stages of at most 64 table rows: every position axis is a stage, colour and normal axes
// (at most 32 rows) share one in pairs, the second one's rows behind the first one's 32.
template <int ND> struct Stages {
    static constexpr int kCount = 3 + (ND - 3 + 1) / 2;
    static constexpr int first(int st) { return st < 3 ? st : 3 + 2 * (st - 3); }
    static constexpr bool paired(int st) { return st >= 3 && first(st) + 1 < ND; }
};

// position of matrix row `row` (0..31 of a 32-row group) in the order in which a 16x16x32 operand takes them: lane
// group g holds rows 2 g, 2 g + 1, 8 + 2 g, ... so that its strided reads fall into banks of their own
__host__ __device__ constexpr int permuted_row(int row) { return ((row % 8) / 2) * 8 + row % 2 + 2 * (row / 8); }

// ---- unit list --------------------------------------------------------------------------------------------------------
// A unit is what a workgroup takes on at a time for one head: up to 64 queries of one window, or all voxels of the
// several small windows of one size that fit 64 columns.  Windows of more than 64 voxels are cut into equal tiles.
struct UnitList {
    const int32_t *total;      // [0]: units
    const int4 *units;         // (first entry, voxels per window, windows, 0) or (first position, voxels, tile, tiles)
    const int32_t *entries;    // first sorted positions of the windows of at most 64 voxels, by size
};
inline size_t list_round(size_t bytes) { return (bytes + 255) / 256 * 256; }
inline size_t list_max_units(int64_t N, int64_t W) { return static_cast<size_t>(W > 0 ? W : 0) + static_cast<size_t>(N > 0 ? N : 0) / 32 + 1; }
inline size_t list_bytes(int64_t N, int64_t W)
{
    return 256 + list_round(sizeof(int4) * list_max_units(N, W)) + list_round(sizeof(int32_t) * static_cast<size_t>(W > 0 ? W : 1));
}
inline UnitList list_at(void *p, int64_t N, int64_t W)
{
    char *base = static_cast<char *>(p);
    UnitList l;
    l.total = reinterpret_cast<const int32_t *>(base);
    l.units = reinterpret_cast<const int4 *>(base + 256);
    l.entries = reinterpret_cast<const int32_t *>(base + 256 + list_round(sizeof(int4) * list_max_units(N, W)));
    return l;
}
int launch_list(const UnitList &l, const int32_t *w_sizes, const int32_t *w2n, int64_t W, hipStream_t stream);

// ---- LDS --------------------------------------------------------------------------------------------------------------
typedef __attribute__((address_space(3))) float lds_f32;
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef __attribute__((address_space(3))) int lds_i32;
typedef __attribute__((address_space(3))) u32x4_t lds_u32x4;
__device__ __forceinline__ float lds_load(uint32_t addr) { return *(lds_f32 *)(addr); }
__device__ __forceinline__ uint32_t lds_load_u32(uint32_t addr) { return *(lds_u32 *)(addr); }
__device__ __forceinline__ void lds_store(uint32_t addr, float v) { *(lds_f32 *)(addr) = v; }
__device__ __forceinline__ void lds_store_u32(uint32_t addr, uint32_t v) { *(lds_u32 *)(addr) = v; }
__device__ __forceinline__ void lds_store4(uint32_t addr, float a, float b, float c, float d)
{
    *(__attribute__((address_space(3))) f32x4_t *)(addr) = f32x4_t{a, b, c, d};
}
__device__ __forceinline__ void lds_add(uint32_t addr, uint32_t v)
{
    __hip_atomic_fetch_add((lds_u32 *)(addr), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_max(uint32_t addr, int v)
{
    __hip_atomic_fetch_max((lds_i32 *)(addr), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// order-preserving integer image of a float
__device__ __forceinline__ int float_order(float f)
{
    const int i = __float_as_int(f);
    return i >= 0 ? i : i ^ 0x7fffffff;
}
__device__ __forceinline__ float order_float(int i) { return __int_as_float(i >= 0 ? i : i ^ 0x7fffffff); }
// a value that the compiler cannot follow
__device__ __forceinline__ int opaque(int x)
{
    asm volatile("" : "+v"(x));
    return x;
}
// zero kWords LDS words with all threads
template <int kWords> __device__ __forceinline__ void lds_zero(uint32_t addr, int tid)
{
    const u32x4_t zero = {0, 0, 0, 0};
    constexpr int kPass = kThreads * 4;
    static_assert(kWords % 4 == 0, "16-byte stores");
    addr += tid * 16;
#pragma unroll
    for (int w = 0; w + kPass <= kWords; w += kPass) *(lds_u32x4 *)(addr + w * 4) = zero;
    if constexpr (kWords % kPass != 0) {
        if (tid * 4 < kWords % kPass) *(lds_u32x4 *)(addr + kWords / kPass * kPass * 4) = zero;
    }
}
// LDS address of a __shared__ array
__device__ __forceinline__ uint32_t lds_base(float *p)
{
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) float *)p));
}

// `fn(s)` for the steps 0 .. steps - 1 of a thread, and for some behind them (whose pairs carry no weight): the first
// three without a branch between them, so that their LDS reads are under way together
template <typename Fn> __device__ __forceinline__ void for_steps(int steps, Fn fn)
{
    static_assert(kSteps == 8, "groups of steps");
    fn(0); fn(1); fn(2);
    if (steps > 3) {
        fn(3);
        if (steps > 4) {
            fn(4);
            if (steps > 5) {
                fn(5);
                if (steps > 6) { fn(6); fn(7); }
            }
        }
    }
}

// ---- matrix operands --------------------------------------------------------------------------------------------------
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Eight values of an operand.  fp16 as they are; fp32 as a sum of three bf16 numbers, which hold its 24 bits exactly:
// the six largest of the nine partial products keep a product to 2^-24 of itself, what fp32 arithmetic rounds to, at
// a third of the time of fp32 matrix instructions.
template <typename T> struct Operand;
template <> struct Operand<__half> {
    f16x8 x;
    struct Raw { uint4 v; };             // as loaded, before any conversion
    static __device__ __forceinline__ Raw fetch(const __half *p) { return {*reinterpret_cast<const uint4 *>(p)}; }
    __device__ __forceinline__ void set(const Raw &r) { x = __builtin_bit_cast(f16x8, r.v); }
    __device__ __forceinline__ void load(const __half *p) { x = __builtin_bit_cast(f16x8, *reinterpret_cast<const uint4 *>(p)); }
    __device__ __forceinline__ void load_lds(uint32_t addr) { x = __builtin_bit_cast(f16x8, *(lds_u32x4 *)(addr)); }
    __device__ __forceinline__ void clear() { x = f16x8{}; }
};
template <> struct Operand<float> {
    bf16x8 s[3];
    struct Raw { float4 v[2]; };
    static __device__ __forceinline__ Raw fetch(const float *p)
    {
        return {{reinterpret_cast<const float4 *>(p)[0], reinterpret_cast<const float4 *>(p)[1]}};
    }
    __device__ __forceinline__ void set(const Raw &r)
    {
        const float v[8] = {r.v[0].x, r.v[0].y, r.v[0].z, r.v[0].w, r.v[1].x, r.v[1].y, r.v[1].z, r.v[1].w};
        split(v);
    }
    __device__ __forceinline__ void split(const float *v)
    {
        u32x4 out[3];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            uint32_t b[3][2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const float x = v[2 * e + u];
                b[0][u] = __float_as_uint(x) & 0xffff0000u;
                const float r = x - __uint_as_float(b[0][u]);
                b[1][u] = __float_as_uint(r) & 0xffff0000u;
                b[2][u] = __float_as_uint(r - __uint_as_float(b[1][u]));
            }
#pragma unroll
            for (int k = 0; k < 3; ++k) out[k][e] = __builtin_amdgcn_perm(b[k][1], b[k][0], 0x07060302u);
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) s[k] = __builtin_bit_cast(bf16x8, out[k]);
    }
    __device__ __forceinline__ void load(const float *p)
    {
        float v[8];
        load_row<8>(p, v);
        split(v);
    }
    __device__ __forceinline__ void load_lds(uint32_t addr)
    {
        float v[8];
#pragma unroll
        for (int c = 0; c < 8; c += 4) {
            const f32x4_t q = *(lds_float4_t *)(addr + 4 * c);
            v[c] = q[0]; v[c + 1] = q[1]; v[c + 2] = q[2]; v[c + 3] = q[3];
        }
        split(v);
    }
    __device__ __forceinline__ void clear()
    {
#pragma unroll
        for (int k = 0; k < 3; ++k) s[k] = __builtin_bit_cast(bf16x8, u32x4{});
    }
};
// a 32 x 32 result over 16 terms: A row lane % 32, B column lane % 32, terms 8 (lane / 32) + 0..7; the result's column
// is lane % 32, its rows 4 (lane / 32) + 8 (e / 4) + e % 4
__device__ __forceinline__ f32x16 mfma32(const Operand<__half> &a, const Operand<__half> &b, f32x16 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a.x, b.x, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma32(const Operand<float> &a, const Operand<float> &b, f32x16 c)
{
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.s[2], b.s[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.s[1], b.s[1], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.s[0], b.s[2], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.s[1], b.s[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.s[0], b.s[1], c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.s[0], b.s[0], c, 0, 0, 0);
}
__device__ __forceinline__ int mfma32_row(int lane, int e) { return 4 * (lane >> 5) + 8 * (e >> 2) + (e & 3); }

// A 16 x 16 result over 32 terms: A row lane % 16, B column lane % 16, terms 8 (lane / 16) + 0..7; the result's column
// is lane % 16, its rows 4 (lane / 16) + e.  B is a set of fp32 values: two fp16 numbers each beside fp16 (21 bits; A is
// exact), three bf16 numbers beside fp32.
template <typename T> struct Cells;
template <> struct Cells<__half> {
    f16x8 hi, lo;
    // rounded to one fp16 number each
    __device__ __forceinline__ void set_single(const float *v)
    {
#pragma unroll
        for (int e = 0; e < 8; ++e) hi[e] = static_cast<_Float16>(v[e]);
    }
    __device__ __forceinline__ void set(const float *v)
    {
        u32x4 h, l;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const auto p = __builtin_amdgcn_cvt_pkrtz(v[2 * e], v[2 * e + 1]);
            h[e] = __builtin_bit_cast(uint32_t, p);
            const float r0 = v[2 * e] - static_cast<float>(p[0]), r1 = v[2 * e + 1] - static_cast<float>(p[1]);
            l[e] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(r0, r1));
        }
        hi = __builtin_bit_cast(f16x8, h);
        lo = __builtin_bit_cast(f16x8, l);
    }
};
template <> struct Cells<float> {
    Operand<float> x;
    __device__ __forceinline__ void set(const float *v) { x.split(v); }
    __device__ __forceinline__ void set_single(const float *v) { x.split(v); }
};
__device__ __forceinline__ f32x4_t mfma16(const Operand<__half> &a, const Cells<__half> &b, f32x4_t c)
{
    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.x, b.lo, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a.x, b.hi, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4_t mfma16_single(const Operand<__half> &a, const Cells<__half> &b, f32x4_t c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a.x, b.hi, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4_t mfma16(const Operand<float> &a, const Cells<float> &b, f32x4_t c)
{
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.s[2], b.x.s[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.s[1], b.x.s[1], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.s[0], b.x.s[2], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.s[1], b.x.s[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.s[0], b.x.s[1], c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.s[0], b.x.s[0], c, 0, 0, 0);
}

__device__ __forceinline__ f32x4_t mfma16_single(const Operand<float> &a, const Cells<float> &b, f32x4_t c) { return mfma16(a, b, c); }

}  // namespace tile
}  // namespace s3d
