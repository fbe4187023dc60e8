// Pieces shared by the kernels on strips of 16 voxels (attn_strip_fwd.hip, attn_strip_records.hip, attn_strip_bwd.hip), and the
// interfaces between the backward's kernels at head_dim 16.
#pragma once

#include "attn_tile.h"

namespace s3d {
namespace tile {

// rows and first row of axis n: a choice among the kernel's arguments (an index would put them into scratch memory)
template <int ND> __device__ __forceinline__ int axis_rows(const AttnArgs &a, int axis)
{
    int r = a.rows[0];
#pragma unroll
    for (int n = 1; n < ND; ++n) r = axis == n ? a.rows[n] : r;
    return r;
}
template <int ND> __device__ __forceinline__ int axis_base(const AttnArgs &a, int axis)
{
    int r = a.base[0];
#pragma unroll
    for (int n = 1; n < ND; ++n) r = axis == n ? a.base[n] : r;
    return r;
}

constexpr int kStripThreads = 512, kStripWaves = kStripThreads / 64;

// 16-row tiles of the histograms: four to a position axis, two to a colour or normal axis, up to as many for each wavefront
// (with a branch around the last one, six axes took 60 registers more)
constexpr int tiles_of_axes(int nd) { return (12 + 2 * (nd - 3) + kStripWaves - 1) / kStripWaves * kStripWaves; }
template <int ND> constexpr int kTiles = tiles_of_axes(ND);
template <int ND> constexpr int kOwnTiles = kTiles<ND> / kStripWaves;
__host__ __device__ constexpr int axis_row0(int axis) { return axis < 3 ? axis * 64 : 192 + (axis - 3) * 32; }
__host__ __device__ constexpr int tile_axis(int tile) { return tile < 12 ? tile / 4 : 3 + (tile - 12) / 2; }
__host__ __device__ constexpr int tile_row0(int tile) { return (tile < 12 ? tile % 4 : tile % 2) * 16; }

// ---- matrix operands of 16 terms: lane % 16 is the row of A or the column of B, terms 4 (lane / 16) + 0..3 ----------------
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef int32_t i32x4_1 __attribute__((ext_vector_type(4), aligned(4)));

// numbers that are exact in the features' type
template <typename TF> struct Exact4;
// fp32 numbers: two fp16 numbers each beside fp16 features (of the numbers times a scale), three bf16 numbers beside fp32
template <typename TF> struct Parts4;
template <> struct Exact4<__half> {
    f16x4 x;
    __device__ __forceinline__ void set(const float *v)
    {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = static_cast<_Float16>(v[e]);
    }
};
__device__ __forceinline__ f16x4 to_half4(float a, float b, float c, float d)
{
    const f16x2 x = __builtin_convertvector(f32x2{a, b}, f16x2), y = __builtin_convertvector(f32x2{c, d}, f16x2);
    return __builtin_shufflevector(x, y, 0, 1, 2, 3);
}
// two numbers times a power of two as fp16 numbers, and what that leaves of them likewise (v_fma_mixlo_f16 and its like, one
// instruction a number in place of one and a half, take twice the time)
__device__ __forceinline__ uint32_t scaled_half2(float x, float y, float scale)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{x * scale, y * scale}), f16x2));
}
__device__ __forceinline__ uint32_t scaled_rest2(float x, float y, float scale, uint32_t h)
{
    const f16x2 t = __builtin_bit_cast(f16x2, h);
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{__builtin_fmaf(x, scale, -static_cast<float>(t[0])),
                                                                       __builtin_fmaf(y, scale, -static_cast<float>(t[1]))}), f16x2));
}
// a choice among the four numbers of an operand; of a number in both halves of a word
struct OneOfFour {
    u32x2 mask;
    __device__ __forceinline__ explicit OneOfFour(int at)
    {
        const uint32_t half = (at & 1) ? 0xffff0000u : 0xffffu;
        mask = {(at >> 1) == 0 ? half : 0u, (at >> 1) == 1 ? half : 0u};
    }
    __device__ __forceinline__ u32x2 of(uint32_t x) const { return {x & mask[0], x & mask[1]}; }
};
template <> struct Parts4<__half> {
    f16x4 hi, lo;
    template <bool kNearest = true> __device__ __forceinline__ void set(const float *v, float scale)
    {
        u32x2 h, l;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            h[e] = scaled_half2(v[2 * e], v[2 * e + 1], scale);
            l[e] = scaled_rest2(v[2 * e], v[2 * e + 1], scale, h[e]);
        }
        hi = __builtin_bit_cast(f16x4, h);
        lo = __builtin_bit_cast(f16x4, l);
    }
    // the number `at` (0..3) of the four, the others zero
    __device__ __forceinline__ void set_one(float v, float scale, const OneOfFour &at)
    {
        const uint32_t h = scaled_half2(v, v, scale), l = scaled_rest2(v, v, scale, h);
        hi = __builtin_bit_cast(f16x4, at.of(h));
        lo = __builtin_bit_cast(f16x4, at.of(l));
    }
};
template <> struct Parts4<float> {
    s16x4 s[3];
    template <bool kNearest = true> __device__ __forceinline__ void set(const float *v, float scale)
    {
        u32x2 out[3];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            f32x2 x = {v[2 * e] * scale, v[2 * e + 1] * scale};
            if constexpr (kNearest) {
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    out[k][e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(x, bf16x2));
                    if (k < 2) x -= f32x2{__uint_as_float(out[k][e] << 16), __uint_as_float(out[k][e] & 0xffff0000u)};
                }
            } else {
                uint32_t b[3][2];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    b[0][u] = __float_as_uint(x[u]) & 0xffff0000u;
                    const float r = x[u] - __uint_as_float(b[0][u]);
                    b[1][u] = __float_as_uint(r) & 0xffff0000u;
                    b[2][u] = __float_as_uint(r - __uint_as_float(b[1][u]));
                }
#pragma unroll
                for (int k = 0; k < 3; ++k) out[k][e] = __builtin_amdgcn_perm(b[k][1], b[k][0], 0x07060302u);
            }
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) s[k] = __builtin_bit_cast(s16x4, out[k]);
    }
    __device__ __forceinline__ void set_one(float v, float scale, const OneOfFour &at)
    {
        float x = v * scale;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const uint32_t b = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{x, x}), bf16x2));
            s[k] = __builtin_bit_cast(s16x4, at.of(b));
            if (k < 2) x -= __uint_as_float(b << 16);
        }
    }
};
template <> struct Exact4<float> : Parts4<float> {
    __device__ __forceinline__ void set(const float *v) { Parts4<float>::set<true>(v, 1.0f); }
};

__device__ __forceinline__ f32x4_t mfma4(f16x4 a, f16x4 b, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x4_t mfma4(s16x4 a, s16x4 b, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x4_t product(const Exact4<__half> &a, const Exact4<__half> &b, f32x4_t c) { return mfma4(a.x, b.x, c); }
__device__ __forceinline__ f32x4_t product(const Exact4<__half> &a, const Parts4<__half> &b, f32x4_t c) { return mfma4(a.x, b.hi, mfma4(a.x, b.lo, c)); }
__device__ __forceinline__ f32x4_t product(const Parts4<__half> &a, const Exact4<__half> &b, f32x4_t c) { return mfma4(a.hi, b.x, mfma4(a.lo, b.x, c)); }
__device__ __forceinline__ f32x4_t product(const Parts4<__half> &a, const Parts4<__half> &b, f32x4_t c)
{
    return mfma4(a.hi, b.hi, mfma4(a.hi, b.lo, mfma4(a.lo, b.hi, c)));
}
// (the six partial products meet before they join the sum, which is then rounded once a product)
__device__ __forceinline__ f32x4_t product(const Parts4<float> &a, const Parts4<float> &b, f32x4_t c)
{
    f32x4_t p = mfma4(a.s[2], b.s[0], f32x4_t{});
    p = mfma4(a.s[1], b.s[1], p);
    p = mfma4(a.s[0], b.s[2], p);
    p = mfma4(a.s[1], b.s[0], p);
    p = mfma4(a.s[0], b.s[1], p);
    p = mfma4(a.s[0], b.s[0], p);
#pragma unroll
    for (int e = 0; e < 4; ++e) c[e] += p[e];
    return c;
}
// the 16 x 16 matrix whose transpose x is, as an operand: multiplied by a permutation matrix `unit`, which is exact
__device__ __forceinline__ Parts4<__half> transposed(const Parts4<__half> &x, f16x4 unit)
{
    Parts4<__half> r;
    const f32x4_t hi = mfma4(x.hi, unit, f32x4_t{}), lo = mfma4(x.lo, unit, f32x4_t{});
    r.hi = to_half4(hi[0], hi[1], hi[2], hi[3]);
    r.lo = to_half4(lo[0], lo[1], lo[2], lo[3]);
    return r;
}
__device__ __forceinline__ Parts4<float> transposed(const Parts4<float> &x, s16x4 unit)
{
    Parts4<float> r;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const f32x4_t v = mfma4(x.s[k], unit, f32x4_t{});
        u32x2 out;
#pragma unroll
        for (int e = 0; e < 2; ++e) out[e] = __builtin_amdgcn_perm(__float_as_uint(v[2 * e + 1]), __float_as_uint(v[2 * e]), 0x07060302u);
        r.s[k] = __builtin_bit_cast(s16x4, out);
    }
    return r;
}
// Four channels of a voxel as loaded.  A lane that wants one channel of four voxels instead, as the products do, gets it from
// a product with the identity, which is exact (and all of a voxel's channels are NaN then where one is not finite).
template <typename TF> struct Raw4;
template <> struct Raw4<__half> {
    f16x4 x;
    __device__ __forceinline__ void load(const __half *p) { x = *reinterpret_cast<const f16x4 *>(p); }
    __device__ __forceinline__ f32x4_t voxels(f16x4 identity) const { return mfma4(x, identity, f32x4_t{}); }
};
template <> struct Raw4<float> {
    f32x4_t x;
    __device__ __forceinline__ void load(const float *p) { x = *reinterpret_cast<const f32x4_t *>(p); }
    __device__ __forceinline__ f32x4_t voxels(s16x4 identity) const
    {
        Parts4<float> y;
        const float v[4] = {x[0], x[1], x[2], x[3]};
        y.set<false>(v, 1.0f);
        return mfma4(y.s[0], identity, mfma4(y.s[1], identity, mfma4(y.s[2], identity, f32x4_t{})));
    }
};
// largest, and sum, over the four lanes of a column (lane % 16)
__device__ __forceinline__ float max_columns(float x)
{
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float sum_columns(float x)
{
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// coordinates of a voxel (rows of 3, 6 or 9 floats: aligned to a float)
template <int ND> __device__ __forceinline__ void load_coords(const float *p, float *c)
{
    typedef float f32x3_1 __attribute__((ext_vector_type(3), aligned(4)));
#pragma unroll
    for (int n = 0; n < ND; n += 3) {
        const f32x3_1 x = *reinterpret_cast<const f32x3_1 *>(p + n);
        c[n] = x[0]; c[n + 1] = x[1]; c[n + 2] = x[2];
    }
}

// a table as operands beside features of type TF
template <typename T, typename TF> struct StripTable { using type = Exact4<TF>; };
template <> struct StripTable<float, __half> { using type = Parts4<__half>; };

// ---- strips of single windows -----------------------------------------------------------------------------------------
// A window of n voxels is ceil(n / 16) strips of equal size.  A strip: first sorted position of the window, n, which of the
// window's strips it is, and the pairs (n^2) of the windows before it.
struct WindowStrips {
    const int32_t *total;
    const int4 *strips;
};
inline size_t window_strips_most(int64_t N, int64_t W) { return static_cast<size_t>(N > 0 ? N : 0) / kStrip + static_cast<size_t>(W > 0 ? W : 0); }

// By one workgroup, as the forward's list.
__device__ __forceinline__ void build_window_strips(const int32_t *__restrict__ w_sizes, const int32_t *__restrict__ w2n, int W,
                                                    int32_t *__restrict__ total, int4 *__restrict__ strips)
{
    __shared__ int at[kSizeBins];
    __shared__ long long wave_pairs[kListThreads / 64];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    place_strips<kListThreads>(w_sizes, W, total, at);
    long long before = 0;              // pairs of the windows of earlier rounds
    for (int w0 = 0; w0 < W; w0 += kListThreads) {
        const int w = w0 + t, n = w < W ? max(w_sizes[w], 0) : 0;
        const long long own = static_cast<long long>(n) * n;
        long long pairs = own;
        for (int off = 1; off < 64; off <<= 1) {
            const long long up = __shfl_up(pairs, off);
            if (lane >= off) pairs += up;
        }
        if (lane == 63) wave_pairs[wave] = pairs;
        __syncthreads();
        pairs += before - own;
        for (int v = 0; v < kListThreads / 64; ++v) {
            pairs += v < wave ? wave_pairs[v] : 0;
            before += wave_pairs[v];
        }
        if (n > 0) {
            const int count = strips_of(n), first = atomicAdd(&at[size_bin(n)], count), pos = w2n[w];
            // (a window that begins beyond 2^31 pairs does not fit any store)
            for (int q = 0; q < count; ++q) strips[first + q] = make_int4(pos, n, q, static_cast<int>(pairs < 0x7fffffffll ? pairs : 0x7fffffffll));
        }
        __syncthreads();
    }
}

// A strip with a block of at most kKeyBlock of its window's keys: what a workgroup works off at a time.
template <int kKeyBlock> struct StripItem {
    int pos0, n, first, cols, blocks, block, first_key, keys_n, pairs;
    __device__ __forceinline__ void set_block(int which)
    {
        const int size = (n + blocks - 1) / blocks;
        block = which;
        first_key = block * size;
        keys_n = min(size, n - first_key);
    }
    __device__ __forceinline__ void set(int4 s)
    {
        pos0 = __builtin_amdgcn_readfirstlane(s.x);
        n = __builtin_amdgcn_readfirstlane(s.y);
        pairs = __builtin_amdgcn_readfirstlane(s.w);
        const int count = strips_of(n), size = (n + count - 1) / count;
        first = __builtin_amdgcn_readfirstlane(s.z) * size;
        cols = min(size, n - first);
        blocks = (n + kKeyBlock - 1) / kKeyBlock;
        set_block(0);
    }
};
// lane `which` of each sixteen
__device__ __forceinline__ float of_sixteen(float value, int which)
{
    const int x = __float_as_int(value);
    // (row_newbcast; the lane is part of the instruction)
    switch (which) {
#define S3D_LANE(N) case N: return __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0x150 + N, 0xf, 0xf, true));
        S3D_LANE(0) S3D_LANE(1) S3D_LANE(2) S3D_LANE(3) S3D_LANE(4) S3D_LANE(5) S3D_LANE(6) S3D_LANE(7)
#undef S3D_LANE
    }
    return __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0x158, 0xf, 0xf, true));
}
typedef __attribute__((address_space(3))) f32x4_t lds_f32x4;

struct StripArgs {
    AttnArgs f;                 // shape, q, k, tables, index arrays, rows[] / base[]
    UnitList list;              // entries and strips
    const void *dout;
    const float2 *records;      // [H][pairs]: (dL, P) at pairs before the window + j n + i  (i, j: query, key inside the window)
    int64_t pairs;              // capacity of records per head; windows beyond it are not there
    const int4 *columns;        // [strip][column]: sorted position, row, window's first position, pairs before it (-1: beyond
                                // the records)
    const int32_t *column_rows; // [strip][column]: the rows alone
    const float *scales;        // [head][Tq, Tk, Tv]: what a product with the table's operand is multiplied by
    float *slots;               // [workgroup][kind][tile][lane][4]: table gradients as the products leave them, by query
    void *dq, *dk, *dv;
    uint32_t grad_stride;       // elements between rows of dq, dk, dv (of q, k, v: f.row_stride)
    float *dtq, *dtk, *dtv;
    float half_rows[kMaxAxes], upper[kMaxAxes];    // what crse_row takes (made here, they would take two vector registers an axis)
    float *key_slots;           // ... and by key
};
// The kernels that leave dL and P of every pair, at head_dim 16: on tiles (attn_tile_bwd.hip, fp32 and small windows) or strips
// (attn_strip_records.hip, fp16 features).
struct RecordsCall {
    AttnArgs f;                 // shape, q, k, v, tables, index arrays, rows[] / base[]
    UnitList list;              // entries and strips of the kernels that sum over pairs (and the units)
    const void *dout, *out;
    const float *stat_max, *stat_sum;
    float2 *records;            // [H][pairs]: (dL, P)
    int64_t pairs;              // capacity of records per head; windows beyond it are skipped
    int4 *strip_columns;        // see StripArgs
    int32_t *strip_rows;
    void *operands;             // the tables as matrix operands, and
    float *scales;              // [head][Tq, Tk, Tv] what a product with them is multiplied by
};
__device__ __forceinline__ bool window_fits(int before, int n, int64_t pairs)
{
    return static_cast<int64_t>(before) + static_cast<int64_t>(n) * n <= pairs;
}
size_t strip_records_bytes(int H, int nd, int64_t N, int64_t W);
int launch_strip_records(const RecordsCall &c, void *room, int dtype, hipStream_t stream);

size_t strip_slots_bytes(int H, int nd);
int launch_strip_gradients(const StripArgs &b, int dtype, hipStream_t stream);

// ---- head_dim 8: what the strips need beside the records of the pair sweep, whose launches of lists make it (attn_sweep.hip) ----
struct StripSetup {
    StripArgs b;
    int64_t *pos_base;          // [N]: at a window's first sorted position, the pairs of the windows before it
};

// The strip list (workgroup 0) and, for fp32 tables beside fp16 features, the scale of a head's operands of Tq and Tk.
template <bool kScales>
__device__ __forceinline__ void strip_setup(const StripArgs &b, int block)
{
    const AttnArgs &a = b.f;
    if (block == 0) {
        build_list(a.w_sizes, a.w2n, static_cast<int>(a.W), const_cast<int32_t *>(b.list.total), nullptr,
                   const_cast<int2 *>(b.list.entries), const_cast<int4 *>(b.list.strips));
        return;
    }
    const int job = block - 1, kind = job % 2, h = job / 2;
    float scale = 1.0f;
    if constexpr (kScales) {
        const float *table = static_cast<const float *>(kind == 0 ? a.table_q : a.table_k) + h * a.D;
        __shared__ int top_s;
        if (threadIdx.x == 0) top_s = 0;
        __syncthreads();
        float top = 0.0f;
        for (int t = threadIdx.x; t < a.total_rows * a.D; t += kListThreads) {
            const float x = table[static_cast<int64_t>(t / a.D) * (a.H * a.D) + t % a.D];
            top = fmaxf(top, finite(x) ? fabsf(x) : 0.0f);
        }
        atomicMax(&top_s, __float_as_int(top));
        __syncthreads();
        scale = power2(min(100, 14 - exponent_of(__int_as_float(top_s))));
    }
    if (threadIdx.x == 0) const_cast<float *>(b.scales)[h * 3 + kind] = 1.0f / scale;
}

// column t of the strips
__device__ __forceinline__ void strip_column(const StripSetup &s, int t)
{
    const StripArgs &b = s.b;
    const int u = t / kStrip, c = t % kStrip;
    if (u >= b.list.total[1]) return;
    const int4 strip = b.list.strips[u];
    const int col = strip.z + min(c, strip.w - 1), n = strip.y;
    const int2 entry = b.list.entries[strip.x + col / n];
    const int pos = entry.x + col % n, row = b.f.n2n ? b.f.n2n[pos] : pos;
    const bool fits = static_cast<int64_t>(entry.y) + static_cast<int64_t>(n) * n <= b.pairs;
    const_cast<int4 *>(b.columns)[t] = make_int4(pos, row, entry.x, fits ? entry.y : -1);
    const_cast<int32_t *>(b.column_rows)[t] = row;
    if (pos == entry.x) s.pos_base[pos] = entry.y;
}

}  // namespace tile
}  // namespace s3d
