// Attention backward at head_dim 16: what is a sum over pairs, from dL and P of every (pair, head) (gfx950).  The mathematics
// is in attn_bwd.hip, the kernel that leaves the pairs in attn_tile_bwd.hip.
//
// A workgroup takes a strip of up to 16 voxels of windows of one size and all their pairs: as queries (dq, dTq, dTv) in one
// launch, as keys (dk, dv, dTk) in another.  It adds up the pairs' dL (and P) by table row into histograms over the rows of
// all axes at once, one column per voxel: integers on a fixed-point image, scaled per voxel by its sum of |dL|, so no order
// of additions shows in a result.  A histogram H then gives, by matrix products,
//     dT[row][c] += sum_columns H[row][column] x[column][c]   (x = q, dout, k: the three table gradients)
//     dx[column][c] += sum_rows H[row][column] T[row][c]      (dq from Tq, dk from Tk)
// and the pairs themselves, read as matrix operands, the rest of dq, dk and dv.  A voxel's pairs are all in its strip, so dq,
// dk and dv are stored once; table gradients stay in the registers of the wavefronts that make them for all strips of a
// workgroup, which works on one head, and meet in a reduction over the workgroups.
//
// Why strips of 16: the histograms of all axes fit LDS side by side (384 rows of 16 columns: 48 KB with P, 24 KB without), so
// a strip passes three barriers, where tiles of 64 x 64 pairs, an axis or two at a time, passed some fifty; a row of 16 cells
// is half of the banks or a quarter of them, and additions of lanes that hold 16 columns meet in none that costs (5.1 and
// 6.7 clocks a wavefront, 4.7 and 6.7 without any conflict; rows of 72 cells: 6.1 and 8.1).  Eight wavefronts and 128
// registers, two workgroups a CU: with four wavefronts and 168 registers, three workgroups, the table gradients and tables of
// a wavefront did not fit beside the rest, and 300 MB a call went to memory and back for it.  Registers are what is scarce:
// with fourteen of them spilled inside the loop the launch by query took 153 us, with none 138.
// Measured, 9 axes, 12,421 voxels in windows of 72, 12 heads, fp32 tables beside fp16 features: by query 138 us, by key 133
// (one kernel on 64 x 64 tiles: 523).  VALU 58 and 56 % of the time, LDS addressed 28 and 24 %, matrix pipe 14 and 12 %; a
// wavefront waits for half of its time, at the barriers and for the pairs and coordinates it reads.
#include "attn_strip.h"

#include <cmath>
#include <type_traits>

namespace s3d {
namespace tile {
namespace {

// dL and P in the gradients.
//  * Summed by table row they are integers in cells of 32 bits: P in units of 2^-28 (a query's weights sum to 1 but for
//    rounding, also of fp16 tables in a forward whose backward has fp32 ones; there is room for 16), dL in units of 2^(e-30),
//    2^e the least power above the sum of |dL| of its query (by key: of its key).  A cell keeps what fp32 would, and no order
//    of additions shows.
//  * They enter the products over 2^-kLiftP and 2^(e-kLift), the cells and the pairs' own alike: beside fp16 operands as two
//    fp16 numbers, 23 bits down to 2^-3 and units of 2^-24 below, that is 2^-35 of P and 2^-39 of the sum of |dL|.
//
// What is not finite stays in its window, though the products take all columns of a strip and all rows of a table, zeros
// among them: features and table entries that are not finite go into their operands as zeros.  The records kernel has left
// their pairs' dL as NaN or infinity, with dout their P as NaN as well, and so dq, dk and dv are what the sums over a window's
// pairs would be, but for channels beside the one that is not finite.  In the integers such a pair counts for nothing; the table rows it belongs to are marked and their gradients stored as NaN.  A P
// beyond 8 says that the statistics are not the forward's, and is treated alike.
constexpr float kFixWeight = 268435456.0f, kMostWeight = 8.0f;
constexpr int kFixGrad = 30;
template <typename TF> constexpr int kLift = sizeof(TF) == 2 ? 15 : 0;       // (fp32 features may be as large as fp32 is)
template <typename TF> constexpr float kLiftP = sizeof(TF) == 2 ? 2048.0f : 1.0f;
template <typename TF> constexpr float kWeightCell = kLiftP<TF> / kFixWeight;
template <typename TF> constexpr float kGradCell = (sizeof(TF) == 2 ? 32768.0f : 1.0f) / 1073741824.0f;
constexpr int kLiftFeature = 15;              // exponent of the strip's largest q or k in the table gradients

constexpr int kStripThreads = 512, kStripWaves = kStripThreads / 64;
constexpr int kStripReach = kStripThreads / kStrip;        // pairs of a voxel that a step of the workgroup takes
constexpr int kKept = 4;                                   // pairs that a thread keeps from the sum of |dL| on: an operand's terms

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
template <> struct Parts4<__half> {
    f16x4 hi, lo;
    template <bool kNearest = true> __device__ __forceinline__ void set(const float *v, float scale)
    {
        hi = to_half4(v[0] * scale, v[1] * scale, v[2] * scale, v[3] * scale);
        float r[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] = __builtin_fmaf(v[e], scale, -static_cast<float>(hi[e]));
        lo = to_half4(r[0], r[1], r[2], r[3]);
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
};
template <> struct Exact4<float> : Parts4<float> {
    __device__ __forceinline__ void set(const float *v) { Parts4<float>::set<true>(v, 1.0f); }
};

__device__ __forceinline__ f32x4_t mfma4(f16x4 a, f16x4 b, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x4_t mfma4(s16x4 a, s16x4 b, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0); }
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
template <typename T, typename TF> struct StripTable { using type = Exact4<TF>; };
template <> struct StripTable<float, __half> { using type = Parts4<__half>; };

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

// largest of a 16-lane group
template <typename V> __device__ __forceinline__ V max16(V v)
{
    auto step = [](V x, auto ctrl) {
        const int moved = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, true);
        const V o = __builtin_bit_cast(V, moved);
        return o > x ? o : x;
    };
    v = step(v, std::integral_constant<int, 0xB1>{});      // quad_perm [1,0,3,2]
    v = step(v, std::integral_constant<int, 0x4E>{});      // quad_perm [2,3,0,1]
    v = step(v, std::integral_constant<int, 0x141>{});     // row_half_mirror
    return step(v, std::integral_constant<int, 0x140>{});  // row_mirror
}

template <typename T, typename TF, int ND, bool kByKey>
__global__ __launch_bounds__(kStripThreads, 4) void strip_gradients_kernel(StripArgs b)
{
    using Table = typename StripTable<T, TF>::type;
    using Cell = Parts4<TF>;
    using Unit4 = typename std::conditional<sizeof(TF) == 2, f16x4, s16x4>::type;
    constexpr int kCellBytes = kByKey ? 4 : 8, kRowBytes = kStrip * kCellBytes;
    constexpr int kKinds = kByKey ? 1 : 2, kOwn = kOwnTiles<ND>;
    const AttnArgs &a = b.f;
    // cells [row][column]: dL, by query behind P; then parts of dx (by key: and dv), one a wavefront
    __shared__ __align__(16) uint32_t cells_s[kTiles<ND> * 16 * kStrip * kKinds];
    __shared__ __align__(16) float part_s[(kByKey ? 2 : 1) * kStripWaves * 256];
    __shared__ float sums_s[kStripWaves][kStrip], grad_s;
    __shared__ __align__(16) Exact4<TF> features_s[kKinds][64];        // q or k, dout of the strip's voxels
    __shared__ uint32_t marks_s[2 * kTiles<ND>], marked_s;
    // Pieces of the table's operands that wait in LDS, as many as leave room for two workgroups a CU (81,864 of 81,920 bytes by
    // query in fp32).  In registers they would not fit beside the rest, and a spilled operand comes back from memory behind the
    // pairs of the next strip, which are on their way then: loads return in order.
    constexpr int kParts = sizeof(Table) / 8, kPieces = kParts * kOwn;
    constexpr int kShared = kByKey || kPieces < kOwn + 2 ? kPieces : kOwn + 2, kKeptPieces = kPieces - kShared;
    struct TableParts { u32x2 part[kParts]; };
    __shared__ u32x2 table_s[kShared][kStripThreads];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int H = a.H, HD = H * D;
    const uint32_t stride = static_cast<uint32_t>(a.row_stride);       // of q, k, v
    const int h = static_cast<int>(blockIdx.x) % H;
    const int group = static_cast<int>(blockIdx.x) / H, groups = static_cast<int>(gridDim.x) / H;
    const int strips = b.list.total[1];
    if (group >= strips) return;       // its slot is not read
    const uint32_t cells = lds_address(cells_s);
    const int c16 = lane & 15, g4 = lane >> 4, reach0 = tid >> 4;
    const float nan = __int_as_float(0x7fc00000);

    const TF *gx = static_cast<const TF *>(kByKey ? a.k : a.q) + h * D, *gy = static_cast<const TF *>(kByKey ? a.q : a.k) + h * D;
    const TF *gd = static_cast<const TF *>(b.dout) + h * D;
    const float2 *records = b.records + static_cast<int64_t>(h) * b.pairs;
    const float scale_table = b.scales[h * 3 + (kByKey ? 1 : 0)];    // what a product with the table is multiplied by

    // The table by channel, for dx: rows 4 e + g4 of a tile, whose cells a read of the histogram takes side by side.  Tile
    // 8 i + wave is this wavefront's.
    u32x2 table[kKeptPieces > 0 ? kKeptPieces : 1];
    {
        const T *from = static_cast<const T *>(kByKey ? a.table_k : a.table_q) + h * D + c16;
#pragma unroll
        for (int i = 0; i < kOwn; ++i) {
            const int tile = i * kStripWaves + wave, axis = tile_axis(tile);
            float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (axis < ND && tile_row0(tile) < axis_rows<ND>(a, axis)) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int r = min(tile_row0(tile) + 4 * e + g4, axis_rows<ND>(a, axis) - 1);
                    const float x = to_float(from[static_cast<int64_t>(axis_base<ND>(a, axis) + r) * HD]);
                    v[e] = finite(x) ? x : 0.0f;
                }
            }
            Table x;
            if constexpr (std::is_same<Table, Parts4<__half>>::value) x.set(v, 1.0f / scale_table);
            else x.set(v);
            const TableParts parts = __builtin_bit_cast(TableParts, x);
#pragma unroll
            for (int k = 0; k < kParts; ++k) {
                const int piece = k * kOwn + i;
                if (piece < kKeptPieces) table[piece] = parts.part[k];
                else table_s[piece - kKeptPieces][tid] = parts.part[k];
            }
        }
    }
    Unit4 unit, identity;                    // for a tile's rows as the histogram is read, for rows in order
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if constexpr (sizeof(TF) == 2) {
            unit[e] = static_cast<_Float16>(4 * e + g4 == c16 ? 1.0f : 0.0f);
            identity[e] = static_cast<_Float16>(4 * g4 + e == c16 ? 1.0f : 0.0f);
        } else {
            unit[e] = static_cast<short>(4 * e + g4 == c16 ? 0x3f80 : 0);
            identity[e] = static_cast<short>(4 * g4 + e == c16 ? 0x3f80 : 0);
        }
    }
    f32x4_t grads[kKinds][kOwn];
#pragma unroll
    for (int kind = 0; kind < kKinds; ++kind)
#pragma unroll
        for (int i = 0; i < kOwn; ++i) grads[kind][i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    for (int t = tid; t < kTiles<ND> * 16 * kStrip * kKinds / 4; t += kStripThreads) reinterpret_cast<uint4 *>(cells_s)[t] = make_uint4(0, 0, 0, 0);
    if (tid < 2 * kTiles<ND>) marks_s[tid] = 0;
    if (tid == 0) marked_s = 0;
    bool incomplete = false;                 // a window did not fit the records

    // A strip's voxels, their features (channels 4 g4 .. of voxel c16) and the first of their pairs.  They are under way while
    // the strip before goes through its products.
    struct Ahead {
        int4 column;
        Raw4<TF> x;                          // (first wavefront: q or k; second one, by query: dout)
        float2 kept[kKept];
    } ahead;
    // pair with the window's j-th voxel: by query [key][query], by key likewise
    auto pair_at = [&](int4 column, int n) { return column.w < 0 ? 0 : column.w + (kByKey ? (column.x - column.z) * n : column.x - column.z); };
    auto pair_step = [&](int4 column, int n) { return column.w < 0 ? 0 : kByKey ? 1 : n; };
    // the first of a lane's four channels, in a form that the compiler does not add to the pointers outside of the loop: that
    // would keep two registers for each
    auto part4 = [&]() {
        uint32_t c = 4 * g4;
        asm volatile("" : "+v"(c));
        return c;
    };
    auto fetch = [&](int n) {
        if (wave < kKinds)
            ahead.x.load((wave == 0 ? gx : gd) + (static_cast<uint64_t>(static_cast<uint32_t>(ahead.column.y)) *
                                                  (wave == 0 ? stride : static_cast<uint32_t>(HD)) + part4()));
        const int first = pair_at(ahead.column, n), step = pair_step(ahead.column, n);
#pragma unroll
        for (int s = 0; s < kKept; ++s) ahead.kept[s] = records[first + min(reach0 + s * kStripReach, n - 1) * step];
    };
    int4 strip = b.list.strips[group];
    ahead.column = b.columns[group * kStrip + c16];
    fetch(__builtin_amdgcn_readfirstlane(strip.y));

    for (int u = group; u < strips; u += groups) {
        const int n = __builtin_amdgcn_readfirstlane(strip.y);
        const int col0 = __builtin_amdgcn_readfirstlane(strip.z), cols = __builtin_amdgcn_readfirstlane(strip.w);
        // window of a column or key (these are below 2^12; of a larger window it is the only one)
        const float inv_n = n > kCols ? 0.0f : 1.0f / static_cast<float>(n);
        auto window_of = [&](int x) { return static_cast<int>((static_cast<float>(x) + 0.5f) * inv_n); };
        // this lane's column
        const int4 column = ahead.column;
        const int own_window = window_of(col0 + min(c16, cols - 1));
        const bool there = c16 < cols, fits = column.w >= 0;
        incomplete = incomplete || !fits;
        const int pair0 = pair_at(column, n), step = pair_step(column, n);
        const int windows = __builtin_amdgcn_readfirstlane(window_of(col0 + cols - 1) + 1);
        const int own_row = column.y;
        // row of key c16 of a step's sixteen: those of the wavefront's pairs, in the order of the operands' terms (the columns
        // of the windows' voxels are side by side)
        const int32_t *rows = b.column_rows + (u * kStrip - col0);
        const int term = wave * (64 / kStrip) + (c16 >> 2) + (c16 & 3) * kStripReach;
        int key_row = rows[min(term, n - 1)];
        // the next strip
        const int u_next = min(u + groups, strips - 1);
        strip = b.list.strips[u_next];
        ahead.column = b.columns[u_next * kStrip + c16];

        // dL and P of this column's pair with a voxel
        auto settle = [&](float2 r, bool pair) {
            if (!fits || !(r.y <= kMostWeight)) r = make_float2(nan, nan);
            return pair ? r : make_float2(0.0f, 0.0f);
        };
        float2 kept[kKept];
        float sum = 0.0f, weights = 0.0f;
#pragma unroll
        for (int s = 0; s < kKept; ++s) {
            const bool pair = there & (reach0 + s * kStripReach < n);
            kept[s] = make_float2(pair ? ahead.kept[s].x : 0.0f, pair ? ahead.kept[s].y : 0.0f);
            sum += fabsf(kept[s].x);
            weights += kept[s].y;
        }
        if (__any(!fits | !finite(sum) | !(weights <= kMostWeight))) {
            sum = 0.0f;
#pragma unroll
            for (int s = 0; s < kKept; ++s) {
                kept[s] = settle(kept[s], there & (reach0 + s * kStripReach < n));
                sum += finite(kept[s].x) ? fabsf(kept[s].x) : 0.0f;
            }
        }
        for (int j0 = kKept * kStripReach; j0 < n; j0 += kStripReach) {
            const int j = j0 + reach0;
            const float2 r = settle(records[pair0 + min(j, n - 1) * step], there & (j < n));
            sum += finite(r.x) ? fabsf(r.x) : 0.0f;
        }
        sum += __shfl_xor(sum, 16);
        sum += __shfl_xor(sum, 32);
        if (lane < kStrip) sums_s[wave][c16] = sum;
        lds_barrier();
        sum = 0.0f;
#pragma unroll
        for (int w = 0; w < kStripWaves; ++w) sum += sums_s[w][c16];
        const int exponent = exponent_of(sum);

        float own[ND], other[2][ND];
        load_coords<ND>(a.n_coords + static_cast<int64_t>(column.x) * ND, own);
        const float *coords = a.n_coords + static_cast<int64_t>(column.z) * ND;
#pragma unroll
        for (int s = 0; s < 2; ++s) load_coords<ND>(coords + min(reach0 + s * kStripReach, n - 1) * ND, other[s]);
        // what the products of the pairs themselves start with, while the histograms are filled
        Raw4<TF> y, z;
        auto fetch_keys = [&](int row) {
            y.load(gy + (static_cast<uint64_t>(static_cast<uint32_t>(row)) * stride + part4()));
            if constexpr (kByKey) z.load(gd + (static_cast<uint64_t>(static_cast<uint32_t>(row)) * static_cast<uint32_t>(HD) + part4()));
        };
        fetch_keys(key_row);

        // ---- histograms
        const int up = kFixGrad - exponent;
        const uint32_t own_at = cells + c16 * kCellBytes;
        bool bad = false;
        auto add = [&](float2 r, const float *its) {
            const bool good = finite(r.x);
            bad = bad | !good;
            const int fix_l = good ? static_cast<int>(rintf(ldexpf(r.x, up))) : 0;
            const uint32_t fix_p = static_cast<uint32_t>(rintf(r.y * kFixWeight));
#pragma unroll
            for (int axis = 0; axis < ND; ++axis) {
                const uint32_t row = static_cast<uint32_t>(kByKey ? crse_row(its[axis], own[axis], b.half_rows[axis], b.upper[axis])
                                                                  : crse_row(own[axis], its[axis], b.half_rows[axis], b.upper[axis]));
                const uint32_t at = row * kRowBytes + own_at + axis_row0(axis) * kRowBytes;
                if constexpr (kByKey) lds_add(at, static_cast<uint32_t>(fix_l));
                else lds_add64(at, fix_p, fix_l);
            }
        };
        add(kept[0], other[0]);
        if (n > kStripReach) add(kept[1], other[1]);
        if (n > 2 * kStripReach) {
#pragma unroll
            for (int s = 2; s < kKept; ++s) load_coords<ND>(coords + min(reach0 + s * kStripReach, n - 1) * ND, other[s - 2]);
            add(kept[2], other[0]);
            if (n > 3 * kStripReach) add(kept[3], other[1]);
            for (int j0 = kKept * kStripReach; j0 < n; j0 += kStripReach) {
                const int j = j0 + reach0;
                load_coords<ND>(coords + min(j, n - 1) * ND, other[0]);
                add(settle(records[pair0 + min(j, n - 1) * step], there & (j < n)), other[0]);
            }
        }
        if (__any(bad)) {
            // rows of pairs that are not finite
            marked_s = 1;
#pragma unroll 1
            for (int j = reach0; j < n; j += kStripReach) {
                const float2 r = settle(records[pair0 + j * step], there);
                if (finite(r.x)) continue;
#pragma unroll 1
                for (int axis = 0; axis < ND; ++axis) {
                    const int rows_n = axis_rows<ND>(a, axis);
                    const float half_rows = static_cast<float>(rows_n / 2), upper = crse_upper(rows_n);
                    const float mine = a.n_coords[static_cast<int64_t>(column.x) * ND + axis], its = coords[j * ND + axis];
                    const int row = axis_row0(axis) + (kByKey ? crse_row(its, mine, half_rows, upper) : crse_row(mine, its, half_rows, upper));
                    atomicOr(&marks_s[row >> 4], 1u << (row & 15));
                    if (!finite(r.y)) atomicOr(&marks_s[kTiles<ND> + (row >> 4)], 1u << (row & 15));
                }
            }
        }

        // ---- the pairs themselves: dx += sum dL y, by key also dv += sum P dout, window by window; terms are the pairs that
        // the wavefront's threads hold
        f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};           // over 2^(exponent - kLift): [channel][column]
        f32x4_t acc_v = {0.0f, 0.0f, 0.0f, 0.0f};
        const float scale = power2(kLift<TF> - exponent);
        for (int w = 0; w < windows; ++w) {
            for (int j0 = 0; j0 < n; j0 += kKept * kStripReach) {
                if (w + j0 > 0) fetch_keys(rows[w * n + min(j0 + term, n - 1)]);
                f32x4_t ys = y.voxels(identity), zs = kByKey ? z.voxels(identity) : f32x4_t{};
                if (__any(!finite(fabsf(ys[0]) + fabsf(ys[1]) + fabsf(ys[2]) + fabsf(ys[3]) + fabsf(zs[0]) + fabsf(zs[1]) + fabsf(zs[2]) + fabsf(zs[3])))) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        ys[e] = finite(ys[e]) ? ys[e] : 0.0f;
                        zs[e] = finite(zs[e]) ? zs[e] : 0.0f;
                    }
                }
                float l[4], p[4];
                const float yv[4] = {ys[0], ys[1], ys[2], ys[3]}, zv[4] = {zs[0], zs[1], zs[2], zs[3]};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float2 r = kept[e];
                    if (j0 > 0) {
                        const int j = j0 + reach0 + e * kStripReach;
                        r = settle(records[pair0 + min(j, n - 1) * step], there & (j < n));
                    }
                    l[e] = own_window == w ? r.x : 0.0f;
                    p[e] = own_window == w ? r.y : 0.0f;
                }
                Exact4<TF> f;
                Cell c;
                f.set(yv);
                c.set(l, scale);
                acc = product(f, c, acc);
                if constexpr (kByKey) {
                    f.set(zv);
                    c.set(p, kLiftP<TF>);
                    acc_v = product(f, c, acc_v);
                }
            }
        }

        // features for the table gradients: q or k over the strip's largest exponent of a column, the largest value below 2^15,
        // as far as can be from where fp16 numbers lose bits
        if (wave < kKinds) {
            f32x4_t x = ahead.x.voxels(identity);
            if (__any(!finite(fabsf(x[0]) + fabsf(x[1]) + fabsf(x[2]) + fabsf(x[3])))) {
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = finite(x[e]) ? x[e] : 0.0f;
            }
            float v[4] = {x[0], x[1], x[2], x[3]};
            if (wave == 0) {
                const int top = __builtin_amdgcn_readfirstlane(max16(there ? exponent : -100));
                const float most16 = max16(fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3]))));
                float most = 0.0f;
#pragma unroll
                for (int g = 0; g < 4; ++g) most = fmaxf(most, __int_as_float(__builtin_amdgcn_readlane(__float_as_int(most16), 16 * g)));
                const int lift = kLiftFeature - exponent_of(most);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = ldexpf(x[e], __shfl(exponent, 4 * g4 + e) - top + lift);
                grad_s = power2(top - lift - kLift<TF>);
            }
            Exact4<TF> f;
            f.set(v);
            features_s[wave][lane] = f;
        }
        fetch(__builtin_amdgcn_readfirstlane(strip.y));
        lds_barrier();

        const Exact4<TF> feature = features_s[0][lane], feature_d = features_s[kKinds - 1][lane];
        const float grad = grad_s;
        // ---- matrix products of the histograms, which are cleared for the next strip (a tile without rows holds zeros)
        f32x4_t acc_t = {0.0f, 0.0f, 0.0f, 0.0f};         // ... the table's part, over scale_table as well
        const bool marked = __builtin_amdgcn_readfirstlane(marked_s) != 0;
        const uint32_t cell_at = cells + (wave * 16 + g4) * kRowBytes + c16 * kCellBytes;
#pragma unroll
        for (int i = 0; i < kOwn; ++i) {
            float l[4], p[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t at = cell_at + (i * kStripWaves * 16 + e * 4) * kRowBytes;
                if constexpr (kByKey) {
                    l[e] = static_cast<float>(static_cast<int>(lds_load_u32(at)));
                } else {
                    const float2 v = lds_load2(at);
                    p[e] = static_cast<float>(__float_as_uint(v.x));
                    l[e] = static_cast<float>(__float_as_int(v.y));
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t at = cell_at + (i * kStripWaves * 16 + e * 4) * kRowBytes;
                if constexpr (kByKey) lds_store_u32(at, 0u);
                else lds_store2(at, 0.0f, 0.0f);
            }
            Cell c;
            c.template set<sizeof(TF) == 2>(l, kGradCell<TF>);       // (the table's operand and the features are the nearest)
            TableParts parts;
#pragma unroll
            for (int k = 0; k < kParts; ++k) {
                const int piece = k * kOwn + i;
                parts.part[k] = piece < kKeptPieces ? table[piece < kKeptPieces ? piece : 0] : table_s[piece < kKeptPieces ? 0 : piece - kKeptPieces][tid];
            }
            acc_t = product(__builtin_bit_cast(Table, parts), c, acc_t);
            f32x4_t g = product(transposed(c, unit), feature, f32x4_t{});
#pragma unroll
            for (int e = 0; e < 4; ++e) grads[0][i][e] = fmaf(g[e], grad, grads[0][i][e]);
            if constexpr (!kByKey) {
                c.template set<sizeof(TF) == 2>(p, kWeightCell<TF>);
                g = product(transposed(c, unit), feature_d, f32x4_t{});
#pragma unroll
                for (int e = 0; e < 4; ++e) grads[kKinds - 1][i][e] = fmaf(g[e], 1.0f / kLiftP<TF>, grads[kKinds - 1][i][e]);
            }
        }
        if (marked) {
#pragma unroll
            for (int i = 0; i < kOwn; ++i)
#pragma unroll
                for (int kind = 0; kind < kKinds; ++kind)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (marks_s[kind * kTiles<ND> + i * kStripWaves + wave] >> (4 * g4 + e) & 1) grads[kind][i][e] = nan;
        }
        // ---- dx and dv: the wavefronts' parts, added up by the last two
        const float back = power2(exponent - kLift<TF>);
        f32x4_t dx;
#pragma unroll
        for (int e = 0; e < 4; ++e) dx[e] = fmaf(acc_t[e], scale_table, acc[e]) * back;
        *reinterpret_cast<f32x4_t *>(&part_s[(wave * 64 + lane) * 4]) = dx;
        if constexpr (kByKey) *reinterpret_cast<f32x4_t *>(&part_s[((kStripWaves + wave) * 64 + lane) * 4]) = acc_v;
        lds_barrier();
        const int which = kStripWaves - 1 - wave;
        if (which < (kByKey ? 2 : 1)) {
            // (eight parts in fp32 would add to an fp32 result's error what its own rounding is)
            using Sum = typename std::conditional<sizeof(TF) == 4, double, float>::type;
            Sum sums[4] = {0, 0, 0, 0};
            float o[4];
#pragma unroll
            for (int w = 0; w < kStripWaves; ++w) {
                const f32x4_t v = *reinterpret_cast<const f32x4_t *>(&part_s[((which * kStripWaves + w) * 64 + lane) * 4]);
#pragma unroll
                for (int e = 0; e < 4; ++e) sums[e] += v[e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = static_cast<float>(sums[e]) * (which > 0 ? 1.0f / kLiftP<TF> : 1.0f);
            if (there) store4(static_cast<TF *>(which > 0 ? b.dv : kByKey ? b.dk : b.dq) + static_cast<uint64_t>(static_cast<uint32_t>(own_row)) * b.grad_stride + h * D + part4(), o);
        }
    }
    // the workgroup's table gradients: [workgroup][kind][tile][lane][4 rows]
    const bool none = __syncthreads_or(incomplete);
    float *slot = b.slots + static_cast<int64_t>(blockIdx.x) * (kKinds * kTiles<ND> * 256);
#pragma unroll
    for (int kind = 0; kind < kKinds; ++kind) {
#pragma unroll
        for (int i = 0; i < kOwn; ++i) {
            const int tile = i * kStripWaves + wave;
            f32x4_t g = grads[kind][i];
            if (none) g = f32x4_t{nan, nan, nan, nan};
            *reinterpret_cast<f32x4_t *>(slot + (kind * kTiles<ND> + tile) * 256 + lane * 4) = g;
        }
    }
}

// The workgroups' table gradients, added up in the workgroups' order: a thread per word of a head's slot.
template <int ND>
__global__ __launch_bounds__(256) void strip_finish_kernel(StripArgs by_query, StripArgs by_key, int groups)
{
    const AttnArgs &a = by_query.f;
    constexpr int kWords = kTiles<ND> * 256;
    const int HD = a.H * D, t = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
    const int word = t % kWords, kind = t / kWords % 3, h = t / kWords / 3;          // dTq, dTv, dTk
    if (h >= a.H) return;
    const int e = word % 4, lane = word / 4 % 64, tile = word / 256;
    const int axis = tile_axis(tile), r = tile_row0(tile) + 4 * (lane / 16) + e;
    if (axis >= ND || r >= axis_rows<ND>(a, axis)) return;
    const int strips = by_query.list.total[1], kinds = kind < 2 ? 2 : 1;
    const int used = min(groups, strips);
    const float *from = (kind < 2 ? by_query.slots + kind * kWords : by_key.slots) + static_cast<int64_t>(h) * (kinds * kWords) + word;
    const int64_t step = static_cast<int64_t>(a.H) * (kinds * kWords);
    // (in 64 bits: a strip at a time, the parts have been rounded four times as often as by tiles of 64)
    double sum = 0.0;
#pragma unroll 8
    for (int g = 0; g < used; ++g) sum += from[g * step];
    (kind == 0 ? by_query.dtq : kind == 1 ? by_query.dtv : by_query.dtk)[static_cast<int64_t>(axis_base<ND>(a, axis) + r) * HD + h * D + lane % 16] = static_cast<float>(sum);
}

// workgroups per head: two per CU
int strip_groups(int H)
{
    const int most = 2 * device_cus();
    return most >= H ? most / H : 1;
}
size_t slot_bytes(int H, int nd, bool by_key)
{
    return align_up(sizeof(float) * 256 * static_cast<size_t>(strip_groups(H)) * H * tiles_of_axes(nd) * (by_key ? 1 : 2), 256);
}

template <typename T, typename TF, int ND>
int launch_strips(const StripArgs &b0, hipStream_t stream)
{
    StripArgs b = b0;
    for (int n = 0; n < ND; ++n) {
        b.half_rows[n] = static_cast<float>(b.f.rows[n] / 2);
        b.upper[n] = std::nextafterf(static_cast<float>(b.f.rows[n]), 0.0f);
    }
    StripArgs by_key = b;
    by_key.slots = b.slots + slot_bytes(b.f.H, ND, false) / sizeof(float);
    const int H = b.f.H, groups = strip_groups(H);
    hipLaunchKernelGGL((strip_gradients_kernel<T, TF, ND, false>), dim3(static_cast<unsigned>(groups * H)), dim3(kStripThreads), 0, stream, b);
    hipLaunchKernelGGL((strip_gradients_kernel<T, TF, ND, true>), dim3(static_cast<unsigned>(groups * H)), dim3(kStripThreads), 0, stream, by_key);
    const int64_t words = static_cast<int64_t>(3) * kTiles<ND> * 256 * H;
    hipLaunchKernelGGL(strip_finish_kernel<ND>, dim3(static_cast<unsigned>(ceil_div(words, 256))), dim3(256), 0, stream, b, by_key, groups);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

}  // namespace

size_t strip_slots_bytes(int H, int nd) { return slot_bytes(H, nd, false) + slot_bytes(H, nd, true); }

int launch_strip_gradients(const StripArgs &b, int dtype, hipStream_t stream)
{
#define S3D_CASE(NN)                                                                                           \
    if (b.f.nd == NN)                                                                                          \
        return dtype == S3D_DTYPE_F32   ? launch_strips<float, float, NN>(b, stream)                           \
               : dtype == S3D_DTYPE_F16 ? launch_strips<__half, __half, NN>(b, stream)                         \
                                        : launch_strips<float, __half, NN>(b, stream);
    S3D_CASE(3) S3D_CASE(6) S3D_CASE(9)
#undef S3D_CASE
    return fail(S3D_ERR_UNSUPPORTED, "s3d_attn_bwd: %d axes in the strip form", b.f.nd);
}

}  // namespace tile
}  // namespace s3d
