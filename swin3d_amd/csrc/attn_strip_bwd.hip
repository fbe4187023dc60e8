// Attention backward at head_dim 16: what is a sum over pairs, from dL and P of every (pair, head) (gfx950).  The mathematics
// is in attn_bwd.hip, the kernels that leave the pairs in attn_strip_records.hip and attn_tile_bwd.hip.
//
// A workgroup takes a strip of up to 16 voxels of windows of one size and all their pairs: as queries (dq, dTq, dTv) in the
// first half of the launch, as keys (dk, dv, dTk) in the second (or in a launch each).  It adds up the pairs' dL (and P) by table row into histograms over the rows of
// all axes at once, one column per voxel: integers on a fixed-point image, scaled per voxel by its sum of |dL|, so no order
// of additions shows in a result.  A histogram H then gives, by matrix products,
//     dT[row][c] += sum_columns H[row][column] x[column][c]   (x = q, dout, k: the three table gradients)
//     dx[column][c] += sum_rows H[row][column] T[row][c]      (dq from Tq, dk from Tk)
// and the pairs themselves, read as matrix operands, the rest of dq, dk and dv.  A voxel's pairs are all in its strip, so dq,
// dk and dv are stored once; table gradients stay in the registers of the wavefronts that make them for all strips of a
// workgroup, which works on one head, and meet in a reduction over the workgroups.  At head_dim 8 the pairs come from a sweep
// (attn_sweep.hip, launch_attn_bwd_records), and q (or k) and dout share the sixteen channels of the products.
//
// Why strips of 16: the histograms of all axes fit LDS side by side (384 rows of 16 columns: 48 KB with P, 24 KB without), so
// a strip passes two barriers, where tiles of 64 x 64 pairs, an axis or two at a time, passed some fifty; a row of 16 cells
// is half of the banks or a quarter of them, and additions of lanes that hold 16 columns meet in none that costs (5.1 and
// 6.7 clocks a wavefront, 4.7 and 6.7 without any conflict; rows of 72 cells: 6.1 and 8.1).  Eight wavefronts and 128
// registers, two workgroups a CU: with four wavefronts and 168 registers, three workgroups, the table gradients and tables of
// a wavefront did not fit beside the rest, and 300 MB a call went to memory and back for it.  Registers are what is scarce:
// with fourteen of them spilled inside the loop the launch by query took 153 us, with none 138.
// Measured, 9 axes, 12,421 voxels in windows of 72, 12 heads, fp32 tables beside fp16 features: by query 128 us, by key 125 in a launch each
// (one kernel on 64 x 64 tiles: 523; with a third barrier before the histograms and coordinates asked for behind it, 138 and
// 133).  head_dim 8, 199,327 voxels in windows of 26, 6 heads, fp16: 543 and 502 us (in one launch 990), where the sweeps' own sums and the kernels
// of the table gradients took 1510.  What bounds them is VALU issue, 73 % of the time: at head_dim 8 some 300 to 350
// instructions a wavefront and strip, a third of them the histograms' conversion into operands, 45 the nine rows of a pair.
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
//  * They enter the products over 2^-kLiftP and 2^(e-kLift), beside fp16 operands as two fp16 numbers, 23 bits down to 2^-3 and
//    units of 2^-24 below: 2^-35 of P, and 2^-39 of the sum of |dL|, in the cells and for the pairs themselves.  The pairs' own P
//    by key, whose sum is nowhere near 1 where no query gives the key much weight, are over a unit that follows the largest P
//    that the wavefront holds of the key: 2^-39 of that.  (Over 2^-kLiftP, dv of a key whose weights are 2^-26 had ten bits.
//    0.6 % of a backward of 199,327 voxels at head_dim 8, 0.2 % of one of 12,421 at 16.)
//
// What is not finite stays in its window, though the products take all columns of a strip and all rows of a table, zeros
// among them: features and table entries that are not finite go into their operands as zeros, with all channels of their
// voxel.  The records kernel has left their pairs' dL as NaN or infinity, and so dq and dk are what the sums over a window's pairs
// would be, but for channels beside the one that is not finite.  In the integers such a pair counts for nothing; the table rows
// it belongs to are marked and their gradients stored as NaN.  A P beyond 8 says that the statistics are not the forward's, and
// is treated alike.  A dout that is not finite leaves P alone.  At head_dim 16 the records kernel makes NaN of it all the same,
// and so of all channels of dv and dTv; at 8 it does where no channel of dout is finite; elsewhere a workgroup goes
// through its strips with such a dL once more and adds up, pair by pair, dv of the windows and what the voxel gives dTv.  (Every dout
// infinite, 199,327 voxels x 6, fp16: 2.4 ms where the call takes 1.5, 8 more pair by pair.)
constexpr float kFixWeight = 268435456.0f, kMostWeight = 8.0f;
constexpr int kFixGrad = 30;
template <typename TF> constexpr int kLift = sizeof(TF) == 2 ? 15 : 0;       // (fp32 features may be as large as fp32 is)
template <typename TF> constexpr float kLiftP = sizeof(TF) == 2 ? 2048.0f : 1.0f;
template <typename TF> constexpr float kWeightCell = kLiftP<TF> / kFixWeight;
template <typename TF> constexpr float kGradCell = (sizeof(TF) == 2 ? 32768.0f : 1.0f) / 1073741824.0f;
// What P enters a product over, by the largest there is: a power of two, by which the largest P is below 2^kLift; and its inverse.
template <typename TF> __device__ __forceinline__ float weight_unit(float most)
{
    if (kLift<TF> == 0) return 1.0f;
    constexpr uint32_t kLeast = 47u << 23, kUp = static_cast<uint32_t>(kLift<TF> - 1) << 23;      // 2^-80
    return __uint_as_float(max(__float_as_uint(most) & 0x7f800000u, kLeast) - kUp);
}
__device__ __forceinline__ float inverse_power2(float x) { return __uint_as_float(0x7f000000u - __float_as_uint(x)); }
constexpr int kLiftFeature = 15;              // exponent of the strip's largest q or k in the table gradients

constexpr int kStripReach = kStripThreads / kStrip;        // pairs of a voxel that a step of the workgroup takes
constexpr int kKept = 4;                                   // pairs that a thread keeps from the sum of |dL| on: an operand's terms

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

// One launch for the sums by query and by key, or one each (strip_gradients_apart_kernel)
template <typename TF, int C> constexpr bool kOneLaunch = C == 16 || sizeof(TF) == 2;

// What the products of head_dim 8 leave out, in the strips that have a dL that is not finite beside a P that is: P dout of the voxels whose dout is
// not finite in some channel, pair by pair.  By key dv of their windows is added up again; by query what they give dTv joins the
// workgroup's slot.  (It takes its arguments from where the launch put them: what is kept for it through the loop over strips comes
// back from memory there, 1 % of a call in fp32.)
constexpr int kMetWords = 64;                              // a bit for each of a workgroup's strips (modulo 2048)
template <typename TF, int ND, bool kByKey>
__device__ __forceinline__ void add_left_out(float *shared, const uint32_t *strips_met)
{
    constexpr int C = 8;
    const void *at_args = (const void *)__builtin_amdgcn_kernarg_segment_ptr();
    constexpr bool kHalf = kOneLaunch<TF, C>;
    const int blocks = static_cast<int>(gridDim.x) / (kHalf ? 2 : 1);
    int tid = threadIdx.x, block = static_cast<int>(blockIdx.x) - (kByKey && kHalf ? blocks : 0);
    asm volatile("" : "+s"(at_args), "+v"(tid), "+s"(block));
    const StripArgs &b = *static_cast<const StripArgs *>(at_args);
    const AttnArgs &a = b.f;
    const int H = a.H, HD = H * C, h = block % H, group = block / H, groups = blocks / H, strips = b.list.total[1];
    const int c16 = tid & 15, channel = tid >> 4 & 7, part = tid >> 7;
    const TF *gd = static_cast<const TF *>(b.dout) + h * C;
    const float2 *records = b.records + static_cast<int64_t>(h) * b.pairs;
    auto met = [&](int u) {
        const int turn = u / groups;
        return (__builtin_amdgcn_readfirstlane(strips_met[turn / 32 % kMetWords]) >> (turn & 31) & 1) != 0;
    };
    auto row_of = [&](int pos) { return static_cast<int64_t>(a.n2n ? a.n2n[pos] : pos) * HD; };
    auto any_bad = [&](const TF *dout) {
        float x[C];
        load_row<C>(dout, x);
        bool bad = false;
#pragma unroll
        for (int c = 0; c < C; ++c) bad = bad || !finite(x[c]);
        return bad;
    };
    __threadfence();      // (what is stored may be stored again, by other lanes)
    __syncthreads();
    if constexpr (kByKey) {
        // a thread for a column, a channel and every fourth query
        for (int u = group; u < strips; u += groups) {
            if (!met(u)) continue;
            const int4 strip = b.list.strips[u], column = b.columns[u * kStrip + c16];
            const int n = strip.y;
            const bool there = c16 < strip.w && column.w >= 0;
            const float2 *from = records + (there ? column.w + (column.x - column.z) * n : 0);
            float sum = 0.0f;
            bool bad = false;
            for (int i = part; there && i < n; i += 4) {
                const TF *dout = gd + row_of(column.z + i);
                bad = bad || any_bad(dout);
                sum = fmaf(from[i].y, to_float(dout[channel]), sum);
            }
            shared[tid] = sum;
            shared[kStripThreads + tid] = bad ? 1.0f : 0.0f;
            __syncthreads();
            bad = false;
            sum = 0.0f;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                sum += shared[(tid & 127) + 128 * p];
                bad = bad || shared[kStripThreads + (tid & 127) + 128 * p] > 0.0f;
            }
            TF *to = static_cast<TF *>(b.dv) + static_cast<uint64_t>(static_cast<uint32_t>(column.y)) * b.grad_stride + h * C + channel;
            if (there && bad && part == 0) {
                if constexpr (sizeof(TF) == 2) *to = __float2half_rn(sum);
                else *to = sum;
            }
            __syncthreads();
        }
    } else {
        // Table rows times channels, four times, in the place of the cells, which are zeros; a thread for an axis, a channel and
        // every fourth column, which has its words to itself.
        constexpr int kWords = kTiles<ND> * 16 * C;
        static_assert(4 * kWords == kTiles<ND> * 16 * kStrip * 2, "the cells, of P and dL");
        const int axis = tid >> 3 & 15, c = tid & 7;
        for (int u = group; u < strips; u += groups) {
            if (!met(u)) continue;
            const int4 strip = b.list.strips[u];
            const int n = strip.y;
            for (int at = part; axis < ND && at < strip.w; at += 4) {
                const int4 column = b.columns[u * kStrip + at];
                const TF *dout = gd + row_of(column.x);
                if (column.w < 0 || !any_bad(dout)) continue;
                const int rows_n = axis_rows<ND>(a, axis);
                const float x = to_float(dout[c]), half_rows = static_cast<float>(rows_n / 2), upper = crse_upper(rows_n);
                const float mine = a.n_coords[static_cast<int64_t>(column.x) * ND + axis];
                const float2 *from = records + column.w + column.x - column.z;
#pragma unroll 4
                for (int j = 0; j < n; ++j) {
                    const int r = crse_row(mine, a.n_coords[static_cast<int64_t>(column.z + j) * ND + axis], half_rows, upper);
                    float *to = shared + part * kWords + (axis_row0(axis) + r) * C + c;
                    *to = fmaf(from[static_cast<int64_t>(j) * n].y, x, *to);
                }
            }
        }
        __syncthreads();
        if (c16 < C) return;       // (the columns of dTq)
        float *slot = b.slots + static_cast<int64_t>(block) * (kTiles<ND> * 256);
        for (int tile = tid >> 6; tile < kTiles<ND>; tile += kStripWaves) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float *from = shared + (tile * 16 + 4 * (tid >> 4 & 3) + e) * C + c16 - C;
                slot[tile * 256 + (tid & 63) * 4 + e] += (from[0] + from[kWords]) + (from[2 * kWords] + from[3 * kWords]);
            }
        }
    }
}

// C channels a head: 16, or 8 (packed): q or k and dout then share the sixteen channels of an operand, dTq and dTv the sixteen
// columns of a product, and dk and dv its rows.
template <typename T, typename TF, int ND, bool kByKey, int C> struct StripForm {
    using Table = typename StripTable<T, TF>::type;
    static constexpr bool kPacked = C == 8;
    static constexpr int kKinds = kByKey ? 1 : 2, kOwn = kOwnTiles<ND>;
    static constexpr int kSets = kPacked ? 1 : kKinds;        // of features, and of table gradients
    static constexpr int kParts = kByKey && !kPacked ? 2 : 1; // of dx: dk and dv
    // Pieces of the table's operands that wait in LDS, as many as leave room for two workgroups a CU (81,864 of 81,920 bytes by
    // query in fp32).  In registers they would not fit beside the rest, and a spilled operand comes back from memory behind the
    // pairs of the next strip, which are on their way then: loads return in order.
    static constexpr int kTableParts = sizeof(Table) / 8, kPieces = kTableParts * kOwn;
    static constexpr int kShared = kByKey || kPieces < kOwn + 2 ? kPieces : kOwn + 2, kKeptPieces = kPieces - kShared;
    using Cells = uint32_t[kTiles<ND> * 16 * kStrip * kKinds];      // [row][column]: dL, by query behind P
    using Sums = float[kParts * kStripWaves * 256];                 // parts of dx (by key: and dv), one a wavefront
    using Features = Exact4<TF>[kSets][64];                         // q or k, dout of the strip's voxels
    using Pieces = u32x2[kShared][kStripThreads];
    using AbsSums = float[kStripWaves][kStrip];
    using Marks = uint32_t[2 * kTiles<ND>];
    using Met = uint32_t[kPacked ? kMetWords : 1];
    struct Lds {
        alignas(16) Cells cells;
        alignas(16) Sums part;
        alignas(16) Features features;
        Pieces table;
        AbsSums sums;
        float grad;
        Marks marks;
        uint32_t marked;
        Met met;
    };
    static_assert(sizeof(Lds) <= 80 * 1024, "two workgroups a CU");
};

// A member of what two forms share in LDS, or (kApart) an array by itself
template <bool kApart, typename A> using Own = typename std::conditional<kApart, A, char>::type;
template <bool kApart, typename L, typename A> __device__ __forceinline__ A &in_lds(Own<kApart, A> &own, L *lds, A L::*member)
{
    if constexpr (kApart) return own;
    else return lds->*member;
}

// (The arguments by value: by reference the same code was 2 % slower at eight channels.)
template <typename T, typename TF, int ND, bool kByKey, int C, bool kApart>
__device__ __forceinline__ void strip_gradients(StripArgs b, typename StripForm<T, TF, ND, kByKey, C>::Lds *lds, int block, int blocks)
{
    using Form = StripForm<T, TF, ND, kByKey, C>;
    using Table = typename Form::Table;
    using Cell = Parts4<TF>;
    using Unit4 = typename std::conditional<sizeof(TF) == 2, f16x4, s16x4>::type;
    constexpr int kCellBytes = kByKey ? 4 : 8, kRowBytes = kStrip * kCellBytes;
    constexpr int kKinds = Form::kKinds, kOwn = Form::kOwn, kSets = Form::kSets, kParts = Form::kParts;
    constexpr int kTableParts = Form::kTableParts, kKeptPieces = Form::kKeptPieces;
    constexpr bool kPacked = Form::kPacked;
    // Windows whose keys are one step's in a form of their own: most are at the level of eight channels.  (At sixteen few are,
    // and the second form costs the other one registers.)
    auto one_step = [](int n) { return kPacked && n <= kStripReach; };
    const AttnArgs &a = b.f;
    __shared__ __align__(16) Own<kApart, typename Form::Cells> own_cells;
    __shared__ __align__(16) Own<kApart, typename Form::Sums> own_part;
    __shared__ Own<kApart, typename Form::AbsSums> own_sums;
    __shared__ Own<kApart, float> own_grad;
    __shared__ __align__(16) Own<kApart, typename Form::Features> own_features;
    __shared__ Own<kApart, typename Form::Marks> own_marks;
    __shared__ Own<kApart, uint32_t> own_marked;
    __shared__ Own<kApart, typename Form::Met> own_met;
    __shared__ Own<kApart, typename Form::Pieces> own_table;
    auto &cells_s = in_lds<kApart>(own_cells, lds, &Form::Lds::cells);
    auto &part_s = in_lds<kApart>(own_part, lds, &Form::Lds::part);
    auto &sums_s = in_lds<kApart>(own_sums, lds, &Form::Lds::sums);
    auto &grad_s = in_lds<kApart>(own_grad, lds, &Form::Lds::grad);
    auto &features_s = in_lds<kApart>(own_features, lds, &Form::Lds::features);
    auto &marks_s = in_lds<kApart>(own_marks, lds, &Form::Lds::marks);
    auto &marked_s = in_lds<kApart>(own_marked, lds, &Form::Lds::marked);
    auto &met_s = in_lds<kApart>(own_met, lds, &Form::Lds::met);
    auto &table_s = in_lds<kApart>(own_table, lds, &Form::Lds::table);
    struct TableParts { u32x2 part[kTableParts]; };
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int H = a.H, HD = H * C;
    const uint32_t stride = static_cast<uint32_t>(a.row_stride);       // of q, k, v
    const int h = block % H, group = block / H, groups = blocks / H;
    const int strips = b.list.total[1];
    if (group >= strips) return;       // its slot is not read
    const uint32_t cells = lds_address(cells_s);
    const int c16 = lane & 15, g4 = lane >> 4, reach0 = tid >> 4;
    const float nan = __int_as_float(0x7fc00000);

    const TF *gx = static_cast<const TF *>(kByKey ? a.k : a.q) + h * C, *gy = static_cast<const TF *>(kByKey ? a.q : a.k) + h * C;
    const TF *gd = static_cast<const TF *>(b.dout) + h * C;
    const float2 *records = b.records + static_cast<int64_t>(h) * b.pairs;
    const float scale_table = b.scales[h * 3 + (kByKey ? 1 : 0)];    // what a product with the table is multiplied by

    // The table by channel, for dx: rows 4 e + g4 of a tile, whose cells a read of the histogram takes side by side.  Tile
    // 8 i + wave is this wavefront's.
    u32x2 table[kKeptPieces > 0 ? kKeptPieces : 1];
    {
        const T *from = static_cast<const T *>(kByKey ? a.table_k : a.table_q) + h * C + c16 % C;
#pragma unroll
        for (int i = 0; i < kOwn; ++i) {
            const int tile = i * kStripWaves + wave, axis = tile_axis(tile);
            float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (axis < ND && tile_row0(tile) < axis_rows<ND>(a, axis)) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int r = min(tile_row0(tile) + 4 * e + g4, axis_rows<ND>(a, axis) - 1);
                    const float x = to_float(from[static_cast<int64_t>(axis_base<ND>(a, axis) + r) * HD]);
                    v[e] = finite(x) && c16 < C ? x : 0.0f;
                }
            }
            Table x;
            if constexpr (std::is_same<Table, Parts4<__half>>::value) x.set(v, 1.0f / scale_table);
            else x.set(v);
            const TableParts parts = __builtin_bit_cast(TableParts, x);
#pragma unroll
            for (int k = 0; k < kTableParts; ++k) {
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
    f32x4_t grads[kSets][kOwn];
#pragma unroll
    for (int kind = 0; kind < kSets; ++kind)
#pragma unroll
        for (int i = 0; i < kOwn; ++i) grads[kind][i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    for (int t = tid; t < kTiles<ND> * 16 * kStrip * kKinds / 4; t += kStripThreads) reinterpret_cast<uint4 *>(cells_s)[t] = make_uint4(0, 0, 0, 0);
    if (tid < 2 * kTiles<ND>) marks_s[tid] = 0;
    if (tid == 0) marked_s = 0;
    if (kPacked && tid < kMetWords) met_s[tid] = 0;
    bool incomplete = false;                 // a window did not fit the records

    // A strip's voxels, their features (channels 4 g4 .. of voxel c16) and the first of their pairs.  They are under way while
    // the strip before goes through its products.
    struct Ahead {
        int4 column;
        Raw4<TF> x;                          // (first wavefront: q or k; second one, by query: dout; packed the first both)
        float2 kept[kKept];
    } ahead;
    // pair with the window's j-th voxel: by query [key][query], by key likewise
    auto pair_at = [&](int4 column, int n) { return column.w < 0 ? 0 : column.w + (kByKey ? (column.x - column.z) * n : column.x - column.z); };
    auto pair_step = [&](int4 column, int n) { return column.w < 0 ? 0 : kByKey ? 1 : n; };
    // the first of a lane's four channels, in a form that the compiler does not add to the pointers outside of the loop: that
    // would keep two registers for each
    auto part4 = [&]() {
        uint32_t c = 4 * g4 % C;
        asm volatile("" : "+v"(c));
        return c;
    };
    // four channels of a row of x or, `other`, of dout
    auto load4 = [&](Raw4<TF> &r, const TF *x, int row, bool other) {
        r.load((other ? gd : x) + (static_cast<uint64_t>(static_cast<uint32_t>(row)) * (other ? static_cast<uint32_t>(HD) : stride) + part4()));
    };
    auto fetch = [&](int n) {
        if (wave < kSets) load4(ahead.x, gx, ahead.column.y, kPacked ? !kByKey && g4 >= 2 : wave > 0);
        const int first = pair_at(ahead.column, n), step = pair_step(ahead.column, n);
        ahead.kept[0] = records[first + min(reach0, n - 1) * step];
        if (!one_step(n)) {
#pragma unroll
            for (int s = 1; s < kKept; ++s) ahead.kept[s] = records[first + min(reach0 + s * kStripReach, n - 1) * step];
        }
    };
    // dL and P of a column's pair with a voxel
    auto settle = [&](float2 r, bool fits, bool pair) {
        if (!fits || !(r.y <= kMostWeight)) r = make_float2(nan, nan);
        return pair ? r : make_float2(0.0f, 0.0f);
    };
    // A strip is opened while the one before waits for its last barrier: its pairs come to rest, their sum of |dL| goes to the
    // others, and what else its threads read is asked for.
    int n, col0, cols, key_row;
    int4 column;
    float2 kept[kKept];
    float own[ND], other[2][ND];
    // (the key of c16 / 4 and, of a window with more than a step's, the term c16 % 4)
    const int key = wave * (64 / kStrip) + (c16 >> 2), term = key + (c16 & 3) * kStripReach;
    // window of a column or key, of the strip's (these are below 2^12; of a larger window it is the only one)
    auto window_of = [](int n, int x) {
        const float inv = __builtin_amdgcn_rcpf(static_cast<float>(n));      // (an error of 2^-22 does not reach a whole number: n is at most 64)
        return static_cast<int>((static_cast<float>(x) + 0.5f) * (n > kCols ? 0.0f : inv));
    };
    auto last_window = [&](int n, int col0, int cols) { return __builtin_amdgcn_readfirstlane(window_of(n, col0 + cols - 1)); };
    auto open = [&](int u, int4 strip) {
        n = __builtin_amdgcn_readfirstlane(strip.y);
        col0 = __builtin_amdgcn_readfirstlane(strip.z);
        cols = __builtin_amdgcn_readfirstlane(strip.w);
        column = ahead.column;
        const bool there = c16 < cols, fits = column.w >= 0;
        incomplete = incomplete || !fits;
        const int pair0 = pair_at(column, n), step = pair_step(column, n);
        float sum = 0.0f, weights = 0.0f;
        auto keep = [&](int s) {
            const bool pair = there & (reach0 + s * kStripReach < n);
            kept[s] = make_float2(pair ? ahead.kept[s].x : 0.0f, pair ? ahead.kept[s].y : 0.0f);
            sum += fabsf(kept[s].x);
            weights += kept[s].y;
        };
        keep(0);
        if (!one_step(n)) {
#pragma unroll
            for (int s = 1; s < kKept; ++s) keep(s);
        }
        if (__any(!fits | !finite(sum) | !(weights <= kMostWeight))) {
            sum = 0.0f;
#pragma unroll
            for (int s = 0; s < kKept; ++s) {
                if (s > 0 && one_step(n)) break;
                kept[s] = settle(kept[s], fits, there & (reach0 + s * kStripReach < n));
                sum += finite(kept[s].x) ? fabsf(kept[s].x) : 0.0f;
            }
        }
        for (int j0 = kKept * kStripReach; j0 < n; j0 += kStripReach) {
            const int j = j0 + reach0;
            const float2 r = settle(records[pair0 + min(j, n - 1) * step], fits, there & (j < n));
            sum += finite(r.x) ? fabsf(r.x) : 0.0f;
        }
        sum = sum_columns(sum);
        if (lane < kStrip) sums_s[wave][c16] = sum;
        // row of key c16 of a step's sixteen: those of the wavefront's pairs, in the order of the operands' terms (the columns
        // of the windows' voxels are side by side)
        key_row = b.column_rows[u * kStrip - col0 + (!one_step(n) ? min(term, n - 1) : min(c16 & 3, last_window(n, col0, cols)) * n + min(key, n - 1))];
        load_coords<ND>(a.n_coords + static_cast<int64_t>(column.x) * ND, own);
        const float *coords = a.n_coords + static_cast<int64_t>(column.z) * ND;
        load_coords<ND>(coords + min(reach0, n - 1) * ND, other[0]);
        if (!one_step(n)) load_coords<ND>(coords + min(reach0 + kStripReach, n - 1) * ND, other[1]);
    };
    int4 strip = b.list.strips[group];
    ahead.column = b.columns[group * kStrip + c16];
    fetch(__builtin_amdgcn_readfirstlane(strip.y));
    open(group, strip);
    lds_barrier();

    for (int u = group; u < strips; u += groups) {
        // this lane's column
        const int own_window = window_of(n, col0 + min(c16, cols - 1));
        const bool there = c16 < cols, fits = column.w >= 0;
        const int pair0 = pair_at(column, n), step = pair_step(column, n);
        const int windows = last_window(n, col0, cols) + 1;
        const int own_row = column.y;
        const int32_t *rows = b.column_rows + (u * kStrip - col0);
        const float *coords = a.n_coords + static_cast<int64_t>(column.z) * ND;
        // the next strip
        const int u_next = min(u + groups, strips - 1);
        strip = b.list.strips[u_next];
        ahead.column = b.columns[u_next * kStrip + c16];

        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < kStripWaves; w += 4) sum += sums_s[w + g4][c16];
        sum = sum_columns(sum);
        const int exponent = exponent_of(sum);
        // what the products of the pairs themselves start with, while the histograms are filled
        Raw4<TF> y, z;
        auto fetch_keys = [&](int row) {
            load4(y, gy, row, kPacked && kByKey && g4 >= 2);
            if constexpr (kByKey && !kPacked) load4(z, gd, row, true);
        };
        fetch_keys(key_row);

        // ---- histograms
        const int up = kFixGrad - exponent;
        const uint32_t own_at = cells + c16 * kCellBytes;
        // (in a form to which the compiler adds an axis' first row as the instruction's offset: it would keep nine sums otherwise)
        auto cell_of = [](uint32_t row, uint32_t at) {
            uint32_t r;
            asm("v_lshl_add_u32 %0, %1, %2, %3" : "=v"(r) : "v"(row), "n"(kByKey ? 6 : 7), "v"(at));
            return r;
        };
        static_assert(kRowBytes == (kByKey ? 64 : 128), "a shift");
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
                const uint32_t at = cell_of(row, own_at), first = axis_row0(axis) * kRowBytes;
                if constexpr (kByKey) lds_add(at + first, static_cast<uint32_t>(fix_l));
                else lds_add64(at + first, fix_p, fix_l);
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
                add(settle(records[pair0 + min(j, n - 1) * step], fits, there & (j < n)), other[0]);
            }
        }
        if (__any(bad)) {
            // rows of pairs that are not finite
            marked_s = 1;
#pragma unroll 1
            for (int j = reach0; j < n; j += kStripReach) {
                const float2 r = settle(records[pair0 + j * step], fits, there);
                if (finite(r.x)) continue;
                if (kPacked && finite(r.y)) atomicOr(&met_s[u / groups / 32 % kMetWords], 1u << (u / groups & 31));
                const bool weight = !finite(r.y);
                int begin = 0;
                if constexpr (ND == 3) asm volatile("" : "+s"(begin));      // (a loop all the same: coordinates kept for it take registers)
#pragma unroll 1
                for (int first = begin; first < ND; first += 3) {
                    float mine[3], its[3];
                    load_coords<3>(a.n_coords + static_cast<int64_t>(column.x) * ND + first, mine);
                    load_coords<3>(coords + j * ND + first, its);
#pragma unroll
                    for (int e = 0; e < 3; ++e) {
                        const int axis = first + e, rows_n = axis_rows<ND>(a, axis);
                        const float half_rows = static_cast<float>(rows_n / 2), upper = crse_upper(rows_n);
                        const int row = axis_row0(axis) + (kByKey ? crse_row(its[e], mine[e], half_rows, upper) : crse_row(mine[e], its[e], half_rows, upper));
                        const uint32_t bit = 1u << (row & 15);
                        // (most have been marked by then)
                        if (!(marks_s[row >> 4] & bit)) atomicOr(&marks_s[row >> 4], bit);
                        if (weight && !(marks_s[kTiles<ND> + (row >> 4)] & bit)) atomicOr(&marks_s[kTiles<ND> + (row >> 4)], bit);
                    }
                }
            }
        }

        // ---- the pairs themselves: dx += sum dL y, by key also dv += sum P dout, window by window; terms are the pairs that
        // the wavefront's threads hold
        f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};           // over 2^(exponent - kLift): [channel][column]
        f32x4_t acc_v = {0.0f, 0.0f, 0.0f, 0.0f};
        const float scale = power2(kLift<TF> - exponent);
        // by key: P over unit_p, and so acc_v
        auto unit_of = [](float most) { return kLift<TF> > 0 ? weight_unit<TF>(max_columns(most)) : 1.0f; };
        float unit_p = 1.0f;
        if constexpr (kByKey) unit_p = unit_of(one_step(n) ? kept[0].y : fmaxf(fmaxf(kept[0].y, kept[1].y), fmaxf(kept[2].y, kept[3].y)));
        // a step's features, [voxel][channel]; what is not finite as zeros
        auto voxels_of = [&](Exact4<TF> &f, Exact4<TF> &fz) {
            f32x4_t ys = y.voxels(identity), zs{};
            if constexpr (kByKey && !kPacked) zs = z.voxels(identity);
            if (__any(!finite(fabsf(ys[0]) + fabsf(ys[1]) + fabsf(ys[2]) + fabsf(ys[3]) + fabsf(zs[0]) + fabsf(zs[1]) + fabsf(zs[2]) + fabsf(zs[3])))) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    ys[e] = finite(ys[e]) ? ys[e] : 0.0f;
                    zs[e] = finite(zs[e]) ? zs[e] : 0.0f;
                }
            }
            const float yv[4] = {ys[0], ys[1], ys[2], ys[3]}, zv[4] = {zs[0], zs[1], zs[2], zs[3]};
            f.set(yv);
            if constexpr (kByKey && !kPacked) fz.set(zv);
            else fz = f;
        };
        // windows of a step: a term of the four is the key's of its window, a column's pair in that of its own
        for (int w0 = 0; one_step(n) && w0 < windows; w0 += 4) {
            if (w0 > 0) fetch_keys(rows[min(w0 + (c16 & 3), windows - 1) * n + min(key, n - 1)]);
            Exact4<TF> f, fz;
            voxels_of(f, fz);
            const OneOfFour window(own_window - w0);
            Cell c;
            c.set_one(kept[0].x, scale, window);
            acc = product(f, c, acc);
            if constexpr (kByKey) {
                c.set_one(kept[0].y, inverse_power2(unit_p), window);
                acc_v = product(fz, c, acc_v);
            }
        }
        for (int w = 0; !one_step(n) && w < windows; ++w) {
            for (int j0 = 0; j0 < n; j0 += kKept * kStripReach) {
                if (w + j0 > 0) fetch_keys(rows[w * n + min(j0 + term, n - 1)]);
                float l[4], p[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float2 r = kept[e];
                    if (j0 > 0) {
                        const int j = j0 + reach0 + e * kStripReach;
                        r = settle(records[pair0 + min(j, n - 1) * step], fits, there & (j < n));
                    }
                    l[e] = own_window == w ? r.x : 0.0f;
                    p[e] = own_window == w ? r.y : 0.0f;
                }
                Exact4<TF> f, fz;
                Cell c;
                voxels_of(f, fz);
                c.set(l, scale);
                acc = product(f, c, acc);
                if constexpr (kByKey) {
                    if (kLift<TF> > 0 && j0 > 0) {
                        const float most = fmaxf(unit_p, unit_of(fmaxf(fmaxf(p[0], p[1]), fmaxf(p[2], p[3]))));
                        const float less = unit_p * inverse_power2(most);
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc_v[e] *= less;
                        unit_p = most;
                    }
                    c.set(p, inverse_power2(unit_p));
                    acc_v = product(fz, c, acc_v);
                }
            }
        }

        // features for the table gradients: q or k over the strip's largest exponent of a column, the largest value below 2^15,
        // as far as can be from where fp16 numbers lose bits
        if (wave < kSets) {
            f32x4_t x = ahead.x.voxels(identity);
            if (__any(!finite(fabsf(x[0]) + fabsf(x[1]) + fabsf(x[2]) + fabsf(x[3])))) {
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = finite(x[e]) ? x[e] : 0.0f;
            }
            float v[4] = {x[0], x[1], x[2], x[3]};
            const bool lifted = c16 < C || kByKey;         // (dout is not)
            if (wave == 0) {
                const int top = __builtin_amdgcn_readfirstlane(max16(there ? exponent : -100));
                const float most16 = max16(lifted ? fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3]))) : 0.0f);
                float most = 0.0f;
#pragma unroll
                for (int g = 0; g < 4; ++g) most = fmaxf(most, __int_as_float(__builtin_amdgcn_readlane(__float_as_int(most16), 16 * g)));
                const int lift = kLiftFeature - exponent_of(most);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int up = __shfl(exponent, 4 * g4 + e) - top + lift;
                    v[e] = ldexpf(x[e], lifted ? up : 0);
                }
                grad_s = power2(top - lift - kLift<TF>);
            }
            Exact4<TF> f;
            f.set(v);
            features_s[wave][lane] = f;
        }
        fetch(__builtin_amdgcn_readfirstlane(strip.y));
        lds_barrier();

        Exact4<TF> feature = features_s[0][lane], feature_d = features_s[kSets - 1][lane];
        const float grad = kPacked && !kByKey && c16 >= C ? 1.0f / kLiftP<TF> : grad_s;
        if constexpr (kPacked && !kByKey) {
            // the columns of dTq, and of dTv
            if (c16 < C) feature_d = Exact4<TF>{};
            else feature = Exact4<TF>{};
        }
        // ---- matrix products of the histograms, which are cleared for the next strip (a tile without rows holds zeros)
        f32x4_t acc_t = {0.0f, 0.0f, 0.0f, 0.0f};         // ... the table's part, over scale_table as well
        const bool marked = __builtin_amdgcn_readfirstlane(marked_s) != 0;
        const uint32_t cell_at = cells + (wave * 16 + g4) * kRowBytes + c16 * kCellBytes;
#pragma unroll
        for (int i = 0; i < kOwn; ++i) {
            uint32_t cell_l[4], cell_p[4], any = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t at = cell_at + (i * kStripWaves * 16 + e * 4) * kRowBytes;
                if constexpr (kByKey) {
                    cell_l[e] = lds_load_u32(at);
                    cell_p[e] = 0;
                } else {
                    const float2 v = lds_load2(at);
                    cell_p[e] = __float_as_uint(v.x);
                    cell_l[e] = __float_as_uint(v.y);
                }
                any |= cell_l[e] | cell_p[e];
            }
            if (!__any(any != 0)) continue;
            float l[4], p[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                l[e] = static_cast<float>(static_cast<int>(cell_l[e]));
                p[e] = static_cast<float>(cell_p[e]);
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
            for (int k = 0; k < kTableParts; ++k) {
                const int piece = k * kOwn + i;
                parts.part[k] = piece < kKeptPieces ? table[piece < kKeptPieces ? piece : 0] : table_s[piece < kKeptPieces ? 0 : piece - kKeptPieces][tid];
            }
            acc_t = product(__builtin_bit_cast(Table, parts), c, acc_t);
            f32x4_t g = product(transposed(c, unit), feature, f32x4_t{});
            if constexpr (!kByKey && kPacked) {
                c.template set<sizeof(TF) == 2>(p, kWeightCell<TF>);
                g = product(transposed(c, unit), feature_d, g);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) grads[0][i][e] = fmaf(g[e], grad, grads[0][i][e]);
            if constexpr (!kByKey && !kPacked) {
                c.template set<sizeof(TF) == 2>(p, kWeightCell<TF>);
                g = product(transposed(c, unit), feature_d, f32x4_t{});
#pragma unroll
                for (int e = 0; e < 4; ++e) grads[kSets - 1][i][e] = fmaf(g[e], 1.0f / kLiftP<TF>, grads[kSets - 1][i][e]);
            }
        }
        if (marked) {
#pragma unroll
            for (int i = 0; i < kOwn; ++i)
#pragma unroll
                for (int set = 0; set < kSets; ++set) {
                    const int kind = kPacked && !kByKey ? c16 / C : set;
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (marks_s[kind * kTiles<ND> + i * kStripWaves + wave] >> (4 * g4 + e) & 1) grads[set][i][e] = nan;
                }
        }
        // ---- dx and dv: the wavefronts' parts, added up by the last two
        const float back = power2(exponent - kLift<TF>);
        f32x4_t dx;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            dx[e] = fmaf(acc_t[e], scale_table, acc[e]) * back;
            if constexpr (kByKey) acc_v[e] *= unit_p;
            if constexpr (kPacked && kByKey) dx[e] = g4 < 2 ? dx[e] : acc_v[e];
        }
        *reinterpret_cast<f32x4_t *>(&part_s[(wave * 64 + lane) * 4]) = dx;
        if constexpr (kParts > 1) *reinterpret_cast<f32x4_t *>(&part_s[((kStripWaves + wave) * 64 + lane) * 4]) = acc_v;
        __builtin_amdgcn_sched_barrier(0);
        open(u_next, strip);
        __builtin_amdgcn_sched_barrier(0);
        lds_barrier();
        const int which = kStripWaves - 1 - wave;
        if (which < kParts) {
            // (eight parts in fp32 would add to an fp32 result's error what its own rounding is)
            using Sum = typename std::conditional<sizeof(TF) == 4, double, float>::type;
            Sum sums[4] = {0, 0, 0, 0};
            float o[4];
#pragma unroll 2
            for (int w = 0; w < kStripWaves; ++w) {
                const f32x4_t v = *reinterpret_cast<const f32x4_t *>(&part_s[((which * kStripWaves + w) * 64 + lane) * 4]);
#pragma unroll
                for (int e = 0; e < 4; ++e) sums[e] += v[e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = static_cast<float>(sums[e]);
            const bool dv = kPacked ? kByKey && g4 >= 2 : which > 0;
            if (there && (!kPacked || kByKey || g4 < 2))
                store4(static_cast<TF *>(dv ? b.dv : kByKey ? b.dk : b.dq) + static_cast<uint64_t>(static_cast<uint32_t>(own_row)) * b.grad_stride + h * C + part4(), o);
        }
    }
    const bool none = __syncthreads_or(incomplete);
    // the workgroup's table gradients: [workgroup][kind][tile][lane][4 rows]
    float *slot = (kByKey ? b.key_slots : b.slots) + static_cast<int64_t>(block) * (kSets * kTiles<ND> * 256);
#pragma unroll
    for (int kind = 0; kind < kSets; ++kind) {
#pragma unroll
        for (int i = 0; i < kOwn; ++i) {
            const int tile = i * kStripWaves + wave;
            f32x4_t g = grads[kind][i];
            if (none) g = f32x4_t{nan, nan, nan, nan};
            *reinterpret_cast<f32x4_t *>(slot + (kind * kTiles<ND> + tile) * 256 + lane * 4) = g;
        }
    }
    if constexpr (kPacked) {
        if (__builtin_amdgcn_readfirstlane(marked_s) != 0) add_left_out<TF, ND, kByKey>(kByKey ? part_s : reinterpret_cast<float *>(cells_s), met_s);
    }
}

// By query, and behind that by key in the places that are free by then: in a launch each the second waits for the longest
// workgroup of the first.  A call, forward included, us, before / so: 12,421 voxels x 12 of 16 615 / 606, 3,105 x 24 397 / 389, 49,682 x 6 979 /
// 968, in fp32 972 / 963 and 1418 / 1402; 199,327 x 6 of 8 1548 / 1531, 60,000 with six axes 490 / 480, with three the same.
template <typename T, typename TF, int ND, int C>
__global__ __launch_bounds__(kStripThreads, 4) void strip_gradients_kernel(StripArgs b)
{
    using Query = typename StripForm<T, TF, ND, false, C>::Lds;
    using Key = typename StripForm<T, TF, ND, true, C>::Lds;
    __shared__ __align__(16) char lds[sizeof(Query) > sizeof(Key) ? sizeof(Query) : sizeof(Key)];
    const int blocks = static_cast<int>(gridDim.x) / 2, block = static_cast<int>(blockIdx.x);
    if (block < blocks) strip_gradients<T, TF, ND, false, C, false>(b, reinterpret_cast<Query *>(lds), block, blocks);
    else strip_gradients<T, TF, ND, true, C, false>(b, reinterpret_cast<Key *>(lds), block - blocks, blocks);
}

// fp32 at head_dim 8 in a launch each, and what is in LDS as arrays by themselves: as parts of one block the compiler takes more
// registers than there are (spilled with six axes 11 by one kernel, 7 and 1 by two with a block each, 5 and none so).  A call, forward
// included, us, by one kernel / so: windows of 60, 100,003 voxels x 6 1810 / 1786, with nine axes 2118 / 2091; of 26, 20,000 and 40,000
// the same.
template <typename T, typename TF, int ND, bool kByKey, int C>
__global__ __launch_bounds__(kStripThreads, 4) void strip_gradients_apart_kernel(StripArgs b)
{
    strip_gradients<T, TF, ND, kByKey, C, true>(b, nullptr, static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x));
}

// The workgroups' table gradients, added up in the workgroups' order: a thread per word of a head's slot.
template <int ND, int C>
__global__ __launch_bounds__(256) void strip_finish_kernel(StripArgs b, int groups)
{
    const AttnArgs &a = b.f;
    constexpr int kWords = kTiles<ND> * 256, kSets = C == 8 ? 1 : 2;
    const int HD = a.H * C, t = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
    const int word = t % kWords, set = t / kWords % (kSets + 1), h = t / kWords / (kSets + 1);       // by query, then by key
    if (h >= a.H) return;
    const int e = word % 4, lane = word / 4 % 64, tile = word / 256;
    const int axis = tile_axis(tile), r = tile_row0(tile) + 4 * (lane / 16) + e;
    if (axis >= ND || r >= axis_rows<ND>(a, axis)) return;
    const int kind = set == kSets ? 2 : C == 8 ? lane % 16 / C : set;                              // dTq, dTv, dTk
    if (kind == 2 && lane % 16 >= C) return;
    const int strips = b.list.total[1], sets = set < kSets ? kSets : 1;
    const int used = min(groups, strips);
    const float *from = (set < kSets ? b.slots + set * kWords : b.key_slots) + static_cast<int64_t>(h) * (sets * kWords) + word;
    const int64_t step = static_cast<int64_t>(a.H) * (sets * kWords);
    // (in 64 bits: a strip at a time, the parts have been rounded four times as often as by tiles of 64)
    double sum = 0.0;
#pragma unroll 8
    for (int g = 0; g < used; ++g) sum += from[g * step];
    (kind == 0 ? b.dtq : kind == 1 ? b.dtv : b.dtk)[static_cast<int64_t>(axis_base<ND>(a, axis) + r) * HD + h * C + lane % C] = static_cast<float>(sum);
}

// workgroups per head: two per CU
int strip_groups(int H)
{
    const int most = 2 * device_cus();
    return most >= H ? most / H : 1;
}
size_t slot_bytes(int H, int nd, int sets)
{
    return align_up(sizeof(float) * 256 * static_cast<size_t>(strip_groups(H)) * H * tiles_of_axes(nd) * sets, 256);
}

template <typename T, typename TF, int ND, int C>
int launch_strips(const StripArgs &b0, hipStream_t stream)
{
    StripArgs b = b0;
    for (int n = 0; n < ND; ++n) {
        b.half_rows[n] = static_cast<float>(b.f.rows[n] / 2);
        b.upper[n] = std::nextafterf(static_cast<float>(b.f.rows[n]), 0.0f);
    }
    constexpr int kSets = C == 8 ? 1 : 2;
    b.key_slots = b.slots + slot_bytes(b.f.H, ND, kSets) / sizeof(float);
    const int H = b.f.H, groups = strip_groups(H);
    const unsigned blocks = static_cast<unsigned>(groups * H);
    if constexpr (kOneLaunch<TF, C>) {
        hipLaunchKernelGGL((strip_gradients_kernel<T, TF, ND, C>), dim3(2 * blocks), dim3(kStripThreads), 0, stream, b);
    } else {
        hipLaunchKernelGGL((strip_gradients_apart_kernel<T, TF, ND, false, C>), dim3(blocks), dim3(kStripThreads), 0, stream, b);
        hipLaunchKernelGGL((strip_gradients_apart_kernel<T, TF, ND, true, C>), dim3(blocks), dim3(kStripThreads), 0, stream, b);
    }
    const int64_t words = static_cast<int64_t>(kSets + 1) * kTiles<ND> * 256 * H;
    hipLaunchKernelGGL((strip_finish_kernel<ND, C>), dim3(static_cast<unsigned>(ceil_div(words, 256))), dim3(256), 0, stream, b, groups);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

}  // namespace

size_t strip_slots_bytes(int H, int nd) { return slot_bytes(H, nd, 2) + slot_bytes(H, nd, 1); }

int launch_strip_gradients(const StripArgs &b, int dtype, hipStream_t stream)
{
#define S3D_CASE(NN, CC)                                                                                       \
    if (b.f.nd == NN && b.f.D == CC)                                                                           \
        return dtype == S3D_DTYPE_F32   ? launch_strips<float, float, NN, CC>(b, stream)                       \
               : dtype == S3D_DTYPE_F16 ? launch_strips<__half, __half, NN, CC>(b, stream)                     \
                                        : launch_strips<float, __half, NN, CC>(b, stream);
    S3D_CASE(3, 16) S3D_CASE(6, 16) S3D_CASE(9, 16)
    S3D_CASE(3, 8) S3D_CASE(6, 8) S3D_CASE(9, 8)
#undef S3D_CASE
    return fail(S3D_ERR_UNSUPPORTED, "s3d_attn_bwd: %d axes in the strip form", b.f.nd);
}

}  // namespace tile

// Where the strips serve a backward at head_dim 8; elsewhere the pair sweeps with the table-gradient kernels, whose cost follows
// the pairs and table rows where a strip's follows its voxels.  Strips over those, forward left out:
//   fp16 features, 9 axes: 0.60 to 0.89 (windows of 2 to 60 voxels, 60,000 to 250,000 voxels of 6 heads), 6 axes 0.61 to 0.94;
//     3 axes 0.61 to 0.98 at 60,000, 1.07 at 250,000 in windows of 26
//   fp32 (three parts a number, twice the products): windows of 60 0.71 to 0.75; of 26, on scans with 6 axes, forward included,
//     0.83 at 20,000 voxels, 0.91 at 40,000, 0.98 at 60,000, 1.01 to 1.05 beyond, with 9 axes 0.77 at 20,000, 0.95 to 0.99 at
//     360,000 to 2,000,000 (voxel, head); with random signals, whose histograms have no empty rows, 1.02 to 1.08 at 360,000 and
//     1.13 to 1.23 at 1,500,000
constexpr int64_t kStripMeanWindow = 40, kStripVoxelHeads = 600000, kStripVoxelHeadsFloat = 250000;

bool attn_strip8_applies(const int32_t *rows, int nd, int D, int dtype, int64_t N, int64_t W, int H, int64_t pairs, size_t room)
{
    if (D != 8 || pairs <= 0 || pairs >= (int64_t(1) << 31) || !rows_fit_tiles(rows, nd) || attn_strip8_bytes(H, nd, N, W) > room) return false;
    if (N >= kStripMeanWindow * W) return true;
    return dtype == S3D_DTYPE_F32 ? N * H <= kStripVoxelHeadsFloat : nd > 3 || N * H <= kStripVoxelHeads;
}

// slots | list | strips | columns | their rows | scales
size_t attn_strip8_bytes(int H, int nd, int64_t N, int64_t W)
{
    return tile::slot_bytes(H, nd, 1) * 2 + tile::list_bytes(N, W) + tile::strips_bytes(N) + tile::strip_columns_bytes(N) +
           align_up(sizeof(float) * 3 * static_cast<size_t>(H), 256);
}

int launch_attn_strip8(const BwdPairArgs &p, float *dtq, float *dtk, float *dtv, void *room, int dtype, hipStream_t stream)
{
    using namespace tile;
    const AttnArgs &a = p.f;
    StripSetup s{};
    StripArgs &g = s.b;
    g.f = a;
    char *at = static_cast<char *>(room);
    g.slots = reinterpret_cast<float *>(at);
    at += slot_bytes(a.H, a.nd, 1) * 2;
    g.list = list_at(at, a.N, a.W);
    at += list_bytes(a.N, a.W);
    g.list.strips = reinterpret_cast<const int4 *>(at);
    at += strips_bytes(a.N);
    g.columns = reinterpret_cast<const int4 *>(at);
    g.column_rows = reinterpret_cast<const int32_t *>(g.columns + kStrip * list_max_strips(a.N));
    at += strip_columns_bytes(a.N);
    g.scales = reinterpret_cast<const float *>(at);
    g.dout = p.dout;
    g.records = p.pd;
    g.pairs = p.pairs;
    g.dq = p.dq; g.dk = p.dk; g.dv = p.dv;
    g.grad_stride = static_cast<uint32_t>(p.grad_stride);
    g.dtq = dtq; g.dtk = dtk; g.dtv = dtv;
    s.pos_base = const_cast<int64_t *>(p.pos_base);
    if (int rc = launch_attn_bwd_records(p, s, dtype, stream)) return rc;
    return launch_strip_gradients(g, dtype, stream);
}

}  // namespace s3d
