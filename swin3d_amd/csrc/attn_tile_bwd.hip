// Attention backward at head_dim 16 on tiles of up to 64 queries by 64 keys of a head (gfx950); the mathematics is in
// attn_bwd.hip.  Two kernels on the forward's unit list:
//
//  * tile_records_kernel: the logits again and dP = dout_i . (v_j + Tv(i,j)), as the forward's tile kernel makes its
//    logits: the products of the tile's queries (q with Tq, dout with Tv) and keys (k with Tk) with all rows of an axis
//    come from the matrix pipe and stay in LDS, where every pair picks its three.  It leaves dL and P of every (pair,
//    head): 8 bytes at [head][pairs before the window + j n + i].
//  * tile_gradients_kernel: everything that is a sum over pairs.  Per axis the pairs' dL and P are added up by table row
//    into histograms over the rows, one column per query (dL and P in one 64-bit cell) and one per key (dL): integers on
//    a fixed-point image, scaled per query or key by its sum of |dL|, so no order of additions shows in a result.  A
//    histogram H then gives, by matrix products,
//        dT[row][c] += sum_columns H[row][column] x[column][c]   (x = q, dout, k: the three table gradients)
//        dx[column][c] += sum_rows H[row][column] T[row][c]      (dq from Tq, dk from Tk)
//    and the tile's dL and P themselves are the histograms over keys and queries that give the rest of dq, dk, dv.
//
// Table gradients stay in the registers of the wavefronts that make them for all units of a workgroup, which works on one
// head, and meet in a reduction over the workgroups.  A key of a window of several tiles gets its dk and dv in parts, one
// per tile of queries, that a last kernel adds up in tile order: dq, dk, dv are the same bits on every call.
//
// Why tiles: the pair sweeps this form replaces run at two wavefronts per SIMD (192 VGPRs) and wait for a gathered table
// row of 64 bytes per pair, axis and table.  Here a pair's term is a word of LDS.  One form for every window size: a unit
// packs windows of up to 64 voxels side by side.  Measured, 9 axes, 12,421 voxels in windows of 72, 12 heads, fp32 tables
// beside fp16 features (forward and backward of a training step): 1860 us -> 947 us; of these the gradients kernel 540,
// records 188, setup, columns and finish 35.  No unit is busy: in the gradients kernel the VALU issues 39 % of the time, the
// LDS is addressed for 35 % (two fifths of it bank conflicts), the matrix pipe works for 4 %, and a wavefront waits for
// 52 % of its time - for the barriers of some 25 phases a tile, at four wavefronts per SIMD, and for 2 GB that a call
// moves, most of it the slots and registers that did not fit; in the records kernel 36, 31, 5 and 47 %.
#include "attn_tile.h"

#include <type_traits>

namespace s3d {
namespace tile {
namespace {

// dL and P in the gradients kernel.
//  * Summed by table row they are integers in cells of 32 bits: P in units of 2^-28 (a query's weights sum to 1 but for
//    rounding, also of fp16 tables in a forward whose backward has fp32 ones; there is room for 16), dL in units of 2^(e-30),
//    2^e the least power above the sum of |dL| of its query (by key: of its key) in the tile.  A cell keeps what fp32 would,
//    and no order of additions shows.
//  * They enter the products over 2^-kLiftP and 2^(e-kLift), the cells and the pairs' own alike: beside fp16 operands as two
//    fp16 numbers, 23 bits down to 2^-3 and units of 2^-24 below, that is 2^-35 of P and 2^-39 of the sum of |dL|.
//
// What is not finite stays in its window, though the products take all columns of a unit and all rows of a table, zeros
// among them: features and table entries that are not finite go into their operands as zeros.  Their pairs' dL is NaN (a
// query's, for q and dout; a key's, for k), with dout their P as well, and so dq, dk and dv are what the sums over a
// window's pairs would be, but for channels beside the one that is not finite.  In the integers such a pair counts for
// nothing; the table rows it belongs to are marked and their gradients stored as NaN.  A P beyond 8 says that the
// statistics are not the forward's, and is treated alike.
constexpr float kFixWeight = 268435456.0f, kMostWeight = 8.0f;
constexpr int kFixGrad = 30;
template <typename TF> constexpr int kLift = sizeof(TF) == 2 ? 15 : 0;       // (fp32 features may be as large as fp32 is)
template <typename TF> constexpr float kLiftP = sizeof(TF) == 2 ? 2048.0f : 1.0f;
template <typename TF> constexpr float kWeightCell = kLiftP<TF> / kFixWeight;
template <typename TF> constexpr float kGradCell = (sizeof(TF) == 2 ? 32768.0f : 1.0f) / 1073741824.0f;
constexpr int kLiftFeature = 15;              // exponent of the tile's largest q or k in the table gradients

// What the matrix products are made of: features (TF) as they are, and tables (T) in the same type, or fp32 tables beside
// fp16 features as pairs of fp16 numbers.
template <typename T, typename TF> struct TableOperand { using type = Operand<T>; };
template <> struct TableOperand<float, __half> { using type = Pair16; };

struct BwdTileArgs {
    AttnArgs f;                 // shape, q, k, v (dense), tables, index arrays, rows[] / base[]
    UnitList list;
    const void *dout, *out;
    const float *stat_max, *stat_sum;
    float2 *records;            // [H][pairs]: (dL, P)
    int64_t pairs;              // capacity of records per head; windows beyond it are skipped
    void *dq, *dk, *dv;
    float *parts;               // [(pairs / 64 + N) positions][H][dk | dv]: see part_row
    float *slots;               // [workgroup][table][stage][16 rows][lane][4]: table gradients as the products leave them
    int32_t *rows, *first_pair; // [unit][column]: the units' voxels, their rows and, of the pairs of their windows, the one
                                // with the window's first key (-1: beyond the records); see tile_columns_kernel
    float *coords;              // [unit][axis][column]
    void *operands;             // the tables as matrix operands, and
    float *scales;              // [head][5] what a product with them is multiplied by: see tile_setup_kernel
    float *dtq, *dtk, *dtv;
    int32_t groups;             // workgroups per head of the gradients kernel
};

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

// first row of a window's parts: windows of more than 64 voxels only, tiles * n rows each, which is at most
// floor((pairs before + n^2) / 64) - floor(pairs before / 64) + n
__device__ __forceinline__ int64_t part_row(const int2 entry) { return entry.y / 64 + entry.x; }

__device__ __forceinline__ bool window_fits(const int2 entry, int n, int64_t pairs)
{
    return static_cast<int64_t>(entry.y) + static_cast<int64_t>(n) * n <= pairs;
}

// ---- setup ------------------------------------------------------------------------------------------------------------
// The unit list (workgroup 0) and, a workgroup for each head and kind, the tables as the lanes' matrix operands:
// [head][q rows, k rows, v rows, q by channel, k by channel][stage][half][lane].  By rows: table row lane % 32 of the
// half, channels 8 (lane / 32) ..; by channel: channel lane % 16, rows in the order of permuted_row.
template <typename T, typename TF, int ND>
__global__ __launch_bounds__(kListThreads) void tile_setup_kernel(BwdTileArgs b)
{
    using S = Stages<ND>;
    using Table = typename TableOperand<T, TF>::type;
    const AttnArgs &a = b.f;
    if (blockIdx.x == 0) {
        build_list(a.w_sizes, a.w2n, static_cast<int>(a.W), const_cast<int32_t *>(b.list.total),
                   const_cast<int4 *>(b.list.units), const_cast<int2 *>(b.list.entries));
        return;
    }
    const int job = static_cast<int>(blockIdx.x) - 1, kind = job % 5, h = job / 5, HD = a.H * D;
    const T *table = static_cast<const T *>(kind == 0 || kind == 3 ? a.table_q : kind == 2 ? a.table_v : a.table_k) + h * D;
    float scale = 1.0f;
    if constexpr (std::is_same<Table, Pair16>::value) {
        __shared__ int top_s;
        if (threadIdx.x == 0) top_s = 0;
        __syncthreads();
        float top = 0.0f;
        for (int t = threadIdx.x; t < a.total_rows * D; t += kListThreads) {
            const float x = table[static_cast<int64_t>(t / D) * HD + t % D];
            top = fmaxf(top, finite(x) ? fabsf(x) : 0.0f);
        }
        atomicMax(&top_s, __float_as_int(top));
        __syncthreads();
        scale = power2(min(100, 14 - exponent_of(__int_as_float(top_s))));
    }
    if (threadIdx.x == 0) b.scales[h * 5 + kind] = 1.0f / scale;
    const int t = threadIdx.x, lane = t % 64, half = t / 64 % 2, st = t / 128;
    if (st >= S::kCount) return;
    const int axis = st < 3 ? st : S::first(st) + half, row0 = st < 3 ? half * 32 : 0;
    T v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = static_cast<T>(0.0f);
    if (axis < ND) {
        const int rows = axis_rows<ND>(a, axis), first = axis_base<ND>(a, axis);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int r = kind < 3 ? row0 + lane % 32 : row0 + 2 * (lane / 16) + (e & 1) + 8 * (e >> 1);
            const int c = kind < 3 ? lane / 32 * 8 + e : lane % 16;
            v[e] = table[static_cast<int64_t>(first + min(r, rows - 1)) * HD + c];
            if (kind >= 3 && !finite(to_float(v[e]))) v[e] = static_cast<T>(0.0f);
        }
    }
    Table x;
    if constexpr (std::is_same<Table, Pair16>::value) x.set_values(v, scale);
    else x.set_values(v);
    static_cast<Table *>(b.operands)[job * (S::kCount * 128) + t] = x;
}

// The voxels of every unit, side by side: what the heads' workgroups then read in one step instead of a chain of four.
template <int ND>
__global__ __launch_bounds__(256) void tile_columns_kernel(BwdTileArgs b)
{
    const AttnArgs &a = b.f;
    const int u = static_cast<int>(blockIdx.x) * 4 + static_cast<int>(threadIdx.x >> 6), c = threadIdx.x & 63;
    if (u >= b.list.total[0]) return;
    const Unit unit(b.list.units[u]);
    const int cc = max(0, min(c, unit.cols - 1));
    const int2 entry = unit.entry_of(b.list, cc);
    const int in = unit.inside(unit.tile, cc), pos = entry.x + in;
    b.rows[u * kCols + c] = a.n2n ? a.n2n[pos] : pos;
    b.first_pair[u * kCols + c] = window_fits(entry, unit.n_w, b.pairs) ? entry.y + in : -1;
#pragma unroll
    for (int n = 0; n < ND; ++n)
        b.coords[(static_cast<int64_t>(u) * ND + n) * kCols + c] = a.n_coords[static_cast<int64_t>(pos) * ND + n];
}

// ---- records ----------------------------------------------------------------------------------------------------------
// As the forward's tile kernel: two workgroups of eight wavefronts per CU (80 KB of LDS and 128 VGPRs each), all products
// of a stage by two wavefronts per table, the pairs' gathers by all.  The next stage's table operands are under way
// while the pairs gather.
template <int ND> struct RecordsLayout {
    static constexpr uint32_t kQueries = kCols * kStride * 8;                    // (q . Tq, dout . Tv), [row][query]
    static constexpr uint32_t kKeys = kCols * kKeyStride * 4;                    // coordinates, k . Tk, [key][row]
    static constexpr uint32_t kCoords = ND * kCols * 4;
    static constexpr uint32_t kBytes = kQueries + kKeys + kCoords;
};

template <typename T, typename TF, int ND>
__global__ __launch_bounds__(kThreads, 4) void tile_records_kernel(BwdTileArgs b)
{
    using L = RecordsLayout<ND>;
    using S = Stages<ND>;
    const AttnArgs &a = b.f;
    extern __shared__ __align__(16) float smem[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int H = a.H, HD = H * D;
    const int h = static_cast<int>(blockIdx.x) % H;
    const int group = static_cast<int>(blockIdx.x) / H, groups = static_cast<int>(gridDim.x) / H;
    const int total_units = b.list.total[0];

    const uint32_t queries = lds_base(smem), keys = queries + L::kQueries, coords = keys + L::kKeys;
    const TF *gq = static_cast<const TF *>(a.q), *gk = static_cast<const TF *>(a.k), *gv = static_cast<const TF *>(a.v);
    const TF *gd = static_cast<const TF *>(b.dout), *go = static_cast<const TF *>(b.out);
    using Table = typename TableOperand<T, TF>::type;
    const Table *operands = static_cast<const Table *>(b.operands) + static_cast<int64_t>(h) * (5 * S::kCount * 128);
    const float scale_q = b.scales[h * 5], scale_k = b.scales[h * 5 + 1], scale_v = b.scales[h * 5 + 2];
    const int tile_c = wave & 1, tile_r = (wave >> 1) & 1;

    for (int u = group; u < total_units; u += groups) {
        const Unit unit(b.list.units[u]);
        const int cols = unit.cols, n_w = unit.n_w;
        const bool small = unit.small;
        if (cols <= 0) continue;
        const int reach = kThreads / cols;
        const int own = tid % cols, first = tid / cols;
        const bool active = first < reach;
        // the query's statistics and dout . out
        const int own_pair = b.first_pair[u * kCols + own];
        float own_max, own_inv, own_delta = 0.0f;
        {
            const int64_t row = b.rows[u * kCols + own];
            own_max = b.stat_max[row * H + h];
            own_inv = 1.0f / b.stat_sum[row * H + h];
#pragma unroll
            for (int c = 0; c < D; c += 8) {
                float x[8], y[8];
                load_row<8>(gd + row * HD + h * D + c, x);
                load_row<8>(go + row * HD + h * D + c, y);
#pragma unroll
                for (int e = 0; e < 8; ++e) own_delta += x[e] * y[e];
            }
        }
        for (int block = 0; block < unit.blocks(); ++block) {
            const int keys_n = unit.keys(block);
            if (keys_n <= 0) break;
            const int other = small ? u : u - unit.tile + block;         // the unit whose voxels are the keys
            const int lane = opaque(tid & 63);
            const int m32 = lane & 31, half32 = lane >> 5;
            const int channel = h * D + half32 * 8;
            Operand<TF> feat, grad, x_k, x_v;
            {
                const uint64_t row = static_cast<uint32_t>(b.rows[(wave < 4 ? u : other) * kCols + tile_c * 32 + m32]);
                feat.load((wave < 4 ? gq : gk) + row * HD + channel);
                if (wave < 4) {
                    const uint64_t key_row = static_cast<uint32_t>(b.rows[other * kCols + tile_r * 32 + m32]);
                    grad.load(gd + row * HD + channel);
                    x_k.load(gk + key_row * HD + channel);
                    x_v.load(gv + key_row * HD + channel);
                }
            }
            float x[ND];
            if (wave < 2) {
#pragma unroll
                for (int n = 0; n < ND; ++n) x[n] = (b.coords + static_cast<int64_t>(wave == 0 ? u : other) * (ND * kCols))[n * kCols + static_cast<uint32_t>(lane)];
            }
            lds_barrier();
            if (wave < 2) {
#pragma unroll
                for (int n = 0; n < ND; ++n) lds_store(wave == 0 ? coords + (n * kCols + lane) * 4 : keys + (lane * kKeyStride + n) * 4, x[n]);
            }
            if (wave < 4) {
                // (q . k, dout . v) of the tile, [key][query]
                const f32x16 dl = mfma32(x_k, feat, f32x16{});
                const f32x16 dp = mfma32(x_v, grad, f32x16{});
                const uint32_t to = queries + ((tile_r * 32 + 4 * half32) * kStride + tile_c * 32 + m32) * 8;
#pragma unroll
                for (int e = 0; e < 16; ++e) lds_store2(to + mfma32_row(0, e) * kStride * 8, dl[e], dp[e]);
            }
            lds_barrier();
            const int key0 = small ? own / n_w * n_w : 0;
            const int per_query = small ? n_w : keys_n;
            const int steps = (per_query + reach - 1) / reach;
            float logit[kSteps], dp[kSteps];
            uint32_t key_at[kSteps];
#pragma unroll
            for (int s = 0; s < kSteps; ++s) {
                const int j = key0 + min(first + s * reach, per_query - 1);
                key_at[s] = opaque(keys + j * (kKeyStride * 4));
                const float2 x = lds_load2(queries + (j * kStride + own) * 8);
                logit[s] = x.x;
                dp[s] = x.y;
            }
            // (rolled: the kernel's code has to stay in the instruction cache)
            auto stage_needed = [&](int st) {
                return (st < 3 ? tile_r * 32 < axis_rows<ND>(a, st) : S::first(st) + tile_r < ND) && tile_c * 32 < (wave < 4 ? cols : keys_n);
            };
            Table rows_a, rows_v;
            auto fetch = [&](int st) {
                const Table *from = operands + ((wave < 4 ? 0 : 1) * S::kCount + st) * 128 + tile_r * 64 + lane;
                rows_a = from[0];
                if (wave < 4) rows_v = from[2 * S::kCount * 128];
            };
            if (stage_needed(0)) fetch(0);
            auto stage = [&](int st, auto paired) {
                lds_barrier();
                if (stage_needed(st)) {
                    if (wave < 4) {
                        const f32x16 dl = mfma32(rows_a, feat, f32x16{});
                        const f32x16 dv = mfma32(rows_v, grad, f32x16{});
                        const uint32_t to = queries + ((tile_r * 32 + 4 * half32) * kStride + tile_c * 32 + m32) * 8;
#pragma unroll
                        for (int e = 0; e < 16; ++e) lds_store2(to + mfma32_row(0, e) * kStride * 8, dl[e], dv[e]);
                    } else {
                        const f32x16 dl = mfma32(feat, rows_a, f32x16{});
                        const uint32_t to = keys + ((tile_c * 32 + 4 * half32) * kKeyStride + kCoordWords + tile_r * 32 + m32) * 4;
#pragma unroll
                        for (int e = 0; e < 16; ++e) lds_store(to + mfma32_row(0, e) * kKeyStride * 4, dl[e]);
                    }
                }
                if (st + 1 < S::kCount && stage_needed(st + 1)) fetch(st + 1);
                lds_barrier();
#pragma unroll
                for (int p = 0; p < (paired ? 2 : 1); ++p) {
                    const int axis = S::first(st) + p;
                    if (axis >= ND) break;
                    const float half_rows = static_cast<float>(axis_rows<ND>(a, axis) / 2), upper = crse_upper(axis_rows<ND>(a, axis));
                    const float ci = lds_load(coords + (axis * kCols + own) * 4);
                    const uint32_t own_at = queries + own * 8 + p * 32 * kStride * 8;
                    for_steps(steps, [&](int s) {
                        const float cj = lds_load(key_at[s] + axis * 4);
                        const uint32_t r = static_cast<uint32_t>(crse_row(ci, cj, half_rows, upper));
                        const float2 x = lds_load2(__umul24(r, kStride * 8) + own_at);
                        const float k = lds_load(r * 4 + key_at[s] + (kCoordWords + p * 32) * 4);
                        logit[s] += fmaf(k, scale_k, x.x * scale_q);      // (the long sum is rounded once an axis)
                        dp[s] = fmaf(x.y, scale_v, dp[s]);
                    });
                }
            };
#pragma unroll 1
            for (int st = 0; st < 3; ++st) stage(st, std::false_type{});
#pragma unroll 1
            for (int st = 3; st < S::kCount; ++st) stage(st, std::true_type{});
            const int my_steps = active && own_pair >= 0 ? (per_query - first + reach - 1) / reach : 0;
            float2 *to = b.records + static_cast<int64_t>(h) * b.pairs + own_pair + static_cast<int64_t>((small ? 0 : block * unit.size) + first) * n_w;
#pragma unroll
            for (int s = 0; s < kSteps; ++s) {
                if (s < my_steps) {
                    const float p = __expf(logit[s] - own_max) * own_inv;
                    // (a logit of minus infinity has no weight, but its dL meets an infinite key or table row in dq)
                    *to = make_float2(finite(logit[s]) ? p * (dp[s] - own_delta) : __int_as_float(0x7fc00000), p);
                }
                to += reach * n_w;
            }
        }
    }
}

// ---- gradients --------------------------------------------------------------------------------------------------------
// Two workgroups per CU as above.  A tile of 64 x 64 pairs takes about 100k clocks of a shared CU: 26k to bring it into
// LDS, 6k for the matrix products of the tile itself, 23k for the additions by row, 20k for the products of the
// histograms (whose operands are columns of LDS), the rest clearing and waiting at barriers.
template <typename TF, int ND> struct GradLayout {
    static constexpr int kSt = Stages<ND>::kCount;
    static constexpr uint32_t kCells = kCols * kStride * 8;                      // [row][query] of (P, dL); P tile; [row][key]
    static constexpr uint32_t kTile = kCols * kStride * 4;                       // dL, [key][query]
    static constexpr uint32_t kFeature = D * kStride * sizeof(TF);               // q, dout, k: [channel][column]
    static constexpr uint32_t kCoords = ND * kCols * 4;
    static constexpr uint32_t kMeta = 2 * kCols * 4 + 32;                        // exponents of queries and keys; maxima, a flag
    static constexpr uint32_t kMarks = 6 * 8 + kSt * 16;                         // features and table rows that are not finite
    static constexpr uint32_t kBytes = kCells + kTile + 3 * kFeature + 2 * kCoords + kMeta + kMarks;
};

template <typename T, typename TF, int ND>
__global__ __launch_bounds__(kThreads, 4) void tile_gradients_kernel(BwdTileArgs b)
{
    using L = GradLayout<TF, ND>;
    using Table = typename TableOperand<T, TF>::type;
    using S = Stages<ND>;
    const AttnArgs &a = b.f;
    extern __shared__ __align__(16) float smem[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int H = a.H, HD = H * D;
    const int h = static_cast<int>(blockIdx.x) % H;
    const int group = static_cast<int>(blockIdx.x) / H, groups = static_cast<int>(gridDim.x) / H;
    const int total_units = b.list.total[0];
    if (group >= total_units) return;       // its slot is not read

    const uint32_t cells = lds_base(smem), tile = cells + L::kCells, feats = tile + L::kTile;
    const uint32_t coords_i = feats + 3 * L::kFeature, coords_j = coords_i + L::kCoords;
    const uint32_t exp_i = coords_j + L::kCoords, exp_j = exp_i + kCols * 4, exp_top = exp_j + kCols * 4;
    const uint32_t not_finite = exp_top + 16;                        // the tile has a pair that is not finite
    const uint32_t bad_columns = exp_top + 32;                       // per wavefront that loads features: 64 bits
    const uint32_t bad_rows = bad_columns + 6 * 8;                   // per stage: rows of such a dL, of such a P, 64 bits each
    const uint32_t feat_q = feats, feat_d = feats + L::kFeature, feat_k = feats + 2 * L::kFeature;

    const bool low = wave < 4;               // wavefronts 0..3 and 4..7 share the products differently
    const int quarter = wave & 3;            // 16 table rows, queries or keys
    // Table gradients of the workgroup: 16 rows of a stage, of Tq and Tv (wavefronts 0..3) or Tk (4..7).  They stay in the
    // workgroup's slot in memory (its L2), where every word is one lane's: 48 registers that the lane does not have.
    float *slot = b.slots + static_cast<int64_t>(blockIdx.x) * (3 * L::kSt * kCols * D);
    constexpr int kKind = L::kSt * kCols * D;
    for (int t = tid; t < 3 * kKind / 4; t += kThreads) reinterpret_cast<float4 *>(slot)[t] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    __syncthreads();
    const Table *operands = static_cast<const Table *>(b.operands) + (static_cast<int64_t>(h) * 5 + 3) * (S::kCount * 128);
    const float table_scale = b.scales[h * 5 + (low ? 4 : 3)];      // of the table this wavefront reads by channel
    bool incomplete = false;                 // a window did not fit the records

    for (int u = group; u < total_units; u += groups) {
        const Unit unit(b.list.units[u]);
        const int cols = unit.cols, n_w = unit.n_w;
        const bool small = unit.small;
        if (cols <= 0) continue;
        const int reach = kThreads / cols;
        const int own = tid % cols, first = tid / cols;
        f32x4_t dq_sum = {0.0f, 0.0f, 0.0f, 0.0f};       // wavefronts 4..7
        for (int block = 0; block < unit.blocks(); ++block) {
            const int keys_n = unit.keys(block);
            if (keys_n <= 0) break;
            const int per_query = small ? n_w : keys_n;
            const int per_key = small ? n_w : cols;
            const int other = small ? u : u - unit.tile + block;         // the unit whose voxels are the keys
            // Coordinates, features and records of the tile.  Every wavefront is past the last barrier of the tile before,
            // behind which nothing of it is read from LDS.
            float grad[kSteps], weight[kSteps], top = 0.0f;
            const int which = wave >> 1, c8 = wave & 1;                  // q, dout, k: eight channels a wavefront
            {
                const uint32_t c = tid & 63;
                if (wave < 6) {
                    const TF *from = static_cast<const TF *>(which == 0 ? a.q : which == 1 ? b.dout : a.k) + h * D + c8 * 8;
                    const int32_t *rows = b.rows + (which == 2 ? other : u) * kCols;
                    float v[8];
                    load_row<8>(from + static_cast<uint64_t>(static_cast<uint32_t>(rows[c])) * static_cast<uint32_t>(HD), v);
                    const bool there = static_cast<int>(c) < (which == 2 ? keys_n : cols);
                    TF *to = reinterpret_cast<TF *>(reinterpret_cast<char *>(smem) + (feats - cells) + which * L::kFeature) + c8 * 8 * kStride + c;
                    bool bad = false;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        bad = bad || !finite(v[e]);
                        const float x = there && finite(v[e]) ? v[e] : 0.0f;
                        to[e * kStride] = static_cast<TF>(x);
                        top = fmaxf(top, fabsf(x));
                    }
                    const uint64_t columns = __ballot(bad && there);
                    if (c < 2) lds_store_u32(bad_columns + wave * 8 + c * 4, static_cast<uint32_t>(columns >> (32 * c)));
                } else {
                    const float *from = b.coords + static_cast<int64_t>(wave == 6 ? u : other) * (ND * kCols);
                    const uint32_t to = (wave == 6 ? coords_i : coords_j) + c * 4;
#pragma unroll
                    for (int n = 0; n < ND; ++n) lds_store(to + n * kCols * 4, from[n * kCols + c]);
                }
            }
            const int own_pair = (b.first_pair + u * kCols)[static_cast<uint32_t>(own)];
            const int my_steps = first < reach ? (per_query - first + reach - 1) / reach : 0;
            const int key0 = small ? own / n_w * n_w : 0;
            {
                // a window beyond the records: its gradients say so
                const float none = own_pair >= 0 ? 0.0f : __int_as_float(0x7fc00000);
                incomplete = incomplete || own_pair < 0;
                const float2 *from = b.records + static_cast<int64_t>(h) * b.pairs +
                                     (max(own_pair, 0) + static_cast<int64_t>((small ? 0 : block * unit.size) + first) * n_w);
#pragma unroll
                for (int s = 0; s < kSteps; ++s) {
                    float2 r = make_float2(none, none);
                    if (s < my_steps && own_pair >= 0) r = *from;
                    from += reach * n_w;
                    grad[s] = s < my_steps ? r.x : 0.0f;
                    weight[s] = s < my_steps ? r.y : 0.0f;
                }
            }
            lds_zero<kCols * kStride>(tile, tid);
            lds_zero<kCols * kStride>(cells, tid);
            if (tid < 5) lds_store_u32(exp_top + tid * 4, tid < 4 ? static_cast<uint32_t>(-100) : 0u);
            lds_barrier();
            // tile and cells [key][query]; the largest exponent of a q or k
            if (wave < 6 && which != 1) lds_max(exp_top + (which == 0 ? 8 : 12), exponent_of(top));
            {
                uint64_t bad[3];           // queries by q, by dout; keys
#pragma unroll
                for (int f = 0; f < 3; ++f) {
                    const u32x4_t m = *(lds_u32x4 *)(bad_columns + f * 16);
                    bad[f] = static_cast<uint64_t>(m[1] | m[3]) << 32 | (m[0] | m[2]);
                }
                bool any = false;
#pragma unroll
                for (int s = 0; s < kSteps; ++s) {
                    if (s < my_steps) {
                        const bool by_dout = (bad[1] >> own & 1) != 0 || !(weight[s] <= kMostWeight);
                        if (by_dout || ((bad[0] >> own | bad[2] >> (key0 + first + s * reach)) & 1) != 0) grad[s] = __int_as_float(0x7fc00000);
                        if (by_dout) weight[s] = __int_as_float(0x7fc00000);
                        any = any || !finite(grad[s]);
                    }
                }
                if (any) lds_store_u32(not_finite, 1u);
                const uint32_t at = ((key0 + first) * kStride + own) * 4, step = reach * (kStride * 4);
#pragma unroll
                for (int s = 0; s < kSteps; ++s) {
                    if (s < my_steps) {
                        lds_store(tile + at + s * step, grad[s]);
                        lds_store(cells + at + s * step, weight[s]);
                    }
                }
            }
            lds_barrier();
            const int lane = opaque(tid & 63);
            const int n16 = lane & 15, group16 = lane >> 4;
            const int column = quarter * 16 + n16;            // this lane's query or key in the products
            const uint32_t term_at = group16 * 8;
            // cells as an operand: a row's eight columns, a column's eight rows
            const uint32_t row_at = (quarter * 16 + n16) * kStride + term_at, column_at = 2 * group16 * kStride + column;
            const uint32_t channel_at = (n16 * kStride + term_at) * sizeof(TF);
            f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};           // dk (wavefronts 0..3) or dq, over 2^(exponent - kLift)
            f32x4_t table_acc = {0.0f, 0.0f, 0.0f, 0.0f};     // ... the tables' part, over table_scale as well
            f32x4_t dv_acc = {0.0f, 0.0f, 0.0f, 0.0f};
            int exponent;
            {
                // a column of dL per lane (the other lane groups hold its other terms), its sum's exponent, and the products
                // dk_j += sum_i dL q_i, dv_j += sum_i P dout_i; dq_i += sum_j dL k_j
                float v[2][8], all = 0.0f;
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) {
                    if (low) {
                        lds_load8(tile + row_at * 4 + ks * 128, v[ks]);
                    } else {
#pragma unroll
                        for (int e = 0; e < 8; ++e) v[ks][e] = lds_load(tile + (term_at * kStride + column) * 4 + (ks * 32 + e) * kStride * 4);
                    }
#pragma unroll
                    for (int e = 0; e < 8; ++e) all += finite(v[ks][e]) ? fabsf(v[ks][e]) : 0.0f;
                }
                all += __shfl_xor(all, 16);
                all += __shfl_xor(all, 32);
                exponent = exponent_of(all);
                if (group16 == 0) {
                    lds_store_u32((low ? exp_j : exp_i) + column * 4, exponent);
                    lds_max(exp_top + (low ? 4 : 0), exponent);
                }
                const float scale = power2(kLift<TF> - exponent);
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) {
                    Cells<TF> c;
                    c.set(v[ks], scale);
                    Operand<TF> x;
                    x.load_lds((low ? feat_q : feat_k) + channel_at + ks * 32 * sizeof(TF));
                    acc = mfma16(x, c, acc);
                    if (low) {
                        float w[8];
                        lds_load8(cells + row_at * 4 + ks * 128, w);
                        c.set(w, kLiftP<TF>);
                        x.load_lds(feat_d + channel_at + ks * 32 * sizeof(TF));
                        dv_acc = mfma16(x, c, dv_acc);
                    }
                }
            }
            lds_barrier();
            // fixed-point images of the pairs' dL and P, by query
            uint32_t fix_p[kSteps];
            int fix_l[kSteps];
            {
                const int up = kFixGrad - static_cast<int>(lds_load_u32(exp_i + own * 4));
#pragma unroll
                for (int s = 0; s < kSteps; ++s) {
                    fix_l[s] = static_cast<int>(rintf(ldexpf(grad[s], up)));
                    fix_p[s] = static_cast<uint32_t>(rintf(weight[s] * kFixWeight));
                }
            }
            const int top_i = static_cast<int>(lds_load_u32(exp_top)), top_j = static_cast<int>(lds_load_u32(exp_top + 4));
            const int lift_q = kLiftFeature - static_cast<int>(lds_load_u32(exp_top + 8)), lift_k = kLiftFeature - static_cast<int>(lds_load_u32(exp_top + 12));
            {
                // q and k over the tile's largest exponent of a query or key, for the table gradients; the largest value
                // below 2^15, as far as can be from where fp16 numbers lose bits
                TF *fq = reinterpret_cast<TF *>(reinterpret_cast<char *>(smem) + (feat_q - cells));
                TF *fk = reinterpret_cast<TF *>(reinterpret_cast<char *>(smem) + (feat_k - cells));
                const int c = tid & 63;
                const float si = power2(static_cast<int>(lds_load_u32(exp_i + c * 4)) - top_i + lift_q);
                const float sj = power2(static_cast<int>(lds_load_u32(exp_j + c * 4)) - top_j + lift_k);
#pragma unroll
                for (int x = 0; x < D; x += kWaves) {
                    const int at = (wave + x) * kStride + c;
                    fq[at] = static_cast<TF>(static_cast<float>(fq[at]) * si);
                    fk[at] = static_cast<TF>(static_cast<float>(fk[at]) * sj);
                }
            }
            const float grad_i = power2(top_i - lift_q - kLift<TF>), grad_j = power2(top_j - lift_k - kLift<TF>);
            const int steps = (per_query + reach - 1) / reach;
            uint32_t other_at[kSteps];           // coordinates of the pairs' other side
#pragma unroll
            for (int s = 0; s < kSteps; ++s) other_at[s] = coords_j + (key0 + min(first + s * reach, per_query - 1)) * 4;
            const bool marks = __builtin_amdgcn_readfirstlane(lds_load_u32(not_finite)) != 0;
            if (marks) {
                if (tid < L::kSt * 4) lds_store_u32(bad_rows + tid * 4, 0u);
                lds_barrier();
#pragma unroll
                for (int s = 0; s < kSteps; ++s) {
                    if (s >= my_steps || finite(grad[s])) continue;
#pragma unroll 1
                    for (int axis = 0; axis < ND; ++axis) {
                        const int rows = axis_rows<ND>(a, axis), st = axis < 3 ? axis : 3 + (axis - 3) / 2;
                        const int r = crse_row(lds_load(coords_i + (axis * kCols + own) * 4), lds_load(other_at[s] + axis * kCols * 4),
                                               static_cast<float>(rows / 2), crse_upper(rows));
                        const uint32_t at = bad_rows + st * 16 + (axis < 3 ? r >> 5 : (axis - 3) & 1) * 4;
                        lds_or(at, 1u << (r & 31));
                        if (!finite(weight[s])) lds_or(at + 8, 1u << (r & 31));
                    }
                }
                // (read behind the next barrier)
            }
            // four rows of a table gradient, marked ones as NaN
            auto marked = [&](int st, int of_weight, float4 g) {
                if (!marks) return g;
                const uint32_t m = lds_load_u32(bad_rows + st * 16 + of_weight * 8 + (quarter >> 1) * 4) >> ((quarter & 1) * 16 + group16 * 4);
                const float nan = __int_as_float(0x7fc00000);
                return make_float4(m & 1 ? nan : g.x, m & 2 ? nan : g.y, m & 4 ? nan : g.z, m & 8 ? nan : g.w);
            };
            // rows of half ks of stage st in use
            auto half_used = [&](int st, int ks) { return st < 3 ? ks * 32 < axis_rows<ND>(a, st) : S::first(st) + ks < ND; };
            // rows of this wavefront's quarter of stage st
            auto quarter_rows = [&](int st) {
                if (st < 3) return axis_rows<ND>(a, st) - quarter * 16;
                const int axis = S::first(st) + (quarter >> 1);
                return axis < ND ? axis_rows<ND>(a, axis) - (quarter & 1) * 16 : 0;
            };
            // what a stage reads from memory is under way while its pairs are added up: this lane's table gradients so far
            // (the wavefronts that make those), or the table as an operand
            float4 *slot_at = reinterpret_cast<float4 *>(slot) + quarter * 64 + lane;
            constexpr int kStageSlot = kCols * D / 4;

            // ---- by query: dTq, dTv (wavefronts 0..3), dq (4..7)
            auto by_query = [&](int st, auto paired) {
                float4 old_q, old_v;
                Table x[2];
                if (low) {
                    old_q = slot_at[st * kStageSlot];
                    old_v = slot_at[2 * kKind / 4 + st * kStageSlot];
                } else {
                    x[0] = operands[st * 128 + lane];
                    x[1] = operands[st * 128 + 64 + lane];
                }
                lds_zero<kCols * kStride * 2>(cells, tid);
                lds_barrier();
#pragma unroll
                for (int p = 0; p < (paired ? 2 : 1); ++p) {
                    const int axis = S::first(st) + p;
                    if (axis >= ND) break;
                    const float half_rows = static_cast<float>(axis_rows<ND>(a, axis) / 2), upper = crse_upper(axis_rows<ND>(a, axis));
                    const float ci = lds_load(coords_i + (axis * kCols + own) * 4);
                    const uint32_t own_at = cells + own * 8 + p * 32 * kStride * 8;
                    const uint32_t axis_at = axis * kCols * 4;
                    // (all reads before the first addition: the compiler keeps the order of the two)
                    float cj[kSteps];
                    for_steps(steps, [&](int s) { cj[s] = lds_load(other_at[s] + axis_at); });
                    for_steps(steps, [&](int s) {
                        const uint32_t r = static_cast<uint32_t>(crse_row(ci, cj[s], half_rows, upper));
                        lds_add64(__umul24(r, kStride * 8) + own_at, fix_p[s], fix_l[s]);
                    });
                }
                lds_barrier();
                if (low) {
                    if (quarter_rows(st) > 0) {
                        f32x4_t gq = {0.0f, 0.0f, 0.0f, 0.0f}, gv = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                        for (int ks = 0; ks < 2; ++ks) {
                            if (ks * 32 >= cols) break;
                            uint32_t w[8];
                            int l[8];
                            lds_load_cells(cells + row_at * 8 + ks * 256, w, l);
                            float v[8];
                            CellsA<TF> c;
                            Operand<TF> x;
#pragma unroll
                            for (int e = 0; e < 8; ++e) v[e] = static_cast<float>(l[e]);
                            c.set(v, kGradCell<TF>);
                            x.load_lds(feat_q + channel_at + ks * 32 * sizeof(TF));
                            gq = mfma16(c, x, gq);
#pragma unroll
                            for (int e = 0; e < 8; ++e) v[e] = static_cast<float>(w[e]);
                            c.set(v, kWeightCell<TF>);
                            x.load_lds(feat_d + channel_at + ks * 32 * sizeof(TF));
                            gv = mfma16(c, x, gv);
                        }
                        slot_at[st * kStageSlot] = marked(st, 0, make_float4(fmaf(gq[0], grad_i, old_q.x), fmaf(gq[1], grad_i, old_q.y),
                                                                             fmaf(gq[2], grad_i, old_q.z), fmaf(gq[3], grad_i, old_q.w)));
                        constexpr float back = 1.0f / kLiftP<TF>;
                        slot_at[2 * kKind / 4 + st * kStageSlot] = marked(st, 1, make_float4(fmaf(gv[0], back, old_v.x), fmaf(gv[1], back, old_v.y),
                                                                                             fmaf(gv[2], back, old_v.z), fmaf(gv[3], back, old_v.w)));
                    }
                } else if (quarter * 16 < cols) {
#pragma unroll
                    for (int ks = 0; ks < 2; ++ks) {
                        if (!half_used(st, ks)) continue;
                        float v[8];
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            v[e] = static_cast<float>(static_cast<int>(lds_load_u32(cells + column_at * 8 + (ks * 32 + (e & 1) + 8 * (e >> 1)) * kStride * 8 + 4)));
                        Cells<TF> c;
                        c.template set<false>(v, kGradCell<TF>);      // (the table's operand is the nearest)
                        table_acc = mfma16(x[ks], c, table_acc);
                    }
                }
                lds_barrier();
            };
#pragma unroll 1
            for (int st = 0; st < 3; ++st) by_query(st, std::false_type{});
#pragma unroll 1
            for (int st = 3; st < S::kCount; ++st) by_query(st, std::true_type{});
            // ---- by key: dTk (wavefronts 4..7), dk (0..3)
            const int reach_k = kThreads / keys_n;
            const int own_k = tid % keys_n, first_k = tid / keys_n;
            const int query0 = small ? own_k / n_w * n_w : 0;
            const int steps_k = (per_key + reach_k - 1) / reach_k;
            {
                const int up = kFixGrad - static_cast<int>(lds_load_u32(exp_j + own_k * 4));
#pragma unroll
                for (int s = 0; s < kSteps; ++s) {
                    const int i = first_k + s * reach_k, at = query0 + min(i, per_key - 1);
                    const float x = lds_load(tile + (own_k * kStride + at) * 4);
                    other_at[s] = coords_i + at * 4;
                    fix_l[s] = first_k < reach_k && i < per_key ? static_cast<int>(rintf(ldexpf(x, up))) : 0;
                }
            }
            lds_zero<kCols * kStride>(cells, tid);
            lds_barrier();
            auto by_key = [&](int st, auto paired) {
                const uint32_t here = cells + (st & 1) * L::kTile, next = cells + (~st & 1) * L::kTile;
                float4 old_k;
                Table x[2];
                if (!low) {
                    old_k = slot_at[kKind / 4 + st * kStageSlot];
                } else {
                    x[0] = operands[(S::kCount + st) * 128 + lane];
                    x[1] = operands[(S::kCount + st) * 128 + 64 + lane];
                }
#pragma unroll
                for (int p = 0; p < (paired ? 2 : 1); ++p) {
                    const int axis = S::first(st) + p;
                    if (axis >= ND) break;
                    const float half_rows = static_cast<float>(axis_rows<ND>(a, axis) / 2), upper = crse_upper(axis_rows<ND>(a, axis));
                    const float cj = lds_load(coords_j + (axis * kCols + own_k) * 4);
                    const uint32_t own_at = here + own_k * 4 + p * 32 * kStride * 4;
                    const uint32_t axis_at = axis * kCols * 4;
                    float ci[kSteps];
                    for_steps(steps_k, [&](int s) { ci[s] = lds_load(other_at[s] + axis_at); });
                    for_steps(steps_k, [&](int s) {
                        const uint32_t r = static_cast<uint32_t>(crse_row(ci[s], cj, half_rows, upper));
                        lds_add(__umul24(r, kStride * 4) + own_at, static_cast<uint32_t>(fix_l[s]));
                    });
                }
                lds_barrier();
                if (!low) {
                    if (quarter_rows(st) > 0) {
                        f32x4_t gk = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                        for (int ks = 0; ks < 2; ++ks) {
                            if (ks * 32 >= keys_n) break;
                            float v[8];
                            lds_load8(here + row_at * 4 + ks * 128, v);
#pragma unroll
                            for (int e = 0; e < 8; ++e) v[e] = static_cast<float>(__float_as_int(v[e]));
                            CellsA<TF> c;
                            c.set(v, kGradCell<TF>);
                            Operand<TF> x;
                            x.load_lds(feat_k + channel_at + ks * 32 * sizeof(TF));
                            gk = mfma16(c, x, gk);
                        }
                        slot_at[kKind / 4 + st * kStageSlot] = marked(st, 0, make_float4(fmaf(gk[0], grad_j, old_k.x), fmaf(gk[1], grad_j, old_k.y),
                                                                                         fmaf(gk[2], grad_j, old_k.z), fmaf(gk[3], grad_j, old_k.w)));
                    }
                } else if (quarter * 16 < keys_n) {
#pragma unroll
                    for (int ks = 0; ks < 2; ++ks) {
                        if (!half_used(st, ks)) continue;
                        float v[8];
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            v[e] = static_cast<float>(static_cast<int>(lds_load_u32(here + column_at * 4 + (ks * 32 + (e & 1) + 8 * (e >> 1)) * kStride * 4)));
                        Cells<TF> c;
                        c.template set<false>(v, kGradCell<TF>);      // (the table's operand is the nearest)
                        table_acc = mfma16(x[ks], c, table_acc);
                    }
                }
                lds_zero<kCols * kStride>(next, tid);
                lds_barrier();
            };
#pragma unroll 1
            for (int st = 0; st < 3; ++st) by_key(st, std::false_type{});
#pragma unroll 1
            for (int st = 3; st < S::kCount; ++st) by_key(st, std::true_type{});
            const float back = power2(exponent - kLift<TF>);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] = fmaf(table_acc[e], table_scale, acc[e]);
            if (!low) {
#pragma unroll
                for (int e = 0; e < 4; ++e) dq_sum[e] += acc[e] * back;
            } else if (column < keys_n) {
                const float o[4] = {acc[0] * back, acc[1] * back, acc[2] * back, acc[3] * back};
                const float w[4] = {dv_acc[0] / kLiftP<TF>, dv_acc[1] / kLiftP<TF>, dv_acc[2] / kLiftP<TF>, dv_acc[3] / kLiftP<TF>};
                if (unit.tiles > 1) {
                    const int2 entry = b.list.entries[unit.entry];
                    if (window_fits(entry, n_w, b.pairs)) {
                        float *part = b.parts + ((part_row(entry) + static_cast<int64_t>(unit.tile) * n_w + block * unit.size + column) * H + h) * (2 * D) + group16 * 4;
                        store4(part, o);
                        store4(part + D, w);
                    }
                } else {
                    const int64_t at = static_cast<int64_t>(b.rows[u * kCols + column]) * HD + h * D + group16 * 4;
                    store4(static_cast<TF *>(b.dk) + at, o);
                    store4(static_cast<TF *>(b.dv) + at, w);
                }
            }
        }
        if (!low) {
            const int n16 = tid & 15, group16 = (tid & 63) >> 4, i = quarter * 16 + n16;
            if (i < cols) {
                const float o[4] = {dq_sum[0], dq_sum[1], dq_sum[2], dq_sum[3]};
                store4(static_cast<TF *>(b.dq) + static_cast<int64_t>(b.rows[u * kCols + i]) * HD + h * D + group16 * 4, o);
            }
        }
    }
    if (__syncthreads_or(incomplete))
        for (int t = tid; t < 3 * kKind; t += kThreads) slot[t] = __int_as_float(0x7fc00000);
}

// ---- finish -----------------------------------------------------------------------------------------------------------
// The first workgroups add up the slots, a thread per word of a head's slots; the others the parts of dk and dv of
// windows of several tiles, a workgroup per tile of keys and quarter of its channels.
template <typename TF, int ND>
__global__ __launch_bounds__(256) void tile_finish_kernel(BwdTileArgs b, int table_groups)
{
    constexpr int kSt = Stages<ND>::kCount;
    const AttnArgs &a = b.f;
    const int HD = a.H * D, total_units = b.list.total[0];
    if (static_cast<int>(blockIdx.x) < table_groups) {
        const int t = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
        const int word = t % (3 * kSt * kCols * D), h = t / (3 * kSt * kCols * D);
        const int e = word % 4, lane = word / 4 % 64, quarter = word / 256 % 4, st = word / 1024 % kSt, kind = word / 1024 / kSt;
        if (h >= a.H) return;
        const int row = quarter * 16 + lane / 16 * 4 + e, c = lane % 16;
        const int axis = st < 3 ? st : Stages<ND>::first(st) + row / 32, r = st < 3 ? row : row % 32;
        if (axis >= ND || r >= axis_rows<ND>(a, axis)) return;
        const float *from = b.slots + static_cast<int64_t>(h) * (3 * kSt * kCols * D) + word;
        const int64_t step = static_cast<int64_t>(a.H) * (3 * kSt * kCols * D);
        const int used = min(b.groups, total_units);
        float sum = 0.0f;
#pragma unroll 8
        for (int g = 0; g < used; ++g) sum += from[g * step];
        (kind == 0 ? b.dtq : kind == 1 ? b.dtk : b.dtv)[static_cast<int64_t>(axis_base<ND>(a, axis) + r) * HD + h * D + c] = sum;
        return;
    }
    const int first = static_cast<int>(blockIdx.x) - table_groups, groups = static_cast<int>(gridDim.x) - table_groups;
    const int quads = 2 * HD / 4, share = (quads + 3) / 4;        // four channels of dk or dv
    for (int w = first; w < 4 * total_units; w += groups) {
        const Unit unit(b.list.units[w / 4]);
        if (unit.tiles <= 1) return;         // the units of several tiles come first
        const int2 entry = b.list.entries[unit.entry];
        const bool complete = window_fits(entry, unit.n_w, b.pairs);
        const int x0 = w % 4 * share, here = min(share, quads - x0);
        for (int t = threadIdx.x; t < unit.cols * here; t += 256) {
            const int key = unit.tile * unit.size + t / here, x = x0 + t % here;
            const int h = x / (2 * D / 4), q4 = x % (2 * D / 4);
            const float *from = b.parts + ((part_row(entry) + key) * a.H + h) * (2 * D) + q4 * 4;
            const int64_t step = static_cast<int64_t>(unit.n_w) * a.H * (2 * D);
            float o[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (complete) {
#pragma unroll 4
                for (int z = 0; z < unit.tiles; ++z) {
                    const float4 p = *reinterpret_cast<const float4 *>(from + z * step);
                    o[0] += p.x; o[1] += p.y; o[2] += p.z; o[3] += p.w;
                }
            } else {
                o[0] = o[1] = o[2] = o[3] = __int_as_float(0x7fc00000);
            }
            const int pos = entry.x + key;
            const int64_t row = a.n2n ? a.n2n[pos] : pos;
            store4(static_cast<TF *>(q4 < D / 4 ? b.dk : b.dv) + row * HD + h * D + q4 % (D / 4) * 4, o);
        }
    }
}

int bwd_groups(int H)
{
    const int slots = 2 * device_cus();
    return slots >= H ? slots / H : 1;
}

template <typename T, typename TF, int ND>
int launch_bwd(const BwdTileArgs &b0, hipStream_t stream)
{
    BwdTileArgs b = b0;
    const AttnArgs &a = b.f;
    b.groups = bwd_groups(a.H);
    constexpr uint32_t lds_r = RecordsLayout<ND>::kBytes, lds_g = GradLayout<TF, ND>::kBytes;
    static_assert(Stages<ND>::kCount * 128 <= kListThreads, "an operand per thread");
    static_assert(lds_r <= 80 * 1024 && lds_g <= 80 * 1024, "two workgroups per CU");
    auto records = tile_records_kernel<T, TF, ND>;
    auto gradients = tile_gradients_kernel<T, TF, ND>;
    if (int rc = allow_dynamic_lds(reinterpret_cast<const void *>(records), lds_r)) return rc;
    if (int rc = allow_dynamic_lds(reinterpret_cast<const void *>(gradients), lds_g)) return rc;
    const dim3 grid(static_cast<unsigned>(b.groups * a.H));
    hipLaunchKernelGGL((tile_setup_kernel<T, TF, ND>), dim3(static_cast<unsigned>(1 + 5 * a.H)), dim3(kListThreads), 0, stream, b);
    const int64_t most_units = static_cast<int64_t>(list_max_units(a.N));
    hipLaunchKernelGGL(tile_columns_kernel<ND>, dim3(static_cast<unsigned>(ceil_div(most_units, 4))), dim3(256), 0, stream, b);
    hipLaunchKernelGGL(records, grid, dim3(kThreads), lds_r, stream, b);
    hipLaunchKernelGGL(gradients, grid, dim3(kThreads), lds_g, stream, b);
    const int table_groups = static_cast<int>(ceil_div(int64_t(3) * Stages<ND>::kCount * kCols * D * a.H, 256));
    const int64_t tiles = 4 * (a.N / 32 + 1);
    const int part_groups = static_cast<int>(tiles < 2048 ? tiles : 2048);
    hipLaunchKernelGGL((tile_finish_kernel<TF, ND>), dim3(static_cast<unsigned>(table_groups + part_groups)), dim3(256), 0, stream,
                       b, table_groups);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

size_t slots_bytes(int H, int nd)
{
    const int stages = 3 + (nd - 3 + 1) / 2;
    return align_up(sizeof(float) * static_cast<size_t>(bwd_groups(H)) * H * 3 * stages * kCols * D, 256);
}

// row, first pair and coordinates of the units' columns
size_t columns_bytes(int64_t N, int nd) { return align_up(sizeof(int32_t) * list_max_units(N) * kCols * (2 + static_cast<size_t>(nd)), 256); }

// tables as operands, at most 48 bytes a lane, and their scales
size_t operand_bytes(int H, int nd)
{
    return align_up(sizeof(Operand<float>) * static_cast<size_t>(H) * 5 * (3 + (nd - 3 + 1) / 2) * 128, 256) +
           align_up(sizeof(float) * 5 * static_cast<size_t>(H), 256);
}

}  // namespace
}  // namespace tile

// Every shape whose tables fit a stage: of windows of 1 to 300 voxels in sets of 300 to 60,000, with 3 and 9 axes and all
// three types, the pair sweeps were faster in none (fp16: tiles take 0.14 to 0.53 of their time; fp32: 0.17 to 0.95, the
// most at 4 to 20 voxels a window and three axes).  At head_dim 8 there is no tile form: half of the 16 terms of a product
// would be empty while a pair's cost on a tile is the same, and the sweeps' rows are half as long.
bool attn_tile_bwd_applies(const int32_t *rows, int nd, int D, int64_t pairs)
{
    return D == 16 && pairs > 0 && pairs < (int64_t(1) << 31) && rows_fit_tiles(rows, nd);
}

size_t attn_tile_bwd_bytes(int H, int nd, int64_t N, int64_t W, int64_t pairs)
{
    return align_up(sizeof(float2) * static_cast<size_t>(H) * pairs, 256) +
           align_up(sizeof(float) * static_cast<size_t>(pairs / 64 + N) * H * 2 * tile::D, 256) + tile::slots_bytes(H, nd) +
           tile::operand_bytes(H, nd) + tile::columns_bytes(N, nd) + tile::list_bytes(N, W);
}

int launch_attn_tile_bwd(const BwdPairArgs &p, const void *out, float *dtq, float *dtk, float *dtv, void *workspace, int dtype,
                         hipStream_t stream)
{
    tile::BwdTileArgs b{};
    b.f = p.f;
    const int H = p.f.H, nd = p.f.nd;
    char *at = static_cast<char *>(workspace);
    b.records = reinterpret_cast<float2 *>(at);
    at += align_up(sizeof(float2) * static_cast<size_t>(H) * p.pairs, 256);
    b.parts = reinterpret_cast<float *>(at);
    at += align_up(sizeof(float) * static_cast<size_t>(p.pairs / 64 + p.f.N) * H * 2 * tile::D, 256);
    b.slots = reinterpret_cast<float *>(at);
    at += tile::slots_bytes(H, nd);
    b.operands = at;
    at += tile::operand_bytes(H, nd);
    b.scales = reinterpret_cast<float *>(at - align_up(sizeof(float) * 5 * static_cast<size_t>(H), 256));
    const size_t columns = tile::list_max_units(p.f.N) * tile::kCols;
    b.rows = reinterpret_cast<int32_t *>(at);
    b.first_pair = b.rows + columns;
    b.coords = reinterpret_cast<float *>(b.first_pair + columns);
    at += tile::columns_bytes(p.f.N, nd);
    b.list = tile::list_at(at, p.f.N, p.f.W);
    b.dout = p.dout;
    b.out = out;
    b.stat_max = p.stat_max;
    b.stat_sum = p.stat_sum;
    b.pairs = p.pairs;
    b.dq = p.dq; b.dk = p.dk; b.dv = p.dv;
    b.dtq = dtq; b.dtk = dtk; b.dtv = dtv;
#define S3D_CASE(NN)                                                                                           \
    if (nd == NN)                                                                                              \
        return dtype == S3D_DTYPE_F32   ? tile::launch_bwd<float, float, NN>(b, stream)                        \
               : dtype == S3D_DTYPE_F16 ? tile::launch_bwd<__half, __half, NN>(b, stream)                      \
                                        : tile::launch_bwd<float, __half, NN>(b, stream);
    S3D_CASE(3) S3D_CASE(6) S3D_CASE(9)
#undef S3D_CASE
    return fail(S3D_ERR_UNSUPPORTED, "s3d_attn_bwd: %d axes in the tile form", nd);
}

}  // namespace s3d
