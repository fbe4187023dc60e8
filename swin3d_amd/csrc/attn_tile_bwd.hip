// Attention backward at head_dim 16 (gfx950): dL and P of every pair, on tiles of up to 64 queries by 64 keys of a head, in fp32
// and of small windows; other fp16 features run on strips (attn_strip_records.hip).  The mathematics is in attn_bwd.hip, what is a
// sum over pairs in attn_strip_bwd.hip.
//
// tile_records_kernel, on the forward's unit list, makes the logits again and dP = dout_i . (v_j + Tv(i,j)) as the forward's
// tile kernel makes its logits: the products of the tile's queries (q with Tq, dout with Tv) and keys (k with Tk) with all
// rows of an axis come from the matrix pipe and stay in LDS, where every pair picks its three.  It leaves dL and P of every
// (pair, head): 8 bytes at [head][pairs before the window + j n + i].
//
// Why tiles: one form for every window size, since a unit packs windows of up to 64 voxels side by side; and an operand of three
// bf16 numbers makes a product six instructions, which tiles of 32 by 32 take at twice the rate of the strips' 16 by 16.  fp32 on
// strips, layers of 6,000 to 49,682 voxels: 1.03 to 1.07 times as long, forward included, with 64 keys at a time, 1.1 to 1.3 with 96
// (registers).
#include "attn_strip.h"

#include <algorithm>
#include <type_traits>

namespace s3d {
namespace tile {
namespace {

// What the matrix products are made of: features (TF) as they are, and tables (T) in the same type, or fp32 tables beside
// fp16 features as pairs of fp16 numbers.
template <typename T, typename TF> struct TableOperand { using type = Operand<T>; };
template <> struct TableOperand<float, __half> { using type = Pair16; };

struct BwdTileArgs : RecordsCall {
    int32_t *rows, *first_pair; // [unit][column]: the units' voxels, their rows and, of the pairs of their windows, the one
                                // with the window's first key (-1: beyond the records); see tile_columns_kernel
    float *coords;              // [unit][axis][column]
    int32_t groups;             // workgroups per head
};

// ---- setup ------------------------------------------------------------------------------------------------------------
// The unit list (workgroup 0) and, a workgroup for each head and table, the tables as the lanes' matrix operands:
// [head][q, k, v][stage][half][lane], table row lane % 32 of the half, channels 8 (lane / 32) ..
template <typename T, typename TF, int ND>
__global__ __launch_bounds__(kListThreads) void tile_setup_kernel(BwdTileArgs b)
{
    using S = Stages<ND>;
    using Table = typename TableOperand<T, TF>::type;
    const AttnArgs &a = b.f;
    if (blockIdx.x == 0) {
        build_list(a.w_sizes, a.w2n, static_cast<int>(a.W), const_cast<int32_t *>(b.list.total),
                   const_cast<int4 *>(b.list.units), const_cast<int2 *>(b.list.entries), const_cast<int4 *>(b.list.strips));
        return;
    }
    const int job = static_cast<int>(blockIdx.x) - 1, kind = job % 3, h = job / 3, HD = a.H * D;
    const T *table = static_cast<const T *>(kind == 0 ? a.table_q : kind == 1 ? a.table_k : a.table_v) + h * D;
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
    if (threadIdx.x == 0) b.scales[h * 3 + kind] = 1.0f / scale;
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
            const int r = row0 + lane % 32, c = lane / 32 * 8 + e;
            v[e] = table[static_cast<int64_t>(first + min(r, rows - 1)) * HD + c];
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
    const int s = u * (64 / kStrip) + c / kStrip;
    if (s < b.list.total[1]) {
        const int4 strip = b.list.strips[s];
        const int col = strip.z + min(c % kStrip, strip.w - 1);
        const int2 entry = b.list.entries[strip.x + col / strip.y];
        const int pos = entry.x + col % strip.y, row = a.n2n ? a.n2n[pos] : pos;
        b.strip_columns[s * kStrip + c % kStrip] = make_int4(pos, row, entry.x, window_fits(entry.y, strip.y, b.pairs) ? entry.y : -1);
        b.strip_rows[s * kStrip + c % kStrip] = row;
    }
    if (u >= b.list.total[0]) return;
    const Unit unit(b.list.units[u]);
    const int cc = max(0, min(c, unit.cols - 1));
    const int2 entry = unit.entry_of(b.list, cc);
    const int in = unit.inside(unit.tile, cc), pos = entry.x + in;
    b.rows[u * kCols + c] = a.n2n ? a.n2n[pos] : pos;
    b.first_pair[u * kCols + c] = window_fits(entry.y, unit.n_w, b.pairs) ? entry.y + in : -1;
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
    using Table = typename TableOperand<T, TF>::type;
    constexpr bool kScaled = std::is_same<Table, Pair16>::value;
    using L = RecordsLayout<ND>;
    using S = Stages<ND>;
    const AttnArgs &a = b.f;
    extern __shared__ __align__(16) float smem[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int H = a.H, HD = H * D;
    const uint64_t stride = static_cast<uint32_t>(a.row_stride);      // of q, k, v
    const int h = static_cast<int>(blockIdx.x) % H;
    const int group = static_cast<int>(blockIdx.x) / H, groups = static_cast<int>(gridDim.x) / H;
    const int total_units = b.list.total[0];

    const uint32_t queries = lds_base(smem), keys = queries + L::kQueries, coords = keys + L::kKeys;
    const TF *gq = static_cast<const TF *>(a.q), *gk = static_cast<const TF *>(a.k), *gv = static_cast<const TF *>(a.v);
    const TF *gd = static_cast<const TF *>(b.dout), *go = static_cast<const TF *>(b.out);
    const Table *operands = static_cast<const Table *>(b.operands) + static_cast<int64_t>(h) * (3 * S::kCount * 128);
    const float scale_q = kScaled ? b.scales[h * 3] : 1.0f, scale_k = kScaled ? b.scales[h * 3 + 1] : 1.0f, scale_v = kScaled ? b.scales[h * 3 + 2] : 1.0f;
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
        float own_max, own_inv, own_delta = 0.0f, own_grad = 0.0f;
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
                for (int e = 0; e < 8; ++e) {
                    own_delta += x[e] * y[e];
                    own_grad = finite(x[e]) ? own_grad : __int_as_float(0x7fc00000);
                }
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
                feat.load((wave < 4 ? gq : gk) + row * stride + channel);
                if (wave < 4) {
                    const uint64_t key_row = static_cast<uint32_t>(b.rows[other * kCols + tile_r * 32 + m32]);
                    grad.load(gd + row * HD + channel);
                    x_k.load(gk + key_row * stride + channel);
                    x_v.load(gv + key_row * stride + channel);
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
                        // (the long sum is rounded once an axis)
                        logit[s] += kScaled ? fmaf(k, scale_k, x.x * scale_q) : k + x.x;
                        dp[s] = kScaled ? fmaf(x.y, scale_v, dp[s]) : dp[s] + x.y;
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
                    // (and a query whose dout is not finite has no weights: the products that follow take its dout as zeros)
                    *to = make_float2(finite(logit[s]) ? p * (dp[s] - own_delta) : __int_as_float(0x7fc00000), p + own_grad);
                }
                to += reach * n_w;
            }
        }
    }
}

int bwd_groups(int H)
{
    const int slots = 2 * device_cus();
    return slots >= H ? slots / H : 1;
}

template <typename T, typename TF, int ND>
int launch_records(const BwdTileArgs &b0, hipStream_t stream)
{
    BwdTileArgs b = b0;
    const AttnArgs &a = b.f;
    b.groups = bwd_groups(a.H);
    constexpr uint32_t lds = RecordsLayout<ND>::kBytes;
    static_assert(Stages<ND>::kCount * 128 <= kListThreads, "an operand per thread");
    static_assert(lds <= 80 * 1024, "two workgroups per CU");
    auto records = tile_records_kernel<T, TF, ND>;
    if (int rc = allow_dynamic_lds(reinterpret_cast<const void *>(records), lds)) return rc;
    const dim3 grid(static_cast<unsigned>(b.groups * a.H));
    hipLaunchKernelGGL((tile_setup_kernel<T, TF, ND>), dim3(static_cast<unsigned>(1 + 3 * a.H)), dim3(kListThreads), 0, stream, b);
    const int64_t most_units = std::max<int64_t>(list_max_units(a.N), ceil_div(static_cast<int64_t>(list_max_strips(a.N)), 64 / kStrip));
    hipLaunchKernelGGL(tile_columns_kernel<ND>, dim3(static_cast<unsigned>(ceil_div(most_units, 4))), dim3(256), 0, stream, b);
    hipLaunchKernelGGL(records, grid, dim3(kThreads), lds, stream, b);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

// row, first pair and coordinates of the units' columns
size_t columns_bytes(int64_t N, int nd) { return align_up(sizeof(int32_t) * list_max_units(N) * kCols * (2 + static_cast<size_t>(nd)), 256); }

// tables as operands
size_t operand_bytes(int H, int nd) { return align_up(sizeof(Operand<float>) * static_cast<size_t>(H) * 3 * (3 + (nd - 3 + 1) / 2) * 128, 256); }
size_t scales_bytes(int H) { return align_up(sizeof(float) * 3 * static_cast<size_t>(H), 256); }

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

// Where strips leave the records: fp16 features, windows of some size (a strip is of one window).  Strips over tiles, forward
// included, layers of 60,000 to 100,000 voxels: 1.26 to 1.32 with windows of 4, 0.99 to 1.04 of 10, 0.91 to 0.95 of 17; fp32 see
// above.  The backward alone, windows of 30 to 98, 6 to 40 heads, by voxels (least, mean, most; fp32 tables | fp16 tables with 9 axes |
// with 6): 98 to 811 0.78 0.87 0.94 | 0.78 0.87 0.94 | 0.78 0.89 0.97; 1,500 to 3,100 0.83 0.92 0.97 | 0.83 0.92 0.97 | 0.86 0.94 1.00;
// 4,700 to 6,000 0.90 0.95 0.99 | 0.92 0.96 0.99 | 0.93 0.97 1.00; 9,400 to 75,000 0.94 0.98 1.02 | 0.96 0.99 1.02 | 0.97 1.01 1.04.
constexpr int64_t kStripRecordsMeanWindow = 14;

// records | slots | lists | strips and their columns | scales | what the kernel that leaves the records has
size_t attn_tile_bwd_bytes(int H, int nd, int64_t N, int64_t W, int64_t pairs)
{
    return align_up(sizeof(float2) * static_cast<size_t>(H) * pairs, 256) + tile::strip_slots_bytes(H, nd) + tile::list_bytes(N, W) +
           tile::strips_bytes(N) + tile::strip_columns_bytes(N) + tile::scales_bytes(H) +
           std::max(tile::operand_bytes(H, nd) + tile::columns_bytes(N, nd), tile::strip_records_bytes(H, nd, N, W));
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
    float *slots = reinterpret_cast<float *>(at);
    at += tile::strip_slots_bytes(H, nd);
    b.list = tile::list_at(at, p.f.N, p.f.W);
    at += tile::list_bytes(p.f.N, p.f.W);
    b.list.strips = reinterpret_cast<const int4 *>(at);
    at += tile::strips_bytes(p.f.N);
    b.strip_columns = reinterpret_cast<int4 *>(at);
    b.strip_rows = reinterpret_cast<int32_t *>(b.strip_columns + tile::kStrip * tile::list_max_strips(p.f.N));
    at += tile::strip_columns_bytes(p.f.N);
    b.scales = reinterpret_cast<float *>(at);
    at += tile::scales_bytes(H);
    b.dout = p.dout;
    b.out = out;
    b.stat_max = p.stat_max;
    b.stat_sum = p.stat_sum;
    b.pairs = p.pairs;
    int rc = fail(S3D_ERR_UNSUPPORTED, "s3d_attn_bwd: %d axes in the tile form", nd);
    if (dtype == S3D_DTYPE_F32 || p.f.N < kStripRecordsMeanWindow * p.f.W) {
        b.operands = at;
        const size_t columns = tile::list_max_units(p.f.N) * tile::kCols;
        b.rows = reinterpret_cast<int32_t *>(at + tile::operand_bytes(H, nd));
        b.first_pair = b.rows + columns;
        b.coords = reinterpret_cast<float *>(b.first_pair + columns);
#define S3D_CASE(NN)                                                                                           \
    if (nd == NN)                                                                                              \
        rc = dtype == S3D_DTYPE_F32   ? tile::launch_records<float, float, NN>(b, stream)                      \
             : dtype == S3D_DTYPE_F16 ? tile::launch_records<__half, __half, NN>(b, stream)                    \
                                      : tile::launch_records<float, __half, NN>(b, stream);
        S3D_CASE(3) S3D_CASE(6) S3D_CASE(9)
#undef S3D_CASE
    } else {
        rc = tile::launch_strip_records(b, at, dtype, stream);
    }
    if (rc) return rc;
    tile::StripArgs g{};
    g.f = p.f;
    g.list = b.list;
    g.dout = p.dout;
    g.records = b.records;
    g.pairs = p.pairs;
    g.columns = b.strip_columns;
    g.column_rows = b.strip_rows;
    g.scales = b.scales;
    g.slots = slots;
    g.dq = p.dq; g.dk = p.dk; g.dv = p.dv;
    g.grad_stride = static_cast<uint32_t>(p.grad_stride);
    g.dtq = dtq; g.dtk = dtk; g.dtv = dtv;
    return tile::launch_strip_gradients(g, dtype, stream);
}

}  // namespace s3d
