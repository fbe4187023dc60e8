// Attention backward at head_dim 16, fp16 features (gfx950): dL and P of every pair, on strips of up to 16 queries of a window and
// a head.  The mathematics is in attn_bwd.hip, what is a sum over pairs in attn_strip_bwd.hip; fp32 and small windows run on tiles
// (attn_tile_bwd.hip, with the rule).
//
// strip_records_kernel makes the logits again and dP = dout_i . (v_j + Tv(i,j)) as the forward's strip kernel makes its logits:
// the products of the strip's queries (q with Tq, dout with Tv) and of up to 96 keys (k with Tk) with 128 table rows at a time
// come from the matrix pipe and stay in LDS, where every pair picks its three; q . k and dout . v are a lane's own results.  It
// leaves dL and P of every (pair, head): 8 bytes at [head][pairs before the window + j n + i].
//
// What bounds it: nothing by itself; the VALU issues for 48 % of the time, the address unit works for 53, the LDS for 36, the matrix
// pipe for 20, and a wavefront waits for 38 %.  12,421 voxels in windows of 72, 9 axes, 12 heads, fp32 tables beside fp16 features:
// 178 us, where tiles of 64 x 64 pairs took 196 (480,000 clocks, 398,000 here): a window of 72 is two such tiles of 36, whose
// products are made at 64 x 64 (by size, against tiles: see the rule).  With 64 keys at a time, and so two blocks a window, 212
// us; with the next item's features asked for behind the last stage, 189.
#include "attn_strip.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace s3d {
namespace tile {
namespace {

template <typename T> using TableOperand = typename StripTable<T, __half>::type;

struct RecordsArgs : RecordsCall {
    WindowStrips window_strips;
    float half_rows[kMaxAxes], upper[kMaxAxes];    // what crse_row takes
};

// ---- setup ------------------------------------------------------------------------------------------------------------
// The lists (workgroups 0 and 1) and, a workgroup for each head and table, the tables as the lanes' matrix operands:
// [head][q, k, v][stage][wavefront][lane]: row lane % 16 of the wavefront's tile of the stage, of q and v in the order in which
// rows of products are stored side by side (see the kernel), channels 4 (lane / 16) ..
template <typename T, int ND>
__global__ __launch_bounds__(kListThreads) void records_setup_kernel(RecordsArgs b)
{
    using Table = TableOperand<T>;
    const AttnArgs &a = b.f;
    if (blockIdx.x == 0) {
        build_list(a.w_sizes, a.w2n, static_cast<int>(a.W), const_cast<int32_t *>(b.list.total), nullptr,
                   const_cast<int2 *>(b.list.entries), const_cast<int4 *>(b.list.strips));
        return;
    }
    if (blockIdx.x == 1) {
        build_window_strips(a.w_sizes, a.w2n, static_cast<int>(a.W), const_cast<int32_t *>(b.window_strips.total),
                            const_cast<int4 *>(b.window_strips.strips));
        return;
    }
    const int job = static_cast<int>(blockIdx.x) - 2, kind = job % 3, h = job / 3, HD = a.H * D;
    const T *table = static_cast<const T *>(kind == 0 ? a.table_q : kind == 1 ? a.table_k : a.table_v) + h * D;
    float scale = 1.0f;
    if constexpr (std::is_same<Table, Parts4<__half>>::value) {
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
    for (int t = threadIdx.x; t < kOwnTiles<ND> * kStripThreads; t += kListThreads) {
        const int lane = t % 64, tile = t / 64, axis = tile_axis(tile), c16 = lane & 15;
        float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (axis < ND) {
            const int r = min(tile_row0(tile) + (kind == 1 ? c16 : 4 * (c16 & 3) + (c16 >> 2)), axis_rows<ND>(a, axis) - 1);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = to_float(table[static_cast<int64_t>(axis_base<ND>(a, axis) + r) * HD + 4 * (lane >> 4) + e]);
        }
        Table x;
        if constexpr (std::is_same<Table, Parts4<__half>>::value) x.set(v, scale);
        else x.set(v);
        static_cast<Table *>(b.operands)[job * (kOwnTiles<ND> * kStripThreads) + t] = x;
    }
}

// The voxels of the strips that the sums over pairs go by, side by side.
__global__ __launch_bounds__(256) void records_columns_kernel(RecordsArgs b)
{
    const AttnArgs &a = b.f;
    const int t = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x), s = t / kStrip;
    if (s >= b.list.total[1]) return;
    const int4 strip = b.list.strips[s];
    const int col = strip.z + min(t % kStrip, strip.w - 1);
    const int2 entry = b.list.entries[strip.x + col / strip.y];
    const int pos = entry.x + col % strip.y, row = a.n2n ? a.n2n[pos] : pos;
    b.strip_columns[t] = make_int4(pos, row, entry.x, window_fits(entry.y, strip.y, b.pairs) ? entry.y : -1);
    b.strip_rows[t] = row;
}

// ---- records ----------------------------------------------------------------------------------------------------------
__device__ __forceinline__ f32x4_t dot4(const Raw4<__half> &x, const Raw4<__half> &y)
{
    f32x4_t p;
#pragma unroll
    for (int e = 0; e < 4; ++e) p[e] = static_cast<float>(x.x[e]) * static_cast<float>(y.x[e]);
    return p;
}

template <typename T, int ND>
__global__ __launch_bounds__(kStripThreads, 4) void strip_records_kernel(RecordsArgs b)
{
    using Table = TableOperand<T>;
    using TF = __half;
    using Feature = Exact4<TF>;
    const AttnArgs &a = b.f;
    constexpr int kKeyBlock = 96, kOwn = kOwnTiles<ND>, kReach = kStripThreads / kStrip, kKeySteps = kKeyBlock / kReach, kKeyTiles = kKeyBlock / 16;
    static_assert(kKeyTiles + 2 <= kStripWaves, "a wavefront an operand");
    constexpr int kStageRows = kStripWaves * 16, kProductStride = kStageRows + 4;      // (see attn_strip_fwd.hip)
    __shared__ __align__(16) float keys_s[kKeyBlock * kProductStride];       // k . Tk, [key][row]
    __shared__ __align__(16) float2 queries_s[kStageRows * kStrip];          // (q . Tq, dout . Tv), [row][query]
    __shared__ __align__(16) Feature features_s[kKeyTiles + 2][64];          // the keys as operands, q, dout
    __shared__ __align__(16) float4 stats_s[kStrip];                         // of a query: maximum, 1 / sum, dout . out, NaN where dout is not finite
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int H = a.H, HD = H * D;
    const int h = static_cast<int>(blockIdx.x) % H;
    const int group = static_cast<int>(blockIdx.x) / H, groups = static_cast<int>(gridDim.x) / H;
    const int4 first_strip = b.window_strips.strips[group];       // (there is room for it where there is no such strip)
    const int strips = b.window_strips.total[0];
    if (group >= strips) return;
    const uint32_t keys = lds_address(keys_s), queries = lds_address(queries_s);
    const int c16 = lane & 15, g4 = lane >> 4;
    const uint32_t stride = static_cast<uint32_t>(a.row_stride);      // of q, k, v
    const TF *gq = static_cast<const TF *>(a.q) + h * D, *gk = static_cast<const TF *>(a.k) + h * D, *gv = static_cast<const TF *>(a.v) + h * D;
    const TF *gd = static_cast<const TF *>(b.dout) + h * D, *go = static_cast<const TF *>(b.out) + h * D;
    auto load4 = [&](Raw4<TF> &r, const TF *x, int row, uint32_t pitch) {
        r.load(x + (static_cast<uint64_t>(static_cast<uint32_t>(row)) * pitch + static_cast<uint32_t>(opaque(4 * g4))));
    };
    const Table *operands = static_cast<const Table *>(b.operands) + static_cast<int64_t>(h) * (3 * kOwn * kStripThreads);
    const float scale_q = b.scales[h * 3], scale_k = b.scales[h * 3 + 1], scale_v = b.scales[h * 3 + 2];
    int tile_rows[kOwn];                           // of the axis of this wavefront's tile, from the tile on
#pragma unroll
    for (int i = 0; i < kOwn; ++i) {
        const int tile = i * kStripWaves + wave, axis = tile_axis(tile);
        tile_rows[i] = axis < ND ? axis_rows<ND>(a, axis) - tile_row0(tile) : 0;
    }

    // The items go through in steps: the rows of the one after the next are asked for, then the features of the next one, and,
    // when the present one's are not needed any more, its coordinates.
    struct Place { StripItem<kKeyBlock> item; int u; } now, next;
    struct Rows { int own, key, operand; } rows;
    Raw4<TF> own_k, own_v, operand, own_out;
    float own_max = 0.0f, own_sum = 1.0f, own[ND], other[kKeySteps];
    const int key0 = wave * (64 / kStrip) + g4;
    auto fetch_rows = [&](const StripItem<kKeyBlock> &i) {
        rows.own = i.pos0 + i.first + min(c16, i.cols - 1);
        rows.key = i.pos0 + i.first_key + min(wave * (64 / kStrip) + (c16 >> 2) + (c16 & 3) * kReach, i.keys_n - 1);
        rows.operand = i.pos0 + i.first_key + min(wave * 16 + c16, i.keys_n - 1);
        if (a.n2n) {
            if (wave >= kKeyTiles) rows.own = a.n2n[rows.own];
            rows.key = a.n2n[rows.key];
            if (wave < kKeyTiles) rows.operand = a.n2n[rows.operand];
        }
    };
    auto fetch = [&]() {
        if (wave < kKeyTiles) load4(operand, gk, rows.operand, stride);
        if (wave == kKeyTiles) load4(operand, gq, rows.own, stride);
        if (wave == kKeyTiles + 1) {
            load4(operand, gd, rows.own, HD);
            load4(own_out, go, rows.own, HD);
            own_max = b.stat_max[static_cast<int64_t>(rows.own) * H + h];
            own_sum = b.stat_sum[static_cast<int64_t>(rows.own) * H + h];
        }
        load4(own_k, gk, rows.key, stride);
        load4(own_v, gv, rows.key, stride);
    };
    auto fetch_coords = [&](const StripItem<kKeyBlock> &i) {
        load_coords<ND>(a.n_coords + static_cast<int64_t>(i.pos0 + i.first + min(c16, i.cols - 1)) * ND, own);
#pragma unroll
        for (int s = 0; s < kKeySteps; ++s)
            other[s] = a.n_coords[static_cast<int64_t>(i.pos0 + i.first_key + min(key0 + s * kReach, i.keys_n - 1)) * ND + min(c16, ND - 1)];
    };
    Table row_q, row_k, row_v;
    auto fetch_tables = [&](int st) {
        if (tile_rows[st] <= 0) return;
        const Table *from = operands + st * kStripThreads + tid;
        row_q = from[0];
        row_k = from[kOwn * kStripThreads];
        row_v = from[2 * kOwn * kStripThreads];
    };
    now.item.set(first_strip);
    now.u = group;
    fetch_rows(now.item);
    fetch_tables(0);
    fetch_coords(now.item);
    int4 strip_ahead = b.window_strips.strips[min(group + groups, strips - 1)];      // (behind the last one: the last one again)
    auto following = [&](const Place &p) {
        Place q = p;
        if (p.item.block + 1 == p.item.blocks) {
            q.u += groups;
            q.item.set(strip_ahead);
            strip_ahead = b.window_strips.strips[min(q.u + groups, strips - 1)];
        } else {
            q.item.set_block(p.item.block + 1);
        }
        return q;
    };
    fetch();
    next = following(now);
    fetch_rows(next.item);
    while (now.u < strips) {
        const StripItem<kKeyBlock> &item = now.item;
        const int keys_n = item.keys_n, n = item.n;
        const bool writes = c16 < item.cols && window_fits(item.pairs, n, b.pairs);
        float2 *to = b.records + (static_cast<int64_t>(h) * b.pairs + item.pairs + static_cast<int64_t>(item.first_key) * n + item.first + c16);
        auto has_step = [&](int s) { return wave * (64 / kStrip) + s * kReach < keys_n; };
        if (wave < kKeyTiles + 2) features_s[wave][lane] = Feature{operand.x};
        if (wave == kKeyTiles + 1) {
            const f32x4_t p = dot4(operand, own_out);
            float bad = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; ++e) bad = finite(static_cast<float>(operand.x[e])) ? bad : __int_as_float(0x7fc00000);
            const float delta = sum_columns((p[0] + p[1]) + (p[2] + p[3]));
            bad = sum_columns(bad);
            if (lane < kStrip) stats_s[c16] = make_float4(own_max, 1.0f / own_sum, delta, bad);
        }
        lds_barrier();
        const float4 stats = stats_s[c16];
        const Feature query = features_s[kKeyTiles][lane], grad = features_s[kKeyTiles + 1][lane];
        Feature key[kKeyTiles];
#pragma unroll
        for (int t = 0; t < kKeyTiles; ++t) key[t] = features_s[t][lane];
        uint32_t key_at[kKeySteps];
        float logit[kKeySteps], dp[kKeySteps];
        {
            const f32x4_t d = product(Feature{own_k.x}, query, f32x4_t{}), e = product(Feature{own_v.x}, grad, f32x4_t{});
#pragma unroll
            for (int s = 0; s < kKeySteps; ++s) {
                logit[s] = d[s];
                dp[s] = e[s];
                key_at[s] = keys + min(key0 + s * kReach, keys_n - 1) * (kProductStride * 4);
            }
        }
        fetch();
        const Place after = following(next);
        fetch_rows(after.item);
#pragma unroll
        for (int st = 0; st < kOwn; ++st) {
            if (st > 0) lds_barrier();
            if (tile_rows[st] > 0) {
                // (rows 4 e + g4 of the tile: the lanes' stores lie in banks of their own)
                const f32x4_t dl = product(row_q, query, f32x4_t{}), dv = product(row_v, grad, f32x4_t{});
                const uint32_t at = queries + ((wave * 16 + g4) * kStrip + c16) * 8;
#pragma unroll
                for (int e = 0; e < 4; ++e) lds_store2(at + 4 * e * kStrip * 8, dl[e], dv[e]);
#pragma unroll
                for (int t = 0; t < kKeyTiles; ++t)
                    if (t * 16 < keys_n)
                        *(lds_f32x4 *)(keys + (t * 16 + c16) * (kProductStride * 4) + (wave * 16 + 4 * g4) * 4) = product(row_k, key[t], f32x4_t{});
            }
            fetch_tables((st + 1) % kOwn);
            lds_barrier();
#pragma unroll
            for (int s = 0; s < kKeySteps; ++s) {
                if (!has_step(s)) break;
#pragma unroll
                for (int axis = 0; axis < ND; ++axis) {
                    if (axis_row0(axis) / kStageRows != st) continue;
                    const uint32_t r = static_cast<uint32_t>(crse_row(own[axis], of_sixteen(other[s], axis), b.half_rows[axis], b.upper[axis]));
                    const int first = axis_row0(axis) % kStageRows;
                    const float2 x = lds_load2(r * (kStrip * 8) + c16 * 8 + queries + first * (kStrip * 8));
                    const float k = lds_load(r * 4 + key_at[s] + first * 4);
                    logit[s] += fmaf(k, scale_k, x.x * scale_q);      // (the long sum is rounded once an axis)
                    dp[s] = fmaf(x.y, scale_v, dp[s]);
                }
            }
        }
        fetch_coords(next.item);
#pragma unroll
        for (int s = 0; s < kKeySteps; ++s) {
            const int j = key0 + s * kReach;
            const float p = __expf(logit[s] - stats.x) * stats.y;
            // (a logit of minus infinity has no weight, but its dL meets an infinite key or table row in dq)
            // (and a query whose dout is not finite has no weights: the products that follow take its dout as zeros)
            if (writes && j < keys_n) to[j * n] = make_float2(finite(logit[s]) ? p * (dp[s] - stats.z) : __int_as_float(0x7fc00000), p + stats.w);
        }
        now = next;
        next = after;
    }
}

template <typename T, int ND>
int launch_records(const RecordsArgs &b0, hipStream_t stream)
{
    RecordsArgs b = b0;
    const AttnArgs &a = b.f;
    for (int n = 0; n < ND; ++n) {
        b.half_rows[n] = static_cast<float>(a.rows[n] / 2);
        b.upper[n] = std::nextafterf(static_cast<float>(a.rows[n]), 0.0f);
    }
    // two workgroups per CU, no more than there may be strips
    const int64_t slots = std::max<int64_t>(1, 2 * device_cus() / a.H), most = static_cast<int64_t>(window_strips_most(a.N, a.W));
    const dim3 grid(static_cast<unsigned>(std::min(slots, most) * a.H));
    hipLaunchKernelGGL((records_setup_kernel<T, ND>), dim3(static_cast<unsigned>(2 + 3 * a.H)), dim3(kListThreads), 0, stream, b);
    const int64_t columns = static_cast<int64_t>(list_max_strips(a.N)) * kStrip;
    hipLaunchKernelGGL(records_columns_kernel, dim3(static_cast<unsigned>(ceil_div(columns, 256))), dim3(256), 0, stream, b);
    hipLaunchKernelGGL((strip_records_kernel<T, ND>), grid, dim3(kStripThreads), 0, stream, b);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

}  // namespace

// window strips | the tables as operands, at most 16 bytes a lane
size_t strip_records_bytes(int H, int nd, int64_t N, int64_t W)
{
    return 256 + align_up(sizeof(int4) * window_strips_most(N, W), 256) +
           align_up(sizeof(Parts4<__half>) * static_cast<size_t>(H) * 3 * tiles_of_axes(nd) * 64, 256);
}

int launch_strip_records(const RecordsCall &c, void *room, int dtype, hipStream_t stream)
{
    RecordsArgs b{};
    static_cast<RecordsCall &>(b) = c;
    char *at = static_cast<char *>(room);
    b.window_strips = {reinterpret_cast<const int32_t *>(at), reinterpret_cast<const int4 *>(at + 256)};
    b.operands = at + 256 + align_up(sizeof(int4) * window_strips_most(c.f.N, c.f.W), 256);
#define S3D_CASE(NN) \
    if (c.f.nd == NN) return dtype == S3D_DTYPE_F16 ? launch_records<__half, NN>(b, stream) : launch_records<float, NN>(b, stream);
    S3D_CASE(3) S3D_CASE(6) S3D_CASE(9)
#undef S3D_CASE
    return fail(S3D_ERR_UNSUPPORTED, "s3d_attn_bwd: %d axes in the strip form", c.f.nd);
}

}  // namespace tile
}  // namespace s3d
