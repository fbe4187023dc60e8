// Sparse-voxel windowed self-attention with cRSE tables (gfx950): the strip kernel of the forward, fp16, head_dim 16, for
// launches that do not fill the chip.
//
// A workgroup takes a strip of up to 16 queries of a window and a head, with up to 64 of the window's keys at a time.  The
// products of its queries and keys with all rows of the axis tables come from the matrix pipe, 128 rows (a tile of 16 for each
// wavefront) to a stage, and stay in LDS, where a pair picks its two words instead of gathering two rows of 32 bytes; the value
// tables enter through histograms of the weights over their rows, one column per query, as in attn_strip_bwd.hip.
//
// No unit bounds it (811 voxels x 24: the VALU issues for 37 % of the time, the LDS is addressed for 27, the address unit works for
// 26, the matrix pipe for 7): a launch of few strips is a chain of loads (list, row map, features: 9000 clocks to the first
// product) and then 9000 to 10,000 clocks for each block of keys, of which a wavefront waits for two fifths, at barriers.  811 voxels
// in windows of 90, 24 heads: 49 us on tiles of 64 x 64 pairs, which passed some thirty barriers a tile, 40 here, where a strip passes
// eight a block of keys and one more, seventeen in all; 390 voxels 33 -> 23, 98 voxels 26 -> 13.  The next strip's loads run ahead: every address that a wavefront's load touches takes a
// clock of the CU's address unit, and with coordinates by lane and each wavefront's own copies of the keys (22 loads a strip in
// place of 10) the same launches took 53, 30 and 16.
#include "attn_strip.h"

#include <algorithm>
#include <cmath>

namespace s3d {
namespace tile {
namespace {

__global__ __launch_bounds__(kListThreads) void strip_list_kernel(const int32_t *w_sizes, const int32_t *w2n, int W, int32_t *total, uint64_t *strips)
{
    build_strip_list<kListThreads>(w_sizes, w2n, W, total, strips);
}

struct FwdArgs {
    AttnArgs a;
    StripList list;
    float half_rows[kMaxAxes], upper[kMaxAxes];    // what crse_row takes
};

// Softmax weights.  A query's weights are at most 1 and sum to less than 2^e (e from their sum l).
//  * summed by table row: 32-bit integers in units of 2^(e-31), below 2^-31 of the sum of all weights, so that a cell keeps
//    what fp32 would whatever else falls into it, and no order of additions shows;
//  * beside a value: as they are, in fp32.
// They enter the matrix products over 2^(e - kLift) as two fp16 numbers, 23 bits from 2^15 down to 2^-3 and units of 2^-24
// below, which is 2^-39 of the sum.
constexpr int kCellBits = 31;
constexpr int kLift = 15;
constexpr float kCellScale = 1.0f / 65536.0f;      // 2^(kLift - kCellBits)

// A NaN or an infinity stays in its window, as on the sweep, though a matrix product takes all keys of a strip and all rows of
// a table, zero weights among them: a value or a value table's entry that is not finite goes into its operand as zero, and the
// sum of weights of the queries that it belongs to - those of its window, all of the head - becomes NaN, as that of a query
// with a NaN among its logits does by itself.  The result of such a query is stored as NaN, and a workgroup that has stored
// any goes through its strips once more and does over, pair by pair, what is NaN.

constexpr int kKeyBlock = 64;                      // keys that a strip takes on at a time
constexpr int kKeyTiles = kKeyBlock / 16, kKeySteps = (kKeyBlock * kStrip + kStripThreads - 1) / kStripThreads;
constexpr int kStageRows = kStripWaves * 16;       // table rows of a stage: a tile of 16 for each wavefront
// words between the products of one voxel and the next: 16-byte stores of 16 voxels meet in no bank
constexpr int kProductStride = kStageRows + 4;

template <int ND, bool kDeviceSizes>
__global__ __launch_bounds__(kStripThreads, 4) void attn_fwd_strip_kernel(FwdArgs f)
{
    using T = __half;
    const AttnArgs &a = f.a;
    constexpr int kOwn = kOwnTiles<ND>;            // stages, and tiles of 16 table rows of a wavefront: one a stage
    constexpr int kReach = kStripThreads / kStrip; // keys of a query that a step of the workgroup takes
    // products of a stage, [key][row] and [row][query]; the queries' give way to the wavefronts' parts of the result
    __shared__ __align__(16) float keys_s[kKeyBlock * kProductStride];
    __shared__ __align__(16) float queries_s[kStageRows * kStrip];
    static_assert(kStageRows * kStrip >= kStripWaves * 256, "room for the parts");
    __shared__ __align__(16) Exact4<T> features_s[kKeyTiles + 1][64];         // the keys as operands, and the queries
    __shared__ __align__(16) uint32_t cells_s[kTiles<ND> * 16 * kStrip];      // weights by table row, [row][query]
    __shared__ float2 states_s[kStripWaves][kStrip];                          // maximum and sum of a wavefront's pairs
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int H = a.H, HD = H * D;
    const int h = static_cast<int>(blockIdx.x) % H;
    const int group = static_cast<int>(blockIdx.x) / H, groups = static_cast<int>(gridDim.x) / H;
    const uint64_t first_strip = f.list.strips[group];       // (there is room for it where there is no such strip)
    const int strips = f.list.total[0];
    if (group >= strips) return;
    // rows and first row of every axis table: kernel arguments, or read from the caller's device tensor of table sizes.
    // The host has not seen those: it launched the sweep kernel as well, and this kernel leaves the call to it when an
    // axis has more rows than it has room for.
    int read_rows[ND], read_first[ND];
    if constexpr (kDeviceSizes) {
        int run = 0;
#pragma unroll
        for (int n = 0; n < ND; ++n) {
            read_first[n] = run;
            run += read_rows[n] = device_rows(a, n, ND, run);
        }
        if (!rows_fit_tiles(read_rows, ND)) return;
    }
    auto rows_n = [&](int n) { return kDeviceSizes ? read_rows[n] : a.rows[n]; };
    auto first_row = [&](int n) { return kDeviceSizes ? read_first[n] : a.base[n]; };
    auto half_rows = [&](int n) { return kDeviceSizes ? static_cast<float>(read_rows[n] / 2) : f.half_rows[n]; };
    auto upper = [&](int n) { return kDeviceSizes ? crse_upper(read_rows[n]) : f.upper[n]; };

    const uint32_t keys = lds_address(keys_s), queries = lds_address(queries_s), cells = lds_address(cells_s);
    const int c16 = lane & 15, g4 = lane >> 4;
    const uint32_t stride = static_cast<uint32_t>(a.row_stride);
    const T *gq = static_cast<const T *>(a.q) + h * D, *gk = static_cast<const T *>(a.k) + h * D, *gv = static_cast<const T *>(a.v) + h * D;
    // (the lane's channels in a form that the compiler does not add to the pointers for good, in two registers each)
    auto load4 = [&](Raw4<T> &r, const T *x, int row) {
        r.load(x + (static_cast<uint64_t>(static_cast<uint32_t>(row)) * stride + static_cast<uint32_t>(opaque(4 * g4))));
    };

    // A strip with a block of its window's keys is what the workgroup works off at a time.
    using Item = StripItem<kKeyBlock>;
    auto set = [](Item &i, uint64_t s) {
        const uint32_t lo = static_cast<uint32_t>(s), hi = static_cast<uint32_t>(s >> 32);
        constexpr uint32_t kMask = (1u << kPosBits) - 1;
        i.set(make_int4(static_cast<int>(lo & kMask), static_cast<int>((lo >> kPosBits | hi << (32 - kPosBits)) & kMask),
                        static_cast<int>(hi >> (2 * kPosBits - 32)), 0));
    };
    Item item;
    // Its rows, then its features and coordinates, are asked for while the item before is worked on.  A lane's pairs are those
    // of query c16 with the keys key0 + kReach s; as rows of a product the wavefront's keys are in the order in which its
    // result has them as these.  A key's coordinates are a number a lane of its sixteen: a broadcast among those is part of the
    // instruction that takes it.  One wavefront loads an operand that all take.
    struct Rows { int own, key, operand; } rows;
    Raw4<T> own_k, own_v, operand;
    float own[ND], other[kKeySteps];
    const int key0 = wave * (64 / kStrip) + g4;
    auto fetch_rows = [&](const Item &i) {
        rows.own = i.pos0 + i.first + min(c16, i.cols - 1);
        rows.key = i.pos0 + i.first_key + min(wave * (64 / kStrip) + (c16 >> 2) + (c16 & 3) * kReach, i.keys_n - 1);
        rows.operand = i.pos0 + i.first_key + min(wave * 16 + c16, i.keys_n - 1);
        if (a.n2n) {
            rows.own = a.n2n[rows.own];
            rows.key = a.n2n[rows.key];
            if (wave < kKeyTiles) rows.operand = a.n2n[rows.operand];
        }
    };
    auto fetch = [&](const Item &i) {
        if (wave <= kKeyTiles) load4(operand, wave == kKeyTiles ? gq : gk, wave == kKeyTiles ? rows.own : rows.operand);
        load4(own_k, gk, rows.key);
        load4(own_v, gv, rows.key);
        load_coords<ND>(a.n_coords + static_cast<int64_t>(i.pos0 + i.first + min(c16, i.cols - 1)) * ND, own);
#pragma unroll
        for (int s = 0; s < kKeySteps; ++s)
            other[s] = a.n_coords[static_cast<int64_t>(i.pos0 + i.first_key + min(key0 + s * kReach, i.keys_n - 1)) * ND + min(c16, ND - 1)];
    };
    set(item, first_strip);
    fetch_rows(item);

    // The tables: tile 8 i + wave is this wavefront's.  Row 4 e + g of the tile is row 4 g + e of an operand: the lanes that
    // store or read side by side then do so in different banks.
    Raw4<T> table_q[kOwn], table_k[kOwn], raw_v[kOwn];
    int tile_rows[kOwn];                           // of the tile's axis from the tile on; none are left where it is not above 0
#pragma unroll
    for (int i = 0; i < kOwn; ++i) {
        const int tile = i * kStripWaves + wave, axis = tile_axis(tile);
        int axis_rows = 0, axis_first = 0;
#pragma unroll
        for (int n = 0; n < ND; ++n)
            if (n == axis) { axis_rows = rows_n(n); axis_first = first_row(n); }
        tile_rows[i] = axis_rows - tile_row0(tile);
        // (of a tile without rows: a row that is there, and nothing is made of it)
        auto row_at = [&](int r) { return static_cast<int64_t>(axis_first + min(tile_row0(tile) + r, max(axis_rows, 1) - 1)) * HD + h * D + 4 * g4; };
        const int64_t by_four = row_at(4 * (c16 & 3) + (c16 >> 2));
        table_q[i].load(static_cast<const T *>(a.table_q) + by_four);
        table_k[i].load(static_cast<const T *>(a.table_k) + row_at(c16));
        raw_v[i].load(static_cast<const T *>(a.table_v) + by_four);
    }
    fetch(item);
    for (int t = tid; t < kTiles<ND> * 16 * kStrip / 4; t += kStripThreads) reinterpret_cast<uint4 *>(cells_s)[t] = make_uint4(0, 0, 0, 0);
    f16x4 identity;
#pragma unroll
    for (int e = 0; e < 4; ++e) identity[e] = static_cast<_Float16>(4 * g4 + e == c16 ? 1.0f : 0.0f);
    // [voxel or table row][channel] as [channel][...]; what is not finite as zeros
    auto by_channel = [&](const Raw4<T> &r, bool &bad, int rows) {
        const f32x4_t x = r.voxels(identity);
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const bool there = 4 * e + g4 < rows;
            bad = bad || (there && !finite(x[e]));
            v[e] = there && finite(x[e]) ? x[e] : 0.0f;
        }
        Exact4<T> y;
        y.set(v);
        return y;
    };
    Exact4<T> table_v[kOwn];
    bool bad_table = false;
#pragma unroll
    for (int i = 0; i < kOwn; ++i) table_v[i] = by_channel(raw_v[i], bad_table, tile_rows[i]);
    bad_table = __any(bad_table);

    bool again = false;
    f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};            // [channel][query], over 2^exponent
    float run_max = -INFINITY, run_sum = 0.0f;
    uint64_t strip_ahead = f.list.strips[min(group + groups, strips - 1)];
    for (int u = group; u < strips;) {
        const bool ends = item.block + 1 == item.blocks;
        const int keys_n = item.keys_n, own_row = rows.own;
        const bool there = c16 < item.cols;
        auto has_step = [&](int s) { return wave * (64 / kStrip) + s * kReach < keys_n; };
        if (wave <= kKeyTiles) features_s[wave][lane] = Exact4<T>{operand.x};
        bool bad_value = false;
        const Exact4<T> value = by_channel(own_v, bad_value, D);
        bad_value = __any(bad_value);
        // what follows
        const int u_next = ends ? u + groups : u;
        Item next = item;
        if (ends) {
            set(next, strip_ahead);
            strip_ahead = f.list.strips[min(u_next + groups, strips - 1)];
        } else {
            next.set_block(item.block + 1);
        }
        fetch_rows(next);
        lds_barrier();
        const Exact4<T> query = features_s[kKeyTiles][lane];
        Exact4<T> key[kKeyTiles];
#pragma unroll
        for (int t = 0; t < kKeyTiles; ++t) key[t] = features_s[t][lane];
        uint32_t key_at[kKeySteps], row_at[kKeySteps][ND];      // of the row of a pair's axis: 64 bytes a row, from the query on
        float logit[kKeySteps];
        {
            const f32x4_t d = product(Exact4<T>{own_k.x}, query, f32x4_t{});
#pragma unroll
            for (int s = 0; s < kKeySteps; ++s) {
                logit[s] = d[s];
                key_at[s] = keys + min(key0 + s * kReach, keys_n - 1) * (kProductStride * 4);
            }
        }
        // The stages: products of the queries and keys with 128 table rows, then every pair's own
#pragma unroll
        for (int st = 0; st < kOwn; ++st) {
            if (st > 0) lds_barrier();
            if (tile_rows[st] > 0) {
                const f32x4_t d = product(Exact4<T>{table_q[st].x}, query, f32x4_t{});
                const uint32_t to = queries + ((wave * 16 + g4) * kStrip + c16) * 4;
#pragma unroll
                for (int e = 0; e < 4; ++e) lds_store(to + 4 * e * kStrip * 4, d[e]);
#pragma unroll
                for (int t = 0; t < kKeyTiles; ++t)
                    if (t * 16 < keys_n)
                        *(lds_f32x4 *)(keys + (t * 16 + c16) * (kProductStride * 4) + (wave * 16 + 4 * g4) * 4) =
                            product(Exact4<T>{table_k[st].x}, key[t], f32x4_t{});
            }
            lds_barrier();
#pragma unroll
            for (int s = 0; s < kKeySteps; ++s) {
                if (!has_step(s)) break;
#pragma unroll
                for (int axis = 0; axis < ND; ++axis) {
                    if (axis_row0(axis) / kStageRows != st) continue;
                    const float its = of_sixteen(other[s], axis);
                    const uint32_t r = static_cast<uint32_t>(crse_row(own[axis], its, half_rows(axis), upper(axis)));
                    const int first = axis_row0(axis) % kStageRows;
                    row_at[s][axis] = r * (kStrip * 4) + c16 * 4;
                    logit[s] += lds_load(row_at[s][axis] + queries + first * (kStrip * 4)) + lds_load(r * 4 + key_at[s] + first * 4);
                }
            }
        }
        item = next;
        fetch(item);
        // softmax of the block: of the wavefront's pairs, then of all
        float top = -INFINITY, sum = 0.0f, p[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        auto valid = [&](int s) { return there && key0 + s * kReach < keys_n; };
#pragma unroll
        for (int s = 0; s < kKeySteps; ++s) top = valid(s) ? fmaxf(top, logit[s]) : top;
        top = max_columns(top);
#pragma unroll
        for (int s = 0; s < kKeySteps; ++s) {
            p[s] = valid(s) ? __expf(logit[s] - top) : 0.0f;
            sum += p[s];
        }
        sum = sum_columns(sum);
        if (bad_value || bad_table) sum = NAN;
        if (lane < kStrip) states_s[wave][c16] = make_float2(top, sum);
        lds_barrier();
        float l, m;
        {
            const float2 x = states_s[g4][c16], y = states_s[4 + g4][c16];
            m = max_columns(fmaxf(x.x, y.x));
            l = sum_columns(fmaf(x.y, __expf(x.x - m), y.y * __expf(y.x - m)));
        }
        const int exponent = exponent_of(l);
        const float to_all = __expf(top - m), fix = power2(kCellBits - exponent);
#pragma unroll
        for (int s = 0; s < kKeySteps; ++s) {
            p[s] = valid(s) ? p[s] * to_all : 0.0f;
            if (!has_step(s)) break;
            const uint32_t weight = static_cast<uint32_t>(rintf(p[s] * fix));
#pragma unroll
            for (int axis = 0; axis < ND; ++axis) {
                lds_add(row_at[s][axis] + cells + axis_row0(axis) * (kStrip * 4), weight);
            }
        }
        f32x4_t block_acc;
        {
            Parts4<T> c;
            c.set(p, power2(kLift - exponent));
            block_acc = product(value, c, f32x4_t{});
        }
        lds_barrier();
        const uint32_t cell_at = cells + ((wave * 16 + g4) * kStrip + c16) * 4;
#pragma unroll
        for (int i = 0; i < kOwn; ++i) {
            if (tile_rows[i] <= 0) continue;
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t at = cell_at + (i * kStageRows + e * 4) * (kStrip * 4);
                v[e] = static_cast<float>(lds_load_u32(at));
                lds_store_u32(at, 0u);
            }
            Parts4<T> c;
            c.set(v, kCellScale);
            block_acc = product(table_v[i], c, block_acc);
        }
        // into the queries' running softmax states
        const float m_all = fmaxf(run_max, m), w_run = __expf(run_max - m_all), w_block = __expf(m - m_all);
        const float w_acc = w_block * power2(exponent - kLift);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = fmaf(acc[e], w_run, block_acc[e] * w_acc);
        run_sum = fmaf(run_sum, w_run, l * w_block);
        run_max = m_all;
        u = u_next;
        if (!ends) continue;
        // the wavefronts' parts meet, and the result is stored
        again = again || (there && !(run_sum == run_sum));
        *reinterpret_cast<f32x4_t *>(&queries_s[(wave * 64 + lane) * 4]) = acc;
        const float inv = 1.0f / run_sum;
        acc = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        run_max = -INFINITY;
        run_sum = 0.0f;
        lds_barrier();
        if (wave == kStripWaves - 1) {
            float o[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int w = 0; w < kStripWaves; ++w) {
                const f32x4_t v = *reinterpret_cast<const f32x4_t *>(&queries_s[(w * 64 + lane) * 4]);
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] += v[e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] *= inv;
            if (there) store4(static_cast<T *>(a.out) + static_cast<int64_t>(own_row) * HD + h * D + 4 * g4, o);
        }
    }
    if (!__syncthreads_or(again)) return;
    for (int u = group; u < strips; u += groups) {
        set(item, f.list.strips[u]);
        const int i = tid >> 3;
        if (i >= item.cols) continue;
        const int pos = item.pos0 + item.first + i;
        const int64_t row = a.n2n ? a.n2n[pos] : pos;
        const float out = to_float(static_cast<const volatile T *>(a.out)[row * HD + h * D]);
        if (out == out) continue;
        float ci[ND];
#pragma unroll
        for (int n = 0; n < ND; ++n) ci[n] = a.n_coords[static_cast<int64_t>(pos) * ND + n];
        exact_query<T, ND>(a, h, row, item.pos0, item.n, tid & 7, ci, rows_n, first_row);
    }
}

template <int ND, bool kDeviceSizes>
int launch_fwd(const AttnArgs &a, const StripList &list, hipStream_t stream)
{
    FwdArgs f{};
    f.a = a;
    f.list = list;
    for (int n = 0; n < ND && !kDeviceSizes; ++n) {
        f.half_rows[n] = static_cast<float>(a.rows[n] / 2);
        f.upper[n] = std::nextafterf(static_cast<float>(a.rows[n]), 0.0f);
    }
    // two workgroups per CU, no more than there may be strips
    const int64_t slots = std::max<int64_t>(1, 2 * device_cus() / a.H);
    const int groups = static_cast<int>(std::min<int64_t>(slots, strip_list_most(a.N, a.W)));
    hipLaunchKernelGGL((attn_fwd_strip_kernel<ND, kDeviceSizes>), dim3(static_cast<unsigned>(groups * a.H)), dim3(kStripThreads), 0, stream, f);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

}  // namespace
}  // namespace tile

// Where the strip kernel serves a forward (fp16, head_dim 16): launches of few strips.  A strip takes a workgroup about 4 us
// whatever is in it, and two of them share a CU, where the sweep gives a query at most eight lanes and a launch that does not
// fill the chip ends when its longest unit ends.  Measured, strips over the sweep (or over the kernel on 64 x 64 tiles that
// served windows of 40 and more up to N^2 / W * H = 4 M), by (N / 16 + W) H, N / 16 + W being the most strips of a head:
//   windows of 24 to 98 voxels, 9 axes: 0.15 to 0.72 up to 2300 (98 voxels, 24 heads 63 -> 9 us and, in two windows, 26 -> 13;
//     1000 x 24 100 -> 33), 0.82 to 0.93 with 0.60 at 3000 x 12 up to 5500; over the sweep alone, 6 to 40 heads, 0.50 to 1.05, 0.91
//     in the mean, at 6000 to 7200, 0.56 to 1.07, 0.94 in the mean, at 7200 to 8000, 0.69 to 1.14, 0.99 in the mean, at 8000 to 8800,
//     1.1 to 1.24 at 11,000 and beyond; 6 axes: 0.16 to 0.91 up to 5500, 0.54 to 1.10, 0.95 in the mean, at 6000 to 7200, 0.63 to
//     1.12, 0.99 in the mean, at 7200 to 8000, 0.78 to 1.23 at 8000 to 8800, 1.15 to 1.31 beyond (the sweep's time jumps with its
//     cut into units, and the lines lie where strips lose little anywhere)
//   windows of 5 to 11 voxels: 0.30 to 0.70 up to 2800, 0.70 to 1.15 at 3000 to 3700, 1.10 to 1.68 at 5500 to 7500
//   windows of 18 to 24: 0.36 to 0.63 at 4000 to 6000, which the line at 24 still leaves to the sweep; nothing is recorded from 12 to 17
constexpr int64_t kStripsMost = 6000, kStripsMostNormals = 7200, kStripsMostSmall = 3000, kStripMeanWindowSmall = 24;

bool attn_strip_shape(int64_t N, int64_t W, int H, int nd)
{
    const int64_t most = N < kStripMeanWindowSmall * W ? kStripsMostSmall : nd < 9 ? kStripsMost : kStripsMostNormals;
    return W > 0 && N < (int64_t(1) << tile::kPosBits) && (N / tile::kStrip + W) * H <= most;
}

bool attn_strip_applies(const AttnArgs &a, int dtype)
{
    if (dtype != S3D_DTYPE_F16 || a.D != tile::D || !attn_strip_shape(a.N, a.W, a.H, a.nd)) return false;
    return a.sizes_dev || rows_fit_tiles(a.rows, a.nd);
}

tile::StripList attn_strip_list(const AttnArgs &a)
{
    char *at = static_cast<char *>(attn_sweep_notes(a)) + kSweepNotesKept;
    static_assert(kSweepNotesKept + 256 + sizeof(uint64_t) * kStripsMostNormals <= kSweepNotesBytes, "the list fits");
    return {reinterpret_cast<const int32_t *>(at), reinterpret_cast<const uint64_t *>(at + 256)};
}

int launch_attn_strip(const AttnArgs &a, hipStream_t stream, int what)
{
    using namespace tile;
    const StripList l = attn_strip_list(a);
    if (what & kAttnBuildList) {
        hipLaunchKernelGGL(strip_list_kernel, dim3(1), dim3(kListThreads), 0, stream, a.w_sizes, a.w2n, static_cast<int>(a.W),
                           const_cast<int32_t *>(l.total), const_cast<uint64_t *>(l.strips));
        S3D_HIP_CHECK(hipGetLastError());
    }
    if (!(what & kAttnSweep)) return S3D_OK;
#define S3D_CASE(NN) \
    if (a.nd == NN) return a.sizes_dev ? launch_fwd<NN, true>(a, l, stream) : launch_fwd<NN, false>(a, l, stream);
    S3D_CASE(3) S3D_CASE(6) S3D_CASE(9)
#undef S3D_CASE
    return fail(S3D_ERR_UNSUPPORTED, "s3d_attn_fwd: %d axes in the strip form", a.nd);
}

}  // namespace s3d
