// Sparse-voxel windowed self-attention with cRSE tables (gfx950): the tile kernel of the forward, fp32, head_dim 16.
//
// A workgroup takes 64 queries by 64 keys of a head.  The products of its queries and keys with all rows of an axis table
// come from the matrix pipe and stay in LDS, where a pair picks its two words instead of gathering two rows of 32 or 64
// bytes; the value tables enter through histograms of the weights over their rows, one column per query.  49,682 voxels, 6
// heads, 6 axes: 413 us (sweep) -> 398.  No unit is busy (VALU 53 % of the time, LDS addressed 33 %, matrix pipe 11 %): a tile
// goes through some thirty phases with a barrier each, and a wavefront waits for half of its time.  fp16 runs on strips
// (attn_strip_fwd.hip), which in fp32, with operands of three parts, took 1.6 to 2.5 times as long as tiles.
#include "attn_tile.h"

namespace s3d {
namespace tile {
namespace {

__global__ __launch_bounds__(kListThreads) void tile_list_kernel(const int32_t *w_sizes, const int32_t *w2n, int W, int32_t *total,
                                                                 int4 *units, int2 *entries)
{
    build_list(w_sizes, w2n, W, total, units, entries, nullptr);
}

struct FwdArgs {
    AttnArgs a;
    UnitList list;
};

// Softmax weights in a tile.  A query's weights are at most 1 and sum to less than 2^e (e from their sum l).
//  * their sum: 64-bit integers in units of 2^-57, which hold a thread's partial sum in fp32 as it is;
//  * summed by table row: 32-bit integers in units of 2^(e-31), below 2^-31 of the sum of all weights, so that a cell keeps
//    what fp32 would whatever else falls into it, and no order of additions shows;
//  * beside a value: as they are, in fp32.
// They enter the matrix products over 2^e, in full.
constexpr float kSumFix = 33554432.0f;               // 2^25: the high word of a sum, at most 64 weights
constexpr float kSumLow = 1.0f / 4294967296.0f;
constexpr int kCellBits = 31;
constexpr float kCellScale = 1.0f / 2147483648.0f;   // 2^-kCellBits

using T = float;
template <int ND> struct FwdLayout {
    static constexpr int kSt = Stages<ND>::kCount;
    static constexpr uint32_t kSums = kCols * kStride * 4;                       // a [row][column] array of fp32 or u32
    static constexpr uint32_t kKeys = kCols * kKeyStride * 4;                    // keys: coordinates and table products
    static constexpr uint32_t kTableT = kSt * D * kStride * sizeof(T);           // value table, [stage][channel][row]
    static constexpr uint32_t kValueT = D * kStride * sizeof(T);                 // values of the tile, [channel][key]
    static constexpr uint32_t kCoords = ND * kCols * 4;
    static constexpr uint32_t kMeta = 5 * kCols * 4 + 48;                        // sums (64 bits), rows of queries and keys, maxima, masks
    static constexpr uint32_t kBytes = kSums + kKeys + kTableT + kValueT + kCoords + kMeta;
};

// A NaN or an infinity stays in its window, as on the sweep, though a matrix product takes the keys of a whole unit and all
// rows of a table, zero weights among them: a value or a value table's entry that is not finite goes into its operand as
// zero, and the queries that it belongs to - those of its window, all of the head - are marked, as is a query with a logit
// that is not finite.  A marked query's result is stored as NaN, and a workgroup that has marked any goes through its units
// once more and does over, pair by pair, what is NaN.  (Done over inside the loop over units, it took the tiles 3 us of 45,
// in registers.)

template <int ND, bool kDeviceSizes>
__global__ __launch_bounds__(kThreads, 4) void attn_fwd_tile_kernel(FwdArgs f)
{
    using L = FwdLayout<ND>;
    using S = Stages<ND>;
    const AttnArgs &a = f.a;
    extern __shared__ __align__(16) float smem[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int H = a.H, HD = H * D;
    const int h = static_cast<int>(blockIdx.x) % H;
    const int group = static_cast<int>(blockIdx.x) / H, groups = static_cast<int>(gridDim.x) / H;
    const int total_units = f.list.total[0];
    if (group >= total_units) return;
    // rows and first row of every axis table: kernel arguments, or read from the caller's device tensor of table sizes.
    // The host has not seen those: it launched the sweep kernel as well, and this kernel leaves the call to it when an
    // axis has more rows than a stage holds.
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

    const uint32_t base = lds_base(smem);
    const uint32_t sums = base, keys = sums + L::kSums, table_t = keys + L::kKeys, value_t = table_t + L::kTableT;
    const uint32_t coords = value_t + L::kValueT, col_sum = coords + L::kCoords, row_i = col_sum + kCols * 8;
    const uint32_t row_j = row_i + kCols * 4, col_max = row_j + kCols * 4;
    const uint32_t marked = col_max + kCols * 4, bad_keys = marked + 8, bad_head = marked + 16;   // 64 bits, 64 bits, 8 words
    auto sum_of = [&](int c) {
        return fmaf(static_cast<float>(lds_load_u32(col_sum + c * 8)), kSumLow / kSumFix,
                    static_cast<float>(lds_load_u32(col_sum + c * 8 + 4)) * (1.0f / kSumFix));
    };

    const T *gq = static_cast<const T *>(a.q), *gk = static_cast<const T *>(a.k), *gv = static_cast<const T *>(a.v);
    const T *table_qk = static_cast<const T *>(wave < 4 ? a.table_q : a.table_k);
    {
        // the head's value table with the channels as rows, unused rows at zero
        bool bad_table = false;
        const T *tv = static_cast<const T *>(a.table_v);
        for (int x = tid; x < L::kSt * kCols * (D / 8); x += kThreads) {
            const int c8 = x % (D / 8), row = (x / (D / 8)) % kCols, st = x / (D / 8) / kCols;
            const int axis = S::first(st) + (st >= 3 && row >= 32 ? 1 : 0);
            const int r = st >= 3 ? row & 31 : row;
            int axis_rows = 0, axis_first = 0;
#pragma unroll
            for (int n = 0; n < ND; ++n)
                if (n == axis) { axis_rows = rows_n(n); axis_first = first_row(n); }
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = 0.0f;
            if (r < axis_rows) load_row<8>(tv + static_cast<int64_t>(axis_first + r) * HD + h * D + c8 * 8, v);
            T *to = reinterpret_cast<T *>(reinterpret_cast<char *>(smem) + (table_t - base)) +
                    (st * D + c8 * 8) * kStride + (row & 32) + permuted_row(row & 31);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                bad_table = bad_table || !finite(v[e]);
                to[e * kStride] = static_cast<T>(finite(v[e]) ? v[e] : 0.0f);
            }
        }
        // (a word per wavefront, cleared by its first lane: as a value of the thread it would sit in registers throughout)
        if ((tid & 63) == 0) lds_store_u32(bad_head + wave * 4, 0u);
        if (bad_table) lds_store_u32(bad_head + wave * 4, 1u);
    }

    const int tile_c = wave & 1, tile_r = (wave >> 1) & 1;
    const uint32_t row_stride = static_cast<uint32_t>(a.row_stride);
    const int out_tile = wave & 3, out_half = wave >> 2;  // 16 queries, 32 of a stage's rows
    bool again = false;

    for (int u = group; u < total_units; u += groups) {
        const Unit unit(f.list.units[u]);
        const int cols = unit.cols, n_w = unit.n_w;
        const bool small = unit.small;
        if (cols <= 0) continue;
        const int reach = kThreads / cols;                // rows of threads: a thread takes every `reach`-th key
        const int own = tid % cols, first = tid / cols;
        const bool active = first < reach;
        f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
        float run_max = -INFINITY, run_sum = 0.0f;
        for (int block = 0; block < unit.blocks(); ++block) {
            const int keys_n = unit.keys(block);
            if (keys_n <= 0) break;
            lds_barrier();
            if (tid < 4 && (tid >= 2 || block == 0)) {
                uint32_t all = 0;
                if (tid < 2) {
#pragma unroll
                    for (int w = 0; w < kWaves; ++w) all |= lds_load_u32(bad_head + w * 4);
                }
                lds_store_u32(marked + tid * 4, all ? 0xffffffffu : 0u);
            }
            // the tile's voxels: threads 0..63 the queries, 64..127 the keys
            if (tid < 2 * kCols) {
                const bool is_key = tid >= kCols;
                const int c = tid & (kCols - 1);
                const int cc = min(c, (is_key ? keys_n : cols) - 1);
                const int pos = unit.entry_of(f.list, cc).x + unit.inside(is_key ? block : unit.tile, cc);
                const int row = a.n2n ? a.n2n[pos] : pos;
                lds_store_u32((is_key ? row_j : row_i) + c * 4, row);
#pragma unroll
                for (int n = 0; n < ND; ++n) {
                    const float x = a.n_coords[static_cast<int64_t>(pos) * ND + n];
                    lds_store(is_key ? keys + (c * kKeyStride + n) * 4 : coords + (n * kCols + c) * 4, x);
                }
                if (!is_key) {
                    lds_store_u32(col_max + c * 4, 0x80000000u);
                    lds_store2(col_sum + c * 8, 0.0f, 0.0f);
                }
            }
            lds_barrier();
            // (re-read per tile, so that what follows from the lane number does not sit in registers for the whole launch)
            const int lane = opaque(tid & 63);
            const int m32 = lane & 31, half32 = lane >> 5;       // row or column, and group of terms, of a 32x32 operand
            const int n16 = lane & 15, group16 = lane >> 4;
            // operands that stay for all stages: queries (wavefronts 0..3) or keys
            Operand<T> feat;
            {
                const int row = static_cast<int>(lds_load_u32((wave < 4 ? row_i : row_j) + (tile_c * 32 + m32) * 4));
                feat.load((wave < 4 ? gq : gk) + static_cast<uint64_t>(static_cast<uint32_t>(row)) * row_stride + h * D + half32 * 8);
            }
            if (wave < 4) {
                // q . k of the tile, [key][query]
                Operand<T> kf;
                const int row = static_cast<int>(lds_load_u32(row_j + (tile_r * 32 + m32) * 4));
                kf.load(gk + static_cast<uint64_t>(static_cast<uint32_t>(row)) * row_stride + h * D + half32 * 8);
                const f32x16 d = mfma32(kf, feat, f32x16{});
                const uint32_t to = sums + ((tile_r * 32 + 4 * half32) * kStride + tile_c * 32 + m32) * 4;
#pragma unroll
                for (int e = 0; e < 16; ++e) lds_store(to + mfma32_row(0, e) * kStride * 4, d[e]);
            } else if (wave - 4 < D / 8) {
                // values of the tile with the channels as rows; keys past the tile are zero
                const int c8 = wave - 4;
                float v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = 0.0f;
                if (lane < keys_n)
                    load_row<8>(gv + static_cast<uint64_t>(lds_load_u32(row_j + lane * 4)) * row_stride + h * D + c8 * 8, v);
                T *to = reinterpret_cast<T *>(reinterpret_cast<char *>(smem) + (value_t - base)) + c8 * 8 * kStride +
                        (lane & 32) + permuted_row(lane & 31);
                bool bad = false;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    bad = bad || !finite(v[e]);
                    to[e * kStride] = static_cast<T>(finite(v[e]) ? v[e] : 0.0f);
                }
                if (bad) lds_or(bad_keys + (lane >> 5) * 4, 1u << (lane & 31));
            }
            lds_barrier();
            // this thread's pairs: query `own`, keys key0 + first + s * reach
            const int key0 = small ? own / n_w * n_w : 0;
            const int per_query = small ? n_w : keys_n;
            const int steps = (per_query + reach - 1) / reach;
            float logit[kSteps];
            uint32_t key_at[kSteps], packed[ND][2];
#pragma unroll
            for (int s = 0; s < kSteps; ++s) {
                const int j = key0 + min(first + s * reach, per_query - 1);
                key_at[s] = opaque(keys + j * (kKeyStride * 4));
                logit[s] = lds_load(sums + (j * kStride + own) * 4);
            }
#pragma unroll
            for (int n = 0; n < ND; ++n) packed[n][0] = packed[n][1] = 0;
            // The stages: products of the queries and keys with all rows of the stage's axes, then every pair's own two.
            // The table rows of the next stage are on their way while the pairs of this one are worked on.
            auto stage_needed = [&](int st) {
                return (st < 3 ? tile_r * 32 < rows_n(S::first(st)) : (tile_r == 0 || S::paired(st))) &&
                       tile_c * 32 < (wave < 4 ? cols : keys_n);
            };
            auto stage_rows = [&](int st) {
                const int one = S::first(st), other = one + (S::paired(st) ? 1 : 0);
                const bool second = st >= 3 && tile_r == 1;
                const int r = min((st < 3 ? tile_r * 32 : 0) + m32, (second ? rows_n(other) : rows_n(one)) - 1);
                return table_qk + (__umul24((second ? first_row(other) : first_row(one)) + r, HD) + h * D + half32 * 8);
            };
            typename Operand<T>::Raw raw{};
            if (stage_needed(0)) raw = Operand<T>::fetch(stage_rows(0));
#pragma unroll
            for (int st = 0; st < S::kCount; ++st) {
                lds_barrier();
                if (stage_needed(st)) {
                    Operand<T> rows;
                    rows.set(raw);
                    // [row][query] for the queries, [key][row] for the keys (16-byte stores of four consecutive words a
                    // lane, which the transposed product would give, met in more banks: +2 %)
                    if (wave < 4) {
                        const f32x16 d = mfma32(rows, feat, f32x16{});
                        const uint32_t to = sums + ((tile_r * 32 + 4 * half32) * kStride + tile_c * 32 + m32) * 4;
#pragma unroll
                        for (int e = 0; e < 16; ++e) lds_store(to + mfma32_row(0, e) * kStride * 4, d[e]);
                    } else {
                        const f32x16 d = mfma32(feat, rows, f32x16{});
                        const uint32_t to = keys + ((tile_c * 32 + 4 * half32) * kKeyStride + kCoordWords + tile_r * 32 + m32) * 4;
#pragma unroll
                        for (int e = 0; e < 16; ++e) lds_store(to + mfma32_row(0, e) * kKeyStride * 4, d[e]);
                    }
                }
                if (st + 1 < S::kCount && stage_needed(st + 1)) raw = Operand<T>::fetch(stage_rows(st + 1));
                lds_barrier();
#pragma unroll
                for (int b = 0; b < (S::paired(st) ? 2 : 1); ++b) {
                    const int axis = S::first(st) + b;
                    const float half_rows = static_cast<float>(rows_n(axis) / 2), upper = crse_upper(rows_n(axis));
                    const float ci = lds_load(coords + (axis * kCols + own) * 4);
                    const uint32_t own_at = sums + own * 4 + b * 32 * kStride * 4;
                    for_steps(steps, [&](int s) {
                        const float cj = lds_load(key_at[s] + axis * 4);
                        const uint32_t r = static_cast<uint32_t>(crse_row(ci, cj, half_rows, upper));
                        packed[axis][s / 4] |= r << (8 * (s % 4));
                        logit[s] += lds_load(__umul24(r, kStride * 4) + own_at) + lds_load(r * 4 + key_at[s] + (kCoordWords + b * 32) * 4);
                    });
                    // summed and packed now: the compiler would keep every gathered value until its sum is used
#pragma unroll
                    for (int s = 0; s < kSteps; ++s) asm volatile("" : "+v"(logit[s]));
                    packed[axis][0] = opaque(packed[axis][0]);
                    packed[axis][1] = opaque(packed[axis][1]);
                }
            }
            {
                bool bad = false;
#pragma unroll
                for (int s = 0; s < kSteps; ++s) bad = bad || !finite(logit[s]);
                // the values of the query's keys: bits key0 .. key0 + per_query - 1
                const uint64_t of_tile = static_cast<uint64_t>(lds_load_u32(bad_keys + 4)) << 32 | lds_load_u32(bad_keys);
                bad = bad || (of_tile >> key0) << (kCols - per_query) != 0;
                if (bad) lds_or(marked + (own >> 5) * 4, 1u << (own & 31));
            }
            // softmax of the tile: maxima per query, weights and their sum.  Only the last step of a thread can lie
            // past the window's keys.
            const int my_steps = active ? (per_query - first + reach - 1) / reach : 0;
            {
                float top = -INFINITY;
#pragma unroll
                for (int s = 0; s < kSteps; ++s) top = s < my_steps ? fmaxf(top, logit[s]) : top;
                if (active) lds_max(col_max + own * 4, float_order(top));
            }
            lds_barrier();
            lds_zero<kCols * kStride>(sums, tid);
            const float top = order_float(static_cast<int>(lds_load_u32(col_max + own * 4)));
            float p[kSteps], sum = 0.0f;
#pragma unroll
            for (int s = 0; s < kSteps; ++s) {
                p[s] = s < my_steps ? __expf(logit[s] - top) : 0.0f;
                sum += p[s];
            }
            if (active) {
                const float fixed = sum * kSumFix, whole = floorf(fixed);
                lds_add64(col_sum + own * 8, static_cast<uint32_t>((fixed - whole) / kSumLow), static_cast<int>(whole));
            }
            lds_barrier();
            uint32_t weight[kSteps];
            {
                const float scale = power2(kCellBits - exponent_of(sum_of(own)));
#pragma unroll
                for (int s = 0; s < kSteps; ++s) {
                    weight[s] = static_cast<uint32_t>(rintf(p[s] * scale));
                    if (s < my_steps) lds_store(sums + ((key0 + first + s * reach) * kStride + own) * 4, p[s]);
                }
            }
            f32x4_t tile_acc = {0.0f, 0.0f, 0.0f, 0.0f};
            const uint32_t cell_at = ((out_half * 32 + 2 * group16) * kStride + out_tile * 16 + n16) * 4;
            const float l_tile = sum_of(out_tile * 16 + n16);
            const int exponent = exponent_of(l_tile);
            auto read_out = [&](uint32_t cells, uint32_t operand, bool table) {
                if (out_tile * 16 >= cols) return;
                float v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const uint32_t at = cells + cell_at + ((e & 1) + 8 * (e >> 1)) * kStride * 4;
                    v[e] = table ? static_cast<float>(lds_load_u32(at)) : lds_load(at);
                }
                Cells<T> b;
                b.template set<false>(v, table ? kCellScale : power2(-exponent));      // (to the nearest: 3 % of a call, no smaller error)
                Operand<T> t;
                t.load_lds(operand + (n16 * kStride + out_half * 32 + group16 * 8) * sizeof(T));
                tile_acc = mfma16(t, b, tile_acc);
            };
            lds_barrier();
            read_out(sums, value_t, false);
            lds_zero<kCols * kStride>(keys, tid);
            lds_barrier();
#pragma unroll
            for (int st = 0; st < S::kCount; ++st) {
                const uint32_t cells = st % 2 == 0 ? keys : sums, next = st % 2 == 0 ? sums : keys;
#pragma unroll
                for (int b = 0; b < (S::paired(st) ? 2 : 1); ++b) {
                    const int axis = S::first(st) + b;
                    const uint32_t own_at = cells + own * 4 + b * 32 * kStride * 4;
                    for_steps(steps, [&](int s) {
                        lds_add(__umul24((packed[axis][s / 4] >> (8 * (s % 4))) & 0xffu, kStride * 4) + own_at, weight[s]);
                    });
                }
                lds_barrier();
                if (st < 3 ? out_half * 32 < rows_n(S::first(st)) : (out_half == 0 || S::paired(st)))
                    read_out(cells, table_t + st * D * kStride * sizeof(T), true);
                if (st + 1 < S::kCount) {
                    lds_zero<kCols * kStride>(next, tid);
                    lds_barrier();
                }
            }
            // into the query's running softmax state
            const int i = out_tile * 16 + n16;
            const float m_tile = order_float(static_cast<int>(lds_load_u32(col_max + i * 4)));
            const float m_all = fmaxf(run_max, m_tile);
            const float w_run = __expf(run_max - m_all), w_tile = __expf(m_tile - m_all), w_acc = w_tile * power2(exponent);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] = acc[e] * w_run + tile_acc[e] * w_acc;
            run_sum = run_sum * w_run + l_tile * w_tile;
            run_max = m_all;
        }
        // the two halves of the rows meet, and the result is stored
        const int n16 = tid & 15, group16 = (tid & 63) >> 4;
        lds_barrier();
        const uint32_t meet = sums + (out_tile * 16 + n16) * 80 + group16 * 16;
        if (out_half == 1) *(__attribute__((address_space(3))) f32x4_t *)(meet) = acc;
        lds_barrier();
        const int i = out_tile * 16 + n16;
        again = again || (lds_load_u32(marked + 4) | lds_load_u32(marked)) != 0;
        if (out_half == 0 && i < cols) {
            const bool mark = (lds_load_u32(marked + (i >> 5) * 4) >> (i & 31) & 1) != 0;
            const f32x4_t other = *(__attribute__((address_space(3))) f32x4_t *)(meet);
            const float inv = 1.0f / run_sum;
            const int64_t row = static_cast<int>(lds_load_u32(row_i + i * 4));
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = mark ? __int_as_float(0x7fc00000) : (acc[e] + other[e]) * inv;
            store4(static_cast<T *>(a.out) + row * HD + h * D + group16 * 4, o);
        }
    }
    if (!again) return;
    __syncthreads();      // the workgroup's stores
    for (int u = group; u < total_units; u += groups) {
        const Unit unit(f.list.units[u]);
        const int i = tid >> 3;
        if (i >= unit.cols) continue;
        const int first = unit.entry_of(f.list, i).x, pos = first + unit.inside(unit.tile, i);
        const int64_t row = a.n2n ? a.n2n[pos] : pos;
        const float out = to_float(static_cast<const volatile T *>(a.out)[row * HD + h * D]);
        if (out == out) continue;
        float ci[ND];
#pragma unroll
        for (int n = 0; n < ND; ++n) ci[n] = a.n_coords[static_cast<int64_t>(pos) * ND + n];
        exact_query<T, ND>(a, h, row, first, unit.n_w, tid & 7, ci, rows_n, first_row);
    }
}

template <int ND, bool kDeviceSizes>
int launch_fwd(const AttnArgs &a, const UnitList &list, hipStream_t stream)
{
    using L = FwdLayout<ND>;
    FwdArgs f;
    f.a = a;
    f.list = list;
    constexpr uint32_t lds = L::kBytes;
    auto kernel = attn_fwd_tile_kernel<ND, kDeviceSizes>;
    if (int rc = allow_dynamic_lds(reinterpret_cast<const void *>(kernel), lds)) return rc;
    const int per_cu = lds <= 80 * 1024 ? 2 : 1;
    const int slots = per_cu * device_cus();
    const int grid = slots >= a.H ? slots / a.H * a.H : a.H;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(kThreads), lds, stream, f);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

}  // namespace

int launch_list(const UnitList &l, const int32_t *w_sizes, const int32_t *w2n, int64_t W, hipStream_t stream)
{
    hipLaunchKernelGGL(tile_list_kernel, dim3(1), dim3(kListThreads), 0, stream, w_sizes, w2n, static_cast<int>(W),
                       const_cast<int32_t *>(l.total), const_cast<int4 *>(l.units), const_cast<int2 *>(l.entries));
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

}  // namespace tile

// Where the tile kernel serves a forward (fp32, head_dim 16).  It leaves every tile's products, sums and histograms in LDS and
// crosses some thirty barriers for them, which costs about what 64 x 64 pairs cost, so it needs windows of some size.  But a
// window is spread over its queries' tiles and a tile's pairs over 512 threads, where the sweep gives a query at most eight
// lanes: a launch that does not fill the chip ends when its longest unit ends, and that is a quarter as long.  Measured on
// windows of 55 to 110 voxels and 6 to 40 heads, tile over sweep kernel, by N^2 / W * H (what the sweep makes of a small
// launch jumps with its cut into units, which is most of the spread):
//   9 axes: 0.67 at 2 M, 0.94 to 1.05 at 4 to 12 M, 0.99 in the mean, 0.91 to 1.09 beyond, 1.01 in the mean
//   6 axes: 0.67 at 2 M, 0.83 to 0.94 at 4 to 26 M, 0.93 and 0.97 at 35 and 29 M
constexpr int kTileMeanWindow = 40;
constexpr double kTilePairsFloat = 35e6, kTilePairsFloatNormals = 12e6;

bool attn_tile_shape(int64_t N, int64_t W, int H, int nd)
{
    const double most = nd < 9 ? kTilePairsFloat : kTilePairsFloatNormals;
    return W > 0 && N >= kTileMeanWindow * W && static_cast<double>(N) * N / W * H <= most;
}

size_t attn_tile_list_bytes(int H, int64_t N, int64_t W)
{
    return attn_tile_shape(N, W, H, 3) ? tile::list_bytes(N, W) : 0;      // (whatever type and axes the call has)
}

bool attn_tile_applies(const AttnArgs &a, int dtype)
{
    if (dtype != S3D_DTYPE_F32 || a.D != tile::D || !attn_tile_shape(a.N, a.W, a.H, a.nd)) return false;
    return a.sizes_dev || rows_fit_tiles(a.rows, a.nd);
}

int launch_attn_tile(const AttnArgs &a, void *list, hipStream_t stream, int what)
{
    const tile::UnitList l = tile::list_at(list, a.N, a.W);
    if (what & kAttnBuildList) {
        if (int rc = tile::launch_list(l, a.w_sizes, a.w2n, a.W, stream)) return rc;
    }
    if (!(what & kAttnSweep)) return S3D_OK;
#define S3D_CASE(NN) \
    if (a.nd == NN) return a.sizes_dev ? tile::launch_fwd<NN, true>(a, l, stream) : tile::launch_fwd<NN, false>(a, l, stream);
    S3D_CASE(3) S3D_CASE(6) S3D_CASE(9)
#undef S3D_CASE
    return fail(S3D_ERR_UNSUPPORTED, "s3d_attn_fwd: %d axes in the tile form", a.nd);
}

}  // namespace s3d
