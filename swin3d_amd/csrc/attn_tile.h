// Pieces shared by the tile kernels of the attention forward and backward (gfx950): the unit list, matrix operands in
// fp16 or split fp32, LDS cells.
#pragma once

#include "attn_kernels.h"
#include "attn_strip_list.h"
#include "sweep_common.h"

namespace s3d {
namespace tile {

using namespace sweep;

constexpr int D = 16;                    // channels of a head
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
    const int32_t *total;      // [0]: units, [1]: strips
    const int4 *units;         // (first entry, voxels per window, windows, 0) or (entry, voxels, tile, tiles)
    const int2 *entries;       // windows by size: first sorted position, pairs (n^2) of the windows before it
    const int4 *strips;        // or null; (entry, voxels per window, first column, columns), see Strip
};
// A strip is up to 16 voxels of windows of one size: the voxels of its windows (of at most 64 voxels) in the order of the
// entries, from column `first` of window `entry` on; of a larger window, 16 of its voxels.
// A unit, decoded: the tile's queries are `cols` voxels; with more than one tile the workgroup goes through the tiles
// of the window's keys.
struct Unit {
    int entry, n_w, tile, tiles, size, cols;
    bool small;
    __device__ __forceinline__ Unit(const int4 u)
    {
        entry = __builtin_amdgcn_readfirstlane(u.x);
        n_w = __builtin_amdgcn_readfirstlane(u.y);
        const int z = __builtin_amdgcn_readfirstlane(u.z);
        tiles = __builtin_amdgcn_readfirstlane(u.w);
        small = tiles == 0;
        size = small ? n_w : (n_w + tiles - 1) / tiles;
        tile = small ? 0 : z;
        cols = small ? z * n_w : min(size, n_w - z * size);
    }
    __device__ __forceinline__ int blocks() const { return small ? 1 : tiles; }
    // keys of block b, and the entry, position inside the window and sorted position of column c of tile t
    __device__ __forceinline__ int keys(int b) const { return small ? cols : min(size, n_w - b * size); }
    __device__ __forceinline__ int2 entry_of(const UnitList &l, int c) const { return l.entries[small ? entry + c / n_w : entry]; }
    __device__ __forceinline__ int inside(int t, int c) const { return small ? c % n_w : t * size + c; }
};
inline size_t list_round(size_t bytes) { return (bytes + 255) / 256 * 256; }
// a unit covers at least 32 voxels (a tile of a window of 65), but for the last one of each window size up to 32
inline size_t list_max_units(int64_t N) { return static_cast<size_t>(N > 0 ? N : 0) / 32 + kCols + 1; }
inline size_t list_bytes(int64_t N, int64_t W)
{
    return 256 + list_round(sizeof(int4) * list_max_units(N)) + list_round(sizeof(int2) * static_cast<size_t>(W > 0 ? W : 1));
}
// a strip is full, but for the last one of each window size up to 64 and of each larger window
inline size_t list_max_strips(int64_t N) { return static_cast<size_t>(N > 0 ? N : 0) / kStrip + static_cast<size_t>(N > 0 ? N : 0) / (kCols + 1) + kCols + 1; }
inline size_t strips_bytes(int64_t N) { return list_round(sizeof(int4) * list_max_strips(N)); }
// a strip's voxels: see StripArgs
inline size_t strip_columns_bytes(int64_t N) { return align_up(kStrip * list_max_strips(N) * (sizeof(int4) + sizeof(int32_t)), 256); }
inline UnitList list_at(void *p, int64_t N, int64_t W)
{
    char *base = static_cast<char *>(p);
    UnitList l;
    l.total = reinterpret_cast<const int32_t *>(base);
    l.units = reinterpret_cast<const int4 *>(base + 256);
    l.entries = reinterpret_cast<const int2 *>(base + 256 + list_round(sizeof(int4) * list_max_units(N)));
    l.strips = nullptr;
    return l;
}
int launch_list(const UnitList &l, const int32_t *w_sizes, const int32_t *w2n, int64_t W, hipStream_t stream);

constexpr int kListThreads = 1024;
constexpr int kBigBins = 31, kListBins = kBigBins + kCols;   // windows of 2 .. 32 and more tiles, then 64 .. 1 voxels

__device__ __forceinline__ int tiles_of(int n) { return (n + kCols - 1) / kCols; }
__device__ __forceinline__ int list_bin(int n) { return n > kCols ? 32 - min(tiles_of(n), 32) : kBigBins + kCols - n; }

// Barrier of the workgroup for what it shares in LDS.  __syncthreads() also waits for every load from memory that is under
// way, among them what a stage has asked for ahead of its use, and for every store.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Unit list: windows in bins of equal size, largest first (a counting sort in LDS), and the pairs of the windows before
// each.  Inside a bin the windows keep their order: where a window lies in its unit decides in which order the matrix pipe
// adds its products, and a result is to be the same bits on every call.
__device__ __forceinline__ void build_list(const int32_t *__restrict__ w_sizes, const int32_t *__restrict__ w2n, int W,
                                           int32_t *__restrict__ total, int4 *__restrict__ units, int2 *__restrict__ entries,
                                           int4 *__restrict__ strips)
{
    __shared__ int windows[kListBins], big_units[kListBins], entry_at[kListBins], unit_at[kListBins], entry_first[kListBins];
    constexpr int kWavesOfList = kListThreads / 64;
    __shared__ long long wave_pairs[kWavesOfList];
    __shared__ int of_wave[kWavesOfList][kListBins];
    __shared__ unsigned long long same_of_wave[kWavesOfList][kListBins];
    __shared__ int big_strips[kListBins], strip_at[kListBins], strips_of_wave[kWavesOfList][kBigBins];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    if (t < kListBins) windows[t] = big_units[t] = big_strips[t] = 0;
    __syncthreads();
    // (loads ahead of their use, here and below: the rounds are a chain of trips to memory otherwise)
    constexpr int kAhead = 8;
    for (int w0 = t; w0 < W; w0 += kAhead * kListThreads) {
        int size[kAhead];
#pragma unroll
        for (int k = 0; k < kAhead; ++k) size[k] = w_sizes[min(w0 + k * kListThreads, W - 1)];
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
            const int n = w0 + k * kListThreads < W ? size[k] : 0;
            if (n <= 0) continue;
            const int b = list_bin(n);
            atomicAdd(&windows[b], 1);
            if (n > kCols) {
                atomicAdd(&big_units[b], tiles_of(n));
                atomicAdd(&big_strips[b], strips_of(n));
            }
        }
    }
    __syncthreads();
    if (wave == 0) {
        // exclusive sums of windows, units and strips over the bins, 64 at a time
        int e_run = 0, u_run = 0, s_run = 0;
        for (int b0 = 0; b0 < kListBins; b0 += 64) {
            const int b = b0 + lane;
            const int count = b < kListBins ? windows[b] : 0;
            const int per = b < kBigBins ? 1 : kCols / max(1, kCols - (b - kBigBins));
            const int mine = b >= kListBins ? 0 : b < kBigBins ? big_units[b] : (count + per - 1) / per;
            const int own_strips = b >= kListBins ? 0 : b < kBigBins ? big_strips[b] : strips_of(count * (kCols - (b - kBigBins)));
            int e = count, u = mine, s = own_strips;
            for (int off = 1; off < 64; off <<= 1) {
                const int ue = __shfl_up(e, off), uu = __shfl_up(u, off), us = __shfl_up(s, off);
                if (lane >= off) { e += ue; u += uu; s += us; }
            }
            if (b < kListBins) {
                strip_at[b] = s_run + s - own_strips;
                entry_at[b] = entry_first[b] = e_run + e - count;
                unit_at[b] = u_run + u - mine;
            }
            e_run += __shfl(e, 63);
            u_run += __shfl(u, 63);
            s_run += __shfl(s, 63);
        }
        if (lane == 0) {
            total[0] = u_run;
            if (strips) total[1] = s_run;
        }
    }
    __syncthreads();
    long long before = 0;              // pairs of the windows that earlier rounds placed
    int next_n = t < W ? w_sizes[t] : 0, next_pos = t < W ? w2n[t] : 0;
    for (int w0 = 0; w0 < W; w0 += kListThreads) {
        const int n = next_n, pos = next_pos;
        const int ahead = w0 + kListThreads + t;
        next_n = ahead < W ? w_sizes[ahead] : 0;
        next_pos = ahead < W ? w2n[ahead] : 0;
        long long incl = n > 0 ? static_cast<long long>(n) * n : 0;
        const long long own = incl;
        for (int off = 1; off < 64; off <<= 1) {
            const long long up = __shfl_up(incl, off);
            if (lane >= off) incl += up;
        }
        if (lane == 63) wave_pairs[wave] = incl;
        for (int i = t; i < kWavesOfList * kListBins; i += kListThreads) {
            of_wave[0][i] = 0;
            same_of_wave[0][i] = 0;
        }
        if (t < kWavesOfList * kBigBins) strips_of_wave[0][t] = 0;
        lds_barrier();
        // A window's place among those of its bin: in its wavefront, by the lanes with windows of the bin, then behind the
        // wavefronts before.  (A bit for each lane, set in LDS: a vote for every size that a wavefront has took 38 us for 7,600
        // windows of some thirty sizes, so 30, and 9.5 for 220 windows, so 8.)
        const int b = n > 0 ? list_bin(n) : -1;
        // (of a bin of larger windows, also the strips of the windows before: all but up to three fewer than four a tile)
        const int fewer = n > kCols ? 4 * tiles_of(n) - strips_of(n) : 0;
        const unsigned long long one = __ballot((fewer & 1) != 0), two = __ballot((fewer & 2) != 0);
        if (b >= 0) atomicOr(&same_of_wave[wave][b], 1ull << lane);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        int rank = 0, strips_before = 0;
        if (b >= 0) {
            const unsigned long long same = same_of_wave[wave][b], below = same & ((1ull << lane) - 1);
            rank = __popcll(below);
            const int most = 4 * (32 - b);             // (not in bin 0, whose windows differ in their tiles)
            if (b < kBigBins) strips_before = most * rank - __popcll(below & one) - 2 * __popcll(below & two);
            if (rank == 0) {
                of_wave[wave][b] = __popcll(same);
                if (b < kBigBins) strips_of_wave[wave][b] = most * __popcll(same) - __popcll(same & one) - 2 * __popcll(same & two);
            }
        }
        long long pairs = before + incl - own, all = 0;
#pragma unroll
        for (int v = 0; v < kWavesOfList; ++v) {
            pairs += v < wave ? wave_pairs[v] : 0;
            all += wave_pairs[v];
        }
        before += all;
        lds_barrier();
        if (t < kListBins) {
            int count[kWavesOfList], run = entry_at[t];
#pragma unroll
            for (int v = 0; v < kWavesOfList; ++v) count[v] = of_wave[v][t];
#pragma unroll
            for (int v = 0; v < kWavesOfList; ++v) {
                of_wave[v][t] = run;
                run += count[v];
            }
            entry_at[t] = run;
        } else if (t >= 128 && t < 128 + kBigBins) {
            const int bin = t - 128;
            int run = strip_at[bin];
#pragma unroll
            for (int v = 0; v < kWavesOfList; ++v) {
                const int own_count = strips_of_wave[v][bin];
                strips_of_wave[v][bin] = run;
                run += own_count;
            }
            if (bin > 0) strip_at[bin] = run;
        }
        lds_barrier();
        if (b >= 0) {
            const int e = of_wave[wave][b] + rank, in_bin = e - entry_first[b];
            // (a window that begins beyond 2^31 pairs does not fit any store of this form)
            entries[e] = make_int2(pos, static_cast<int>(pairs < 0x7fffffffll ? pairs : 0x7fffffffll));
            if (n > kCols) {
                const int tiles = tiles_of(n);
                // (the windows of the first bin differ in their tiles)
                const int u = b > 0 ? unit_at[b] + in_bin * tiles : atomicAdd(&unit_at[b], tiles);
                if (units)
                    for (int q = 0; q < tiles; ++q) units[u + q] = make_int4(e, n, q, tiles);
                if (strips) {
                    const int count = strips_of(n), first = b > 0 ? strips_of_wave[wave][b] + strips_before : atomicAdd(&strip_at[b], count);
                    for (int q = 0; q < count; ++q) strips[first + q] = make_int4(e, n, q * kStrip, min(kStrip, n - q * kStrip));
                }
            } else {
                const int per = kCols / n;
                if (units && in_bin % per == 0) units[unit_at[b] + in_bin / per] = make_int4(e, n, min(per, windows[b] - in_bin), 0);
                if (strips) {
                    // the strips whose first column is this window's
                    const int begin = in_bin * n, end = begin + n, columns = windows[b] * n;
                    for (int q = strips_of(begin); q * kStrip < end; ++q)
                        strips[strip_at[b] + q] = make_int4(e, n, q * kStrip - begin, min(kStrip, columns - q * kStrip));
                }
            }
        }
        lds_barrier();
    }
}

// ---- LDS --------------------------------------------------------------------------------------------------------------
typedef __attribute__((address_space(3))) float lds_f32;
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef __attribute__((address_space(3))) int lds_i32;
typedef __attribute__((address_space(3))) u32x4_t lds_u32x4;
__device__ __forceinline__ float lds_load(uint32_t addr) { return *(lds_f32 *)(addr); }
__device__ __forceinline__ uint32_t lds_load_u32(uint32_t addr) { return *(lds_u32 *)(addr); }
__device__ __forceinline__ void lds_store(uint32_t addr, float v) { *(lds_f32 *)(addr) = v; }
__device__ __forceinline__ void lds_store_u32(uint32_t addr, uint32_t v) { *(lds_u32 *)(addr) = v; }
__device__ __forceinline__ float2 lds_load2(uint32_t addr)
{
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    const f32x2 v = *(__attribute__((address_space(3))) f32x2 *)(addr);
    return make_float2(v[0], v[1]);
}
__device__ __forceinline__ void lds_store2(uint32_t addr, float a, float b)
{
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    *(__attribute__((address_space(3))) f32x2 *)(addr) = f32x2{a, b};
}
// cell += hi 2^32 + lo
__device__ __forceinline__ void lds_add64(uint32_t addr, uint32_t lo, int hi)
{
    typedef __attribute__((address_space(3))) uint64_t lds_u64;
    const uint64_t v = (static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32) | lo;
    __hip_atomic_fetch_add((lds_u64 *)(addr), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// four channels of a row
__device__ __forceinline__ void store4(float *p, const float *v) { *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]); }
__device__ __forceinline__ void store4(__half *p, const float *v)
{
    uint2 x;
    reinterpret_cast<__half2 *>(&x)[0] = __floats2half2_rn(v[0], v[1]);
    reinterpret_cast<__half2 *>(&x)[1] = __floats2half2_rn(v[2], v[3]);
    *reinterpret_cast<uint2 *>(p) = x;
}
__device__ __forceinline__ void lds_add(uint32_t addr, uint32_t v)
{
    __hip_atomic_fetch_add((lds_u32 *)(addr), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_or(uint32_t addr, uint32_t v)
{
    __hip_atomic_fetch_or((lds_u32 *)(addr), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_max(uint32_t addr, int v)
{
    __hip_atomic_fetch_max((lds_i32 *)(addr), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ bool finite(float x) { return fabsf(x) < INFINITY; }
// exponent e with |x| < 2^e, and 2^e
__device__ __forceinline__ int exponent_of(float x)
{
    return x != 0.0f ? max(-100, static_cast<int>((__float_as_uint(x) >> 23) & 0xff) - 126) : -100;
}
__device__ __forceinline__ float power2(int e) { return ldexpf(1.0f, e); }
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
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Eight values of an operand.  fp16 as they are; fp32 as a sum of three bf16 numbers, which hold its 24 bits exactly: of the
// nine partial products the six largest are taken, at a third of the time of fp32 matrix instructions.  What is left out of
// a product is 2^-25 of it, half of what fp32 arithmetic rounds to, and of either sign as long as one of its operands is
// split into the nearest numbers (split); the other may be cut off (cut, cheaper by a sixth), but with both cut off what is
// left out has the product's sign, and the backward's errors against 64 bits are a third larger.
template <typename T> struct Operand;
template <> struct Operand<__half> {
    f16x8 x;
    __device__ __forceinline__ void load(const __half *p) { x = __builtin_bit_cast(f16x8, *reinterpret_cast<const uint4 *>(p)); }
    __device__ __forceinline__ void set_values(const __half *v)
    {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = __builtin_bit_cast(_Float16, v[e]);
    }
};
template <> struct Operand<float> {
    bf16x8 s[3];
    struct Raw { float4 v[2]; };         // as loaded, before any conversion
    static __device__ __forceinline__ Raw fetch(const float *p)
    {
        return {{reinterpret_cast<const float4 *>(p)[0], reinterpret_cast<const float4 *>(p)[1]}};
    }
    __device__ __forceinline__ void set(const Raw &r)
    {
        const float v[8] = {r.v[0].x, r.v[0].y, r.v[0].z, r.v[0].w, r.v[1].x, r.v[1].y, r.v[1].z, r.v[1].w};
        cut(v);
    }
    __device__ __forceinline__ void split(const float *v)
    {
        u32x4 out[3];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            f32x2 x = {v[2 * e], v[2 * e + 1]};
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                out[k][e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(x, bf16x2));
                if (k < 2) x -= f32x2{__uint_as_float(out[k][e] << 16), __uint_as_float(out[k][e] & 0xffff0000u)};
            }
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) s[k] = __builtin_bit_cast(bf16x8, out[k]);
    }
    __device__ __forceinline__ void cut(const float *v)
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
    __device__ __forceinline__ void set_values(const float *v) { split(v); }
    template <typename TF> __device__ __forceinline__ void load(const TF *p)
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
        cut(v);
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
// is lane % 16, its rows 4 (lane / 16) + e.  B is a set of fp32 values: two fp16 numbers each beside fp16 (23 bits,
// where the caller's scale brings them to; A is exact), three bf16 numbers beside fp32.
template <typename T> struct Cells;
template <> struct Cells<__half> {
    f16x8 hi, lo;
    // v * scale as the sum of two fp16 numbers
    template <bool kNearest = true> __device__ __forceinline__ void set(const float *v, float scale)
    {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            hi[e] = static_cast<_Float16>(v[e] * scale);
            lo[e] = static_cast<_Float16>(__builtin_fmaf(v[e], scale, -static_cast<float>(hi[e])));
        }
    }
};
template <> struct Cells<float> {
    Operand<float> x;
    template <bool kNearest = true> __device__ __forceinline__ void set(const float *v, float scale)
    {
        float y[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = v[e] * scale;
        if constexpr (kNearest) x.split(y); else x.cut(y);
    }
};
// (the six partial products meet before they join the sum, which is then rounded once a product: the forward's error against
// 64 bits on 3000 voxels of near-uniform weights is 1.0e-7 so, 2.4e-7 one after the other, 1.9e-7 in the sweep)
__device__ __forceinline__ f32x4_t mfma16(const Operand<float> &a, const Cells<float> &b, f32x4_t c)
{
    f32x4_t p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.s[2], b.x.s[0], f32x4_t{}, 0, 0, 0);
    p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.s[1], b.x.s[1], p, 0, 0, 0);
    p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.s[0], b.x.s[2], p, 0, 0, 0);
    p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.s[1], b.x.s[0], p, 0, 0, 0);
    p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.s[0], b.x.s[1], p, 0, 0, 0);
    p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.s[0], b.x.s[0], p, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < 4; ++e) c[e] += p[e];
    return c;
}

// fp32 values beside fp16 ones: the sum of two fp16 numbers (23 bits) of the values times a power of two that brings the
// largest of them to 2^14
struct Pair16 {
    f16x8 hi, lo;
    __device__ __forceinline__ void set_values(const float *v, float scale)
    {
        Cells<__half> c;
        c.set(v, scale);
        hi = c.hi;
        lo = c.lo;
    }
};
__device__ __forceinline__ f32x16 mfma32(const Pair16 &a, const Operand<__half> &b, f32x16 c)
{
    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.lo, b.x, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a.hi, b.x, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma32(const Operand<__half> &a, const Pair16 &b, f32x16 c)
{
    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.x, b.lo, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a.x, b.hi, c, 0, 0, 0);
}

// ---- the forward's last resort: a query pair by pair, where something in its window is not finite
template <typename T, int ND, typename Rows, typename First>
__device__ __forceinline__ void exact_query(const AttnArgs &a, int h, int64_t row, int pos0, int n_w, int sub, const float *own, Rows rows_n, First first_row)
{
    // eight neighbouring lanes a query, which take every eighth key
    const int HD = a.H * D;
    const T *gq = static_cast<const T *>(a.q) + h * D, *gk = static_cast<const T *>(a.k) + h * D, *gv = static_cast<const T *>(a.v) + h * D;
    const T *table_q = static_cast<const T *>(a.table_q) + h * D, *table_k = static_cast<const T *>(a.table_k) + h * D;
    const T *table_v = static_cast<const T *>(a.table_v) + h * D;
    float q[D], acc[D], m = -INFINITY, l = 0.0f;
    load_row<D>(gq + row * a.row_stride, q);
#pragma unroll
    for (int c = 0; c < D; ++c) acc[c] = 0.0f;
    for (int j = sub; j < n_w; j += 8) {
        const int pos = pos0 + j;
        const int64_t key = a.n2n ? a.n2n[pos] : pos;
        float k[D], x[D], logit = 0.0f;
        int at[ND];
        load_row<D>(gk + key * a.row_stride, k);
#pragma unroll
        for (int c = 0; c < D; ++c) logit = fmaf(q[c], k[c], logit);
#pragma unroll
        for (int n = 0; n < ND; ++n) {
            const float cj = a.n_coords[static_cast<int64_t>(pos) * ND + n];
            at[n] = (first_row(n) + crse_row(own[n], cj, static_cast<float>(rows_n(n) / 2), crse_upper(rows_n(n)))) * HD;
            float part = 0.0f;
            load_row<D>(table_q + at[n], x);
#pragma unroll
            for (int c = 0; c < D; ++c) part = fmaf(q[c], x[c], part);
            load_row<D>(table_k + at[n], x);
#pragma unroll
            for (int c = 0; c < D; ++c) part = fmaf(k[c], x[c], part);
            logit += part;
        }
        const float top = fmaxf(m, logit);
        const float scale = m == -INFINITY ? 0.0f : __expf(m - top), p = logit == -INFINITY ? 0.0f : __expf(logit - top);
        m = top;
        l = fmaf(l, scale, p);
        load_row<D>(gv + key * a.row_stride, x);
#pragma unroll
        for (int c = 0; c < D; ++c) acc[c] = fmaf(p, x[c], acc[c] * scale);
#pragma unroll
        for (int n = 0; n < ND; ++n) {
            load_row<D>(table_v + at[n], x);
#pragma unroll
            for (int c = 0; c < D; ++c) acc[c] = fmaf(p, x[c], acc[c]);
        }
    }
#pragma unroll
    for (int other = 1; other < 8; other <<= 1) {
        const float m_o = __shfl_xor(m, other), l_o = __shfl_xor(l, other), top = fmaxf(m, m_o);
        const float w = m == -INFINITY ? 0.0f : __expf(m - top), w_o = m_o == -INFINITY ? 0.0f : __expf(m_o - top);
        l = l * w + l_o * w_o;
#pragma unroll
        for (int c = 0; c < D; ++c) acc[c] = acc[c] * w + __shfl_xor(acc[c], other) * w_o;
        m = top;
    }
    if (sub > 0) return;
    const float inv = 1.0f / l;
#pragma unroll
    for (int c = 0; c < D; ++c) acc[c] *= inv;
    store_row<D>(static_cast<T *>(a.out) + row * HD + h * D, acc);
}

}  // namespace tile
}  // namespace s3d
