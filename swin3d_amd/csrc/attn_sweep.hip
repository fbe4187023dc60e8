// Sparse-voxel windowed self-attention with cRSE tables (gfx950): the sweep kernel of the forward and, on the same
// work list, the pair sweeps of the backward (dq; dk and dv - further down).
//
// Covers every dtype / shape the library accepts on the vector ALU (fp32 arithmetic; fp16 inputs enter through
// packed dot products and mixed-precision FMAs with fp32 accumulation).  A workgroup serves one to three heads
// for its whole life and keeps the slices of the three relative-signal tables in LDS (loaded once, not once
// per window).  Lane = one query against (a share of) the keys of its window: q_i, the running
// maximum, sum and output stay in the lane's registers while the lane streams its own window's keys, one per
// step, no atomic on data and no O(pairs) index array; the result is
// deterministic.  The slots of all windows, sorted by step count, are packed into units of 64 (the lanes of a
// wavefront carry queries of several small windows); wavefronts draw units from the head's work queues.
// A query of a window of more than the step target gets 2, 4 or 8 adjacent lanes that take alternate keys and merge
// their softmax states by shuffles at the end of the unit.
//
// Math (per window, sorted positions i, j, head h), following the reference kernels
// Swin3D/src/attn/self_attn_aio_fwd.cu:16-52 and :111-188:
//   row_n(i,j) = quantised (n_coords[i][n] - n_coords[j][n])   (attn_utils.cuh:437-453)
//   T*(i,j)[c] = sum_n table_*[n][row_n(i,j)][h][c]            (attn_utils.cuh:455-464)
//   L(i,j)     = sum_c q_i[c] k_j[c] + q_i[c] Tq(i,j)[c] + k_j[c] Tk(i,j)[c]
//   out_i[c]   = sum_j softmax_j(L(i,j)) (v_j[c] + Tv(i,j)[c])
#include "attn_kernels.h"
#include "attn_strip.h"
#include "sweep_common.h"

#include <algorithm>
#include <mutex>
#include <vector>

namespace s3d {

// Raises a kernel's dynamic-LDS limit to `bytes`.  The runtime keeps the limit per function and device, so it is
// set when a (function, device) pair first needs that much and not again: a call under stream capture then issues
// kernel launches only (one eager call per shape and device has to come before the capture).
int allow_dynamic_lds(const void *kernel, size_t bytes)
{
    struct Granted { const void *kernel; int device; size_t bytes; };
    static std::mutex mutex;
    static std::vector<Granted> granted;
    int device = 0;
    S3D_HIP_CHECK(hipGetDevice(&device));
    std::lock_guard<std::mutex> lock(mutex);
    for (Granted &g : granted) {
        if (g.kernel == kernel && g.device == device) {
            if (g.bytes >= bytes) return S3D_OK;
            S3D_HIP_CHECK(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes)));
            g.bytes = bytes;
            return S3D_OK;
        }
    }
    S3D_HIP_CHECK(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes)));
    granted.push_back({kernel, device, bytes});
    return S3D_OK;
}

int device_cus()
{
    int device = 0, v = 0;
    if (hipGetDevice(&device) == hipSuccess &&
        hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && v > 0)
        return v;
    return 256;
}

namespace {

using namespace sweep;

constexpr int kChunk = 64;   // lanes of a wavefront = lanes of a unit
constexpr int kListThreads = 256, kListGroups = 32;   // the list builder's workgroups: size, and how many at most
constexpr float kSlack = 10.0f;   // how far a logit may exceed the softmax reference exponent before it moves
// A window of n voxels belongs to class g (0..kMaxSplit): each of its queries is served by 2^g adjacent lanes that
// take alternate keys, g the smallest value for which a lane streams at most `target` keys (the launch's step
// target: 64, or 32 / 16 in small launches that would otherwise not fill the chip).  Windows of more than
// target << kMaxSplit voxels stay in the last class and take more steps.
constexpr int kMaxSplit = 3;
constexpr int kClasses = kMaxSplit + 1;
constexpr int kMaxSteps = 64;                    // step counts that have a bin of their own; longer ones share the last
constexpr int kBins = kClasses * kMaxSteps;      // (class, steps), class 3 first, longest first inside a class
constexpr int kSections = kMaxSplit + 3;         // classes 3..1, then class 0 in units of 64, 32 and 16 queries
static_assert(kBins == kListThreads, "one thread per bin");
__host__ __device__ inline int window_class(int n, int target_shift)
{
    int g = 0;
    while (g < kMaxSplit && ((n + (1 << g) - 1) >> g) > (1 << target_shift)) ++g;
    return g;
}
__host__ __device__ inline int window_bin(int n, int g)
{
    const int steps = (n + (1 << g) - 1) >> g;
    return (kMaxSplit - g) * kMaxSteps + (kMaxSteps - (steps < kMaxSteps ? steps : kMaxSteps));
}
// The step target of a launch, as a shift.  The launch ends when its last wavefront does, so a unit must stay
// short against what a wavefront does in the whole launch: N^2 / W pairs at least, per head group, over the
// lanes of `waves` wavefronts that serve the group.  64 steps unless that leaves fewer than about six units per
// wavefront; not below 32 where the mean window has at most 32 voxels: a target of 16 would give the typical
// window two lanes per query, whose softmax states are merged at the end of the unit, where one lane per query
// serves it in 32 steps without a merge (-3.5 % on 26-voxel windows; on window-7 levels, 57 voxels a window and
// most pairs in windows of more than 64, the target of 32 measured +4 %: longer units, the same merges).
__host__ inline int target_shift_for(int64_t N, int64_t W, int waves)
{
    if (N <= 0 || W <= 0) return 6;
    const double lane_steps = static_cast<double>(N) * static_cast<double>(N) / static_cast<double>(W);
    const int least = N <= 32 * W ? 5 : 4;
    int shift = 6;
    while (shift > least && lane_steps / (64.0 * (1 << shift)) < 6.0 * (waves > 0 ? waves : 1)) --shift;
    return shift;
}

// byte offsets inside the workspace: the queue counters, the totals, one record per unit, the sorted window
// entries, the placement notes and per-workgroup bin totals of the list builder
__host__ __device__ inline size_t ws_round(size_t bytes) { return (bytes + 255) / 256 * 256; }
__host__ __device__ inline size_t ws_total_offset(int H) { return sizeof(int32_t) * static_cast<size_t>(H) * kQueues * kCounterStride; }
// after the totals (one cache line): one exit counter per queue index, each on a cache line of its own
__host__ __device__ inline size_t ws_units_offset(int H) { return ws_total_offset(H) + 256 * (1 + kQueues); }
// a unit holds at least 64 >> kMaxSplit = 8 queries, except the last one of each section
__host__ __device__ inline size_t ws_max_units(int64_t N)
{
    return static_cast<size_t>(N > 0 ? N : 0) / (kChunk >> kMaxSplit) + kSections + 1;
}
__host__ __device__ inline size_t ws_entries_offset(int H, int64_t N)
{
    return ws_units_offset(H) + ws_round(sizeof(int4) * ws_max_units(N));
}
__host__ __device__ inline size_t ws_place_offset(int H, int64_t W, int64_t N)
{
    return ws_entries_offset(H, N) + ws_round(sizeof(int4) * (static_cast<size_t>(W > 0 ? W : 0) + kChunk));
}
__host__ __device__ inline size_t ws_bins_offset(int H, int64_t W, int64_t N)
{
    return ws_place_offset(H, W, N) + ws_round(sizeof(int2) * static_cast<size_t>(W > 0 ? W : 1));
}
__host__ __device__ inline size_t ws_end_offset(int H, int64_t W, int64_t N)
{
    return ws_bins_offset(H, W, N) + ws_round(sizeof(unsigned long long) * kListGroups * (kListThreads / 64 + 1) * kBins);
}

// How the queries of class 0 (sorted by steps, longest first) are cut into units.  A unit is one pass of a
// wavefront: 64 queries, or 32 queries with two adjacent lanes each (alternate keys, half the steps), or 16
// queries with four lanes each (a quarter).  The launch ends when the last wavefront ends, so the last queries
// go into the finer units: about two 16-query units and one 32-query unit per wavefront of a head group
// (`waves`), everything before them into 64-query units.
struct UnitPlan {
    int units[3];   // units of 64, 32 and 16 queries, in this order along the queries
    __host__ __device__ int first_slot(int g) const { return g == 0 ? 0 : g == 1 ? units[0] * kChunk : units[0] * kChunk + units[1] * (kChunk / 2); }
    __host__ __device__ int first_unit(int g) const { return g == 0 ? 0 : g == 1 ? units[0] : units[0] + units[1]; }
};
__host__ __device__ inline UnitPlan plan_units(int total_slots, int waves)
{
    const int fine = 32 * (waves > 0 ? waves : 1);   // queries of each finer kind
    const int in_c = total_slots < fine ? total_slots : fine;
    const int in_b = total_slots - in_c < fine ? total_slots - in_c : fine;
    UnitPlan plan;
    plan.units[0] = (total_slots - in_c - in_b + kChunk - 1) / kChunk;
    const int left_b = total_slots - plan.units[0] * kChunk;            // may be negative by rounding
    const int take_b = left_b < 0 ? 0 : (left_b < in_b ? left_b : in_b);
    plan.units[1] = (take_b + kChunk / 2 - 1) / (kChunk / 2);
    const int left_c = total_slots - plan.units[0] * kChunk - plan.units[1] * (kChunk / 2);
    plan.units[2] = left_c <= 0 ? 0 : (left_c + kChunk / 4 - 1) / (kChunk / 4);
    return plan;
}

// Work list of the launch, built by two small kernels.  The windows are sorted by (class, steps), highest class and
// longest first - a counting sort over the kBins possible keys - and the queries of each class are numbered
// back to back in that order, [window][voxel], and cut into units: 64 >> g queries of class g, each on 2^g
// adjacent lanes.  A wavefront's lanes so carry queries of several windows when the windows are small, every
// lane of a unit runs (almost) the same number of steps, a query's keys never leave its wavefront (the lanes
// that share a query merge their softmax states by shuffles), and the launch ends on its shortest units.
//
// sweep_count_kernel: every wavefront takes a run of consecutive windows, 64 at a time.  A window's place in the
// bin of its (class, steps) - its rank there and the queries before it - follows the window numbers: the lanes
// of each bin present among the 64 are ranked by their lane numbers on top of the bin's running totals, which
// the wavefront keeps in registers (lane b % 64 holds bin b), and the wavefront leaves its bin totals.  No
// atomics: the list, and with it the cut of the queries into units and so every bit of the result, is the same
// on every run.
__device__ __forceinline__ void count_windows(const AttnArgs &a, int group, int groups)
{
    constexpr int kWaves = kListThreads / 64;
    const int lane = threadIdx.x & 63;
    const int table = group * kWaves + static_cast<int>(threadIdx.x >> 6);
    const int tables = groups * kWaves;
    char *ws = static_cast<char *>(a.workspace);
    int2 *place = reinterpret_cast<int2 *>(ws + ws_place_offset(a.H, a.W, a.N));
    unsigned long long *group_bins = reinterpret_cast<unsigned long long *>(ws + ws_bins_offset(a.H, a.W, a.N));
    const int W = static_cast<int>(a.W);
    const int per = (W + tables - 1) / tables;
    const int begin = min(table * per, W), end = min(begin + per, W);
    uint32_t held_c[kBins / 64], held_s[kBins / 64];   // bins lane, lane + 64, ...: windows and queries so far
#pragma unroll
    for (int j = 0; j < kBins / 64; ++j) held_c[j] = held_s[j] = 0;
    for (int w0 = begin; w0 < end; w0 += 64) {
        const int w = w0 + lane;
        const int n = w < end ? a.w_sizes[w] : 0;
        const int b = n > 0 ? window_bin(n, window_class(n, a.block_shift)) : -1;
        int2 got = make_int2(-1, 0);
        unsigned long long todo = __ballot(b >= 0);
        while (todo != 0) {
            const int leader = __ffsll(todo) - 1;
            const int cb = __builtin_amdgcn_readlane(b, leader), n_lead = __builtin_amdgcn_readlane(n, leader);
            const bool in = b == cb;
            const unsigned long long same = __ballot(in);
            const int below = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(same >> 32),
                                                        __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(same), 0u));
            int before_n, all_n;
            if (__ballot(in && n != n_lead) == 0) {   // the usual case: a bin of class 0 is one window size
                before_n = below * n_lead;
                all_n = __popcll(same) * n_lead;
            } else {
                int incl = in ? n : 0;
                for (int off = 1; off < 64; off <<= 1) {
                    const int up = __shfl_up(incl, off);
                    if (lane >= off) incl += up;
                }
                before_n = incl - (in ? n : 0);
                all_n = __builtin_amdgcn_readlane(incl, 63);
            }
            uint32_t c = 0, q = 0;
#pragma unroll
            for (int j = 0; j < kBins / 64; ++j)
                if ((cb >> 6) == j) { c = held_c[j]; q = held_s[j]; }
            c = __builtin_amdgcn_readlane(c, cb & 63);
            q = __builtin_amdgcn_readlane(q, cb & 63);
            if (in) got = make_int2(static_cast<int>(c) + below, static_cast<int>(q) + before_n);
#pragma unroll
            for (int j = 0; j < kBins / 64; ++j)
                if ((cb >> 6) == j && lane == (cb & 63)) { held_c[j] += __popcll(same); held_s[j] += all_n; }
            todo &= ~same;
        }
        if (w < end) place[w] = got;
    }
    // the wavefront's totals, and the workgroup's (what the place kernel sums over the launch)
    __shared__ unsigned long long wave_bins[kWaves][kBins];
    unsigned long long *sum_bins = group_bins + static_cast<size_t>(kListGroups) * kWaves * kBins;
#pragma unroll
    for (int j = 0; j < kBins / 64; ++j) {
        const unsigned long long v = (static_cast<unsigned long long>(held_c[j]) << 32) | held_s[j];
        group_bins[static_cast<size_t>(table) * kBins + j * 64 + lane] = v;
        wave_bins[threadIdx.x >> 6][j * 64 + lane] = v;
    }
    __syncthreads();
    unsigned long long sum = 0;
#pragma unroll
    for (int v = 0; v < kWaves; ++v) sum += wave_bins[v][threadIdx.x];
    sum_bins[static_cast<size_t>(group) * kBins + threadIdx.x] = sum;
}
__global__ __launch_bounds__(kListThreads) void sweep_count_kernel(AttnArgs a) { count_windows(a, blockIdx.x, gridDim.x); }

// sweep_place_kernel (same grid): bins in order, wavefronts in order inside a bin.  Writes one entry (first
// query of its class, voxels, first sorted position, class) per window in sorted order, one record per unit
// (the entry that holds its first query, lanes per query as a shift, first query, queries), the totals, and
// the queue counters at zero.
__device__ __forceinline__ void place_windows(const AttnArgs &a, int group, int groups)
{
    constexpr int kWaves = kListThreads / 64;
    __shared__ int bin_entry[kWaves][kBins], bin_slot[kWaves][kBins];
    __shared__ int wave_c[kWaves], wave_s[kWaves];
    __shared__ int class_base[kClasses + 1];       // queries before each class (index = kMaxSplit - g), and all
    __shared__ int total_entries_s;
    char *ws = static_cast<char *>(a.workspace);
    int *counters = reinterpret_cast<int *>(ws);
    int *total = reinterpret_cast<int *>(ws + ws_total_offset(a.H));
    int4 *unit_info = reinterpret_cast<int4 *>(ws + ws_units_offset(a.H));
    int4 *entries = reinterpret_cast<int4 *>(ws + ws_entries_offset(a.H, a.N));
    const int2 *place = reinterpret_cast<const int2 *>(ws + ws_place_offset(a.H, a.W, a.N));
    const unsigned long long *group_bins =
        reinterpret_cast<const unsigned long long *>(ws + ws_bins_offset(a.H, a.W, a.N));
    const int tables = groups * kWaves, first_table = group * kWaves;
    const unsigned long long *sum_bins = group_bins + static_cast<size_t>(kListGroups) * kWaves * kBins;
    // thread t holds bin t: the launch's total, and what the workgroups before this one put there; an exclusive
    // scan over the threads gives the bins their places (entries over all bins, queries restarting per class)
    {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        unsigned long long all = 0, before = 0;
#pragma unroll 8
        for (int g = 0; g < groups; ++g) {
            const unsigned long long v = sum_bins[static_cast<size_t>(g) * kBins + threadIdx.x];
            all += v;
            before += g < group ? v : 0;
        }
        const int cnt = static_cast<int>(all >> 32), slots = static_cast<int>(all & 0xffffffffu);
        int incl_c = cnt, incl_s = slots;
        for (int off = 1; off < 64; off <<= 1) {
            const int up_c = __shfl_up(incl_c, off), up_s = __shfl_up(incl_s, off);
            if (lane >= off) { incl_c += up_c; incl_s += up_s; }
        }
        if (lane == 63) { wave_c[wave] = incl_c; wave_s[wave] = incl_s; }
        __syncthreads();
        int base_c = 0, base_s = 0;
        for (int v = 0; v < wave; ++v) { base_c += wave_c[v]; base_s += wave_s[v]; }
        static_assert(kMaxSteps == 64, "a class is the bins of one wavefront of the scan");
        // queries are numbered per class: the class's bins are this wavefront's, so drop the earlier wavefronts' sum
#pragma unroll
        for (int v = 0; v < kWaves; ++v) {
            bin_entry[v][threadIdx.x] = base_c + incl_c - cnt + static_cast<int>(before >> 32);
            bin_slot[v][threadIdx.x] = incl_s - slots + static_cast<int>(before & 0xffffffffu);
            before += group_bins[static_cast<size_t>(first_table + v) * kBins + threadIdx.x];
        }
        if (lane == 0) class_base[wave] = base_s;
        if (threadIdx.x == kListThreads - 1) { class_base[kClasses] = base_s + incl_s; total_entries_s = base_c + incl_c; }
    }
    __syncthreads();
    const int total_entries = total_entries_s;
    // sections: classes kMaxSplit..1 in units of 64 >> g queries, then class 0 in its three kinds of unit
    int sec_unit[kSections + 1], class_total[kClasses];
#pragma unroll
    for (int c = 0; c < kClasses; ++c) class_total[c] = class_base[c + 1] - class_base[c];
    const UnitPlan plan = plan_units(class_total[kMaxSplit], a.target_items);
    sec_unit[0] = 0;
#pragma unroll
    for (int c = 0; c < kMaxSplit; ++c) {
        const int per = kChunk >> (kMaxSplit - c);
        sec_unit[c + 1] = sec_unit[c] + (class_total[c] + per - 1) / per;
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) sec_unit[kMaxSplit + k + 1] = sec_unit[kMaxSplit + k] + plan.units[k];
    const int W = static_cast<int>(a.W);
    const int my_wave = threadIdx.x >> 6;
    const int per_wave = (W + tables - 1) / tables;     // the count kernel's runs
    const int begin = min((first_table + my_wave) * per_wave, W), end = min(begin + per_wave, W);
    for (int w = begin + (threadIdx.x & 63); w < end; w += 64) {
        const int2 got = place[w];
        if (got.x < 0) continue;
        const int n = a.w_sizes[w];
        const int g = window_class(n, a.block_shift), b = window_bin(n, g);
        const int e = bin_entry[my_wave][b] + got.x;
        const int s = bin_slot[my_wave][b] + got.y;      // first query of the window inside its class
        entries[e] = make_int4(s, n, a.w2n[w], g);
        const int s_end = s + n;
        if (g > 0) {
            // the units whose first query is one of this window's
            const int size = kChunk >> g, c = kMaxSplit - g, all = class_total[c];
            for (int v = (s + size - 1) / size; v * size < s_end; ++v)
                unit_info[sec_unit[c] + v] = make_int4(e, g, v * size, min(size, all - v * size));
        } else {
            const int all = class_total[kMaxSplit];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const int size = kChunk >> k, from = plan.first_slot(k), count = plan.units[k];
                int v = s <= from ? 0 : (s - from + size - 1) / size;
                for (; v < count && from + v * size < s_end; ++v)
                    unit_info[sec_unit[kMaxSplit + k] + v] = make_int4(e, k, from + v * size, min(size, all - (from + v * size)));
            }
        }
    }
    if (group == 0) {
        // a wavefront reads 64 entries from a unit's first one: pad the list with entries no query belongs to
        if (threadIdx.x < kChunk) entries[total_entries + threadIdx.x] = make_int4(0x7fffffff, 1, 0, -1);
        if (threadIdx.x == 0) {
            total[0] = sec_unit[kSections];
            total[1] = 0;   // exit counters of a sweep launch: cache lines that are complete, and one per line
        }
        if (threadIdx.x < kQueues) total[(1 + threadIdx.x) * kCounterStride] = 0;
        for (int t = threadIdx.x; t < a.H * kQueues; t += kListThreads) counters[t * kCounterStride] = 0;
    }
}
__global__ __launch_bounds__(kListThreads) void sweep_place_kernel(AttnArgs a) { place_windows(a, blockIdx.x, gridDim.x); }

// Few windows, of which every wavefront has one round: both steps by one workgroup, and the strip list, where it is asked for, by
// another beside it.  A plan for strips of 2 windows 10.1 us (three launches) -> 5.8, of 84 windows 14.4 -> 8.9; at 340 windows, two
// rounds, one launch takes 17.2 and two 11.6.
__global__ __launch_bounds__(kListThreads) void sweep_list_kernel(AttnArgs a, tile::StripList also)
{
    if (blockIdx.x == 1) {
        tile::build_strip_list<kListThreads>(a.w_sizes, a.w2n, static_cast<int>(a.W), const_cast<int32_t *>(also.total),
                                             const_cast<uint64_t *>(also.strips));
        return;
    }
    count_windows(a, 0, 1);
    __threadfence();
    __syncthreads();
    place_windows(a, 0, 1);
}

void launch_work_list(const AttnArgs &a, hipStream_t stream, bool strips_too = false)
{
    if (a.W <= kFewWindows) {
        hipLaunchKernelGGL(sweep_list_kernel, dim3(strips_too ? 2 : 1), dim3(kListThreads), 0, stream, a,
                           strips_too ? attn_strip_list(a) : tile::StripList{});
        return;
    }
    const int64_t want = ceil_div(a.W, kListThreads);
    const dim3 grid(static_cast<unsigned>(want > kListGroups ? kListGroups : want));
    hipLaunchKernelGGL(sweep_count_kernel, grid, dim3(kListThreads), 0, stream, a);
    hipLaunchKernelGGL(sweep_place_kernel, grid, dim3(kListThreads), 0, stream, a);
}

// The work list of a records sweep beside the lists of the strips that read the records (head_dim 8): the strips' list is one
// workgroup's for 30 us where windows are many, and the sweep's, two short launches, is made meanwhile.  A call, forward included, us, with
// launches of their own / so: 199,327 voxels x 6 fp16 1466 / 1457, fp32 beside fp16 rows 1564 / 1555, 60,001 x 10 with six axes 754 / 746.
template <bool kScales>
__global__ __launch_bounds__(tile::kListThreads) void records_lists_kernel(tile::StripArgs strips, AttnArgs a, int jobs)
{
    const int block = static_cast<int>(blockIdx.x) - jobs, groups = static_cast<int>(gridDim.x) - jobs;
    if (block < 0) {
        tile::strip_setup<kScales>(strips, block + jobs);
        return;
    }
    if (threadIdx.x >= kListThreads) return;
    count_windows(a, block, groups);
    if (a.W > kFewWindows) return;
    __threadfence();
    __syncthreads();
    place_windows(a, 0, 1);
}
__global__ __launch_bounds__(kListThreads) void records_places_kernel(tile::StripSetup strips, AttnArgs a, int groups)
{
    const int block = static_cast<int>(blockIdx.x);
    if (block < groups) place_windows(a, block, groups);
    else tile::strip_column(strips, (block - groups) * kListThreads + static_cast<int>(threadIdx.x));
}
int launch_records_lists(const tile::StripSetup &strips, const AttnArgs &a, bool scales, hipStream_t stream)
{
    const int groups = a.W <= kFewWindows ? 1 : static_cast<int>(std::min<int64_t>(ceil_div(a.W, kListThreads), kListGroups));
    const int jobs = 1 + 2 * a.H, places = a.W <= kFewWindows ? 0 : groups;
    hipLaunchKernelGGL(scales ? records_lists_kernel<true> : records_lists_kernel<false>, dim3(static_cast<unsigned>(jobs + groups)),
                       dim3(tile::kListThreads), 0, stream, strips.b, a, jobs);
    const int64_t columns = static_cast<int64_t>(tile::list_max_strips(a.N)) * tile::kStrip;
    hipLaunchKernelGGL(records_places_kernel, dim3(static_cast<unsigned>(places + ceil_div(columns, kListThreads))), dim3(kListThreads), 0, stream,
                       strips, a, places);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

// Which head group a workgroup serves, for its whole life, and which of its workgroups it is.  Workgroups go to the XCDs in turn:
// runs of eight consecutive ones serve one head group, as far as whole sets of (XCDs x head groups) go, so that every XCD serves
// every head group and the rows of a unit reach one L2; the head groups take the workgroups behind those in turn.  (All in turn, an
// even number of head groups meets only some of the XCDs: 199,327 voxels x 6 heads of 8 200 -> 215 us.  Without the ones behind,
// sixteen of 256 CUs had no workgroup at 6, 10, 12 and 20 heads of 16: with them 149,993 x 10 1036 -> 1018 us, 49,682 x 6 278 -> 271,
// 37,485 x 20 664 -> 651.  At 24 and 40 heads, all of whose workgroups came in turn, 9,000 x 24 285 -> 266, 9,400 x 40 443 -> 432.)
struct GroupPlace {
    int head_group, nth, of;       // its workgroups are numbered
    __device__ __forceinline__ GroupPlace(const AttnArgs &a, int groups)
    {
        const int block = static_cast<int>(blockIdx.x), behind = block - a.set_groups;
        head_group = behind < 0 ? block / kQueues % groups : behind % groups;
        nth = behind < 0 ? block / (kQueues * groups) * kQueues + block % kQueues : (a.set_groups + behind) / groups;
        of = static_cast<int>(gridDim.x) / groups;
    }
};
// The units of a head group, by queues, of which a wavefront starts on that of its workgroup's number: its XCD's, for workgroups of
// whole sets; those behind them need not meet theirs.  (By the number and not by the XCD's register, so that a wavefront's own unit is
// one no other has.)
// In launches of up to two units a wavefront the first one is the wavefront's own: the first four wavefronts of all workgroups
// come before their next four, so that all CUs get some, long ones and short ones.  By tickets alone the workgroups that had
// their tables first took more than their share.  us by tickets / so, 9 axes, fp16: 20,001 voxels x 6 heads of 8 70.1 / 55.7,
// 50,001 x 6 96.3 / 79.8, 2,003 x 10 49.5 / 42.1, 9,001 x 12 of 16 148.4 / 145.2; fp32 20,001 x 6 of 8 83.4 / 68.2.  Where there are
// more units, tickets leave those of a window to one CU's wavefronts, whose lines they share: 12,421 x 12 of 16 174, all first units
// given 185.  (One wavefront at a time instead of four 54.6 and 183.5 at the first and the last of these; six 70 and 185.)
// The line at two: of 113 shapes of up to two units, 64 of them with more than one, 0.55 to 1.01 of the time by tickets, but fp16 with
// three or six axes at 1.1 to 1.4 units takes 1.01 to 1.07 with 24 heads of 16 (2,701 voxels, six axes 99.9 / 107.1, nine 117.3 /
// 114.2) and 1.02 to 1.05 with 12 (6,001).  A line at 9/8 for those takes some of that back and loses more elsewhere: 15,001 x 6 with six
// axes, 1.56 units, 91 -> 102, 5,501 x 12 94 -> 97.5.
// Another stream's work can keep a workgroup, and its units, from a CU.  Calls on two streams at once, us a pair, by tickets / so: two
// of 20,001 x 6 87.0 / 83.0, two of 50,001 x 6 146.4 / 149.5, two of 9,001 x 12 of 16 266.0 / 263.8, in fp32 two of 20,001 x 6 107.9 /
// 112.6; beside products of 50,000 x 192 x 192 50,001 x 6 94.8 / 87.1, 20,001 x 6 71.7 / 71.9; 20,001 x 6 beside copies 96.5 / 88.2,
// beside 149,993 x 10 of 16 998 / 998, beside a call with gradients 358 / 354.
template <int kWaves> struct UnitQueues {
    static constexpr int kSide = kWaves % 4 == 0 ? 4 : 1;
    int *counters;
    int of, total, lane, queue, drawn, tried = 0;      // drawn: the ticket, of lane 0
    __device__ __forceinline__ UnitQueues(int *head_counters, const GroupPlace &p, int units)
        : counters(head_counters), of(p.of), total(units), lane(static_cast<int>(threadIdx.x & 63)), queue(p.nth % kQueues)
    {
        const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
        drawn = (wave / kSide * places(queue) + p.nth / kQueues) * kSide + wave % kSide;
        if (given(queue) == 0) draw();
    }
    __device__ __forceinline__ int places(int q) const { return (of - q + kQueues - 1) / kQueues; }      // workgroups that start on it
    // how many of a queue's units have a wavefront of their own
    __device__ __forceinline__ int given(int q) const
    {
        const int waves = kWaves * places(q);
        return total - q <= 2 * kQueues * waves ? waves : 0;
    }
    __device__ __forceinline__ void draw()
    {
        const int first = given(queue);
        if (lane == 0) drawn = first + atomicAdd(counters + queue * kCounterStride, 1);
    }
    // the unit drawn, or one of the other queues where there is none; -1: all are empty
    __device__ __forceinline__ int unit()
    {
        int u = __builtin_amdgcn_readfirstlane(drawn) * kQueues + queue;
        while (u >= total && ++tried < kQueues) {
            queue = (queue + 1) % kQueues;
            u = given(queue) * kQueues + queue;
            if (u >= total) continue;
            draw();
            u = __builtin_amdgcn_readfirstlane(drawn) * kQueues + queue;
        }
        return u < total ? u : -1;
    }
};
// The grid for `slots` workgroups at a time.  The work list is cut for as many wavefronts as whole sets have, or, where those
// leave more than a tenth of the slots empty, for all.  (The key-owned sweep of the backward, whose records' lines bound it, stays
// with whole sets: 370 us, 386 with workgroups behind them, 199,327 voxels x 6 heads of 8 in fp32.)
int place_groups(AttnArgs &a, int slots, int groups, int threads, bool whole_sets = false)
{
    const int set = kQueues * groups, all = slots >= groups ? slots / groups * groups : groups;
    a.set_groups = slots / set * set;
    a.target_items = (10 * a.set_groups < 9 * slots ? all : a.set_groups) / groups * (threads / 64);
    return whole_sets && 10 * a.set_groups >= 9 * slots ? a.set_groups : all;
}

// Workgroup shapes.  A workgroup holds its heads' table slices once: up to head_dim 16 one of twelve wavefronts a CU, three per SIMD
// with 168 registers (fp16 75 KB of tables for two heads of 16, 45 for three of 8; fp32 65 for two heads of 8, 75 for one of 16).
// With the rows read ahead three wavefronts hide what four hid, and the tables are staged once: against four workgroups of four
// wavefronts at head_dim 8 with one and two heads, fp16, 9 axes, us 595,677 voxels x 10 heads 918 / 919, 100,003 x 10 213 / 200,
// 20,003 x 10 87 / 72, 2,003 x 10 76 / 50, 100,003 x 5 138 / 123, fp32 20,001 x 5 77 / 54; two of eight, three or four per SIMD, 978
// and 939 at 595,677; two of eight for pairs of heads in fp32 330 for 299 (199,327 x 6).  Two of six at head_dim 16 25 % slower than
// one of twelve.  fp16, one head of 16 a wavefront, which reads nothing ahead, three workgroups of four / one of twelve: 9,001 x 15
// 213 / 199, 60,001 x 5 298 / 294, 20,001 x 5 138 / 136, 150,001 x 3 390 / 388, with six axes 150,001 x 5 435 / 434.
// head_dim 32 (an fp32 query, key, value and output row are 128 registers): two of four wavefronts in fp16, one of eight in fp32
// (125 KB of tables).
template <typename T, int D> __host__ __device__ constexpr int group_threads() { return D <= 16 ? 768 : sizeof(T) == 4 ? 512 : 256; }
template <typename T, int D> __host__ __device__ constexpr int groups_per_cu() { return D <= 16 || sizeof(T) == 4 ? 1 : 2; }

// elements of T between table rows in LDS when a workgroup holds the slices of HP heads side by side
template <typename T, int D, int HP> __host__ __device__ constexpr int table_row_stride_heads()
{
    return HP * 3 * D + ((HP * 3 * D * static_cast<int>(sizeof(T)) / 4) % 8 == 0 ? 16 / static_cast<int>(sizeof(T)) : 0);
}

// HP: heads a wavefront carries through a unit (adjacent heads HP * g .. HP * g + HP - 1).  The cRSE rows and
// LDS addresses of a pair do not depend on the head, so two or three heads share that part of the work.
// kSorted: q, k, v and out rows are in window-sorted order already (no n2n).
template <typename T, int D, int ND, int HP, bool kSorted>
__global__ __launch_bounds__((group_threads<T, D>()), (groups_per_cu<T, D>())) void attn_fwd_sweep_kernel(AttnArgs a)
{
    constexpr int kThreads = group_threads<T, D>();
    // streamed keys per loop iteration: in fp16 at head_dim 16 with one head two interleaved chains hide the LDS round trips
    constexpr int kKeys = sizeof(T) == 2 && D == 16 && HP == 1 ? 2 : 1;
    // lazy softmax reference (see the loop): -4 % for fp16; fp32 measured no gain (head_dim 8) or a loss (16)
    constexpr bool kLazy = sizeof(T) == 2;
    // What hides the round trips where a lane has one key at a time.  The table rows of the next axis are read from LDS before the
    // products of this one's, and the next key with its signals is asked for once its predecessor's logits stand, in its
    // registers; the compiler's own order waited for every row right behind its read.  us without / so, 9 axes, fp16: 149,993
    // voxels x 10 heads of 16 1104 / 1019, 12,421 x 12 192 / 176, 9,400 x 40 470 / 431, 199,327 x 6 of 8 207 / 200; fp32: 120,001 x
    // 6 of 16 868 / 798, with six axes 60,001 x 12 785 / 746 (two keys at a time before), 199,327 x 6 of 8 327 / 299, 20,001 x 5 83 / 77.
    // Two rows ahead at head_dim 16 in fp16 spills 30 registers (1469), and eight wavefronts with room for it are slower (1111).
    constexpr bool kAhead = D <= 16 && kKeys == 1;
    // fp32, head_dim 16: a pair's value and its rows of the value table are added before they are weighted, so that the output's sums are
    // rounded once a key.  One key at a time moves the softmax's reference more often than two did, at 1.0004 times their error against
    // 64 bits (31 of 33 shapes, voxels 3,001 to 120,001, 3 to 9 axes); summed first it is 0.69 to 0.87 of it, 2.77e-7 -> 2.03e-7 at
    // 60,001 x 6 with 9 axes, in the same time: 120,001 x 6 in windows of 26 367 / 362 us, of 57 796 / 790 (two keys at a time 404 and 898).
    constexpr bool kSumFirst = sizeof(T) == 4 && D == 16;
    static_assert(!kSumFirst || kAhead, "in the loop that reads ahead");
    // 16-byte aligned like the table rows behind it, which are read 16 bytes at a time
    extern __shared__ __align__(16) float smem[];
    __shared__ __align__(16) int group_exit_counter[4];   // [0]: wavefronts of this workgroup that have left their loop
    int &group_exited = group_exit_counter[0];
    if (threadIdx.x == 0) group_exited = 0;
    const int H = a.H;
    const int HD = H * D;
    if (a.leave_to_tiles) {
        int rows[ND], run = 0;
#pragma unroll
        for (int n = 0; n < ND; ++n) run += rows[n] = device_rows(a, n, ND, run);
        if (rows_fit_tiles(rows, ND)) return;
    }
    const GroupPlace place(a, H / HP);
    const int hg = place.head_group;
    const int h = hg * HP;   // first head of the group
    // table slices of the heads in the I/O type, interleaved per row: [head][q-side | k-side | v-side]
    constexpr int kRowStride = table_row_stride_heads<T, D, HP>();
    T *tab = reinterpret_cast<T *>(smem);
    {
        const T *gq = static_cast<const T *>(a.table_q);
        const T *gk = static_cast<const T *>(a.table_k);
        const T *gv = static_cast<const T *>(a.table_v);
        // 16-byte pieces: a (row, head) slice of a table is D * sizeof(T) / 16 of them
        constexpr int kPieces = D * static_cast<int>(sizeof(T)) / 16;
        constexpr int kPerPiece = 16 / static_cast<int>(sizeof(T));
        for (int t = threadIdx.x; t < a.total_rows * HP * kPieces; t += kThreads) {
            const int r = t / (HP * kPieces), hp = t - r * (HP * kPieces);
            const int hh = hp / kPieces, c = (hp - hh * kPieces) * kPerPiece;
            const int64_t g = static_cast<int64_t>(r) * HD + (h + hh) * D + c;
            T *row = tab + r * kRowStride + hh * 3 * D + c;
            *reinterpret_cast<uint4 *>(row) = *reinterpret_cast<const uint4 *>(gq + g);
            *reinterpret_cast<uint4 *>(row + D) = *reinterpret_cast<const uint4 *>(gk + g);
            *reinterpret_cast<uint4 *>(row + 2 * D) = *reinterpret_cast<const uint4 *>(gv + g);
        }
    }
    __syncthreads();   // the only workgroup barrier

    const int lane = threadIdx.x & 63;
    const T *gq = static_cast<const T *>(a.q);
    const T *gk = static_cast<const T *>(a.k);
    const T *gv = static_cast<const T *>(a.v);
    const char *ws = static_cast<const char *>(a.workspace);
    const int4 *unit_info = reinterpret_cast<const int4 *>(ws + ws_units_offset(H));
    const int4 *entries = reinterpret_cast<const int4 *>(ws + ws_entries_offset(H, a.N));
    const int total_units = __builtin_amdgcn_readfirstlane(reinterpret_cast<const int *>(ws + ws_total_offset(H))[0]);
    int *counters = static_cast<int *>(a.workspace) + hg * kQueues * kCounterStride;
    constexpr int kRowBytes = kRowStride * static_cast<int>(sizeof(T));
    constexpr uint32_t kHeadBytes = 3 * D * sizeof(T);   // one head's slices inside a row
    const uint32_t tab_addr = __builtin_amdgcn_readfirstlane(lds_address(tab));
    const uint32_t row_bytes = kRowBytes;
    float half_rows[ND], upper[ND];
    uint32_t base_off[ND];
    {
        // rows of every axis table: kernel arguments, or (sizes_dev) read from the caller's device tensor of table
        // sizes, which the host has not seen - clipped so that every axis keeps a row inside the head's table
        int run = 0;
#pragma unroll
        for (int n = 0; n < ND; ++n) {
            int rows = a.rows[n], first = a.base[n];
            if (a.sizes_dev) {
                rows = device_rows(a, n, ND, run);
                first = run;
                run += rows;
            }
            half_rows[n] = static_cast<float>(rows / 2);
            upper[n] = crse_upper(rows);
            // LDS byte address of the axis table's first row
            base_off[n] = __builtin_amdgcn_readfirstlane(tab_addr + first * kRowBytes);
        }
    }

    UnitQueues<kThreads / 64> queues(counters, place, total_units);
    for (;;) {
        const int unit = queues.unit();
        if (unit < 0) break;
        // The unit: 64 >> gshift queries (consecutive in the sorted numbering of their class), each on 2^gshift
        // adjacent lanes that take alternate keys.  The queries lie in at most 64 consecutive entries from the
        // unit's first one; each lane reads one entry and finds its own (the last entry of the class that starts at
        // or before its query) by a search across the lanes.
        const int4 info = unit_info[unit];
        const int first = __builtin_amdgcn_readfirstlane(info.x);
        const int gshift = __builtin_amdgcn_readfirstlane(info.y);
        const int queries = __builtin_amdgcn_readfirstlane(info.w);
        const int sub = lane & ((1 << gshift) - 1);
        const bool own_valid = (lane >> gshift) < queries;
        const int query = __builtin_amdgcn_readfirstlane(info.z) + min(lane >> gshift, queries - 1);   // lanes past the end repeat the last one
        const int4 seen = entries[first + lane];
        const int seen_from = seen.w == __builtin_amdgcn_readfirstlane(seen.w) ? seen.x : 0x7fffffff;   // the next class restarts at 0
        int at = 0;
#pragma unroll
        for (int half = 32; half > 0; half >>= 1)
            if (__shfl(seen_from, at + half) <= query) at += half;
        const int n_w = __shfl(seen.y, at), s0 = __shfl(seen.z, at);
        const int own_pos = s0 + (query - __shfl(seen.x, at));
        const int own_row = kSorted ? own_pos : a.n2n[own_pos];
        // the longest lane of the unit (entries are sorted by steps, but windows beyond the longest bin are not)
        int max_steps = (n_w + (1 << gshift) - 1) >> gshift;
#pragma unroll
        for (int other = 32; other > 0; other >>= 1) max_steps = max(max_steps, __shfl_xor(max_steps, other));
        max_steps = __builtin_amdgcn_readfirstlane(max_steps);
        // the lane's keys: sub, sub + 2^gshift, ... of the window's n_k
        const int n_k = n_w;
        const int k0 = s0;
        const int grp = sub;

        Slice<T, D> qv[HP];
        float ci[ND], acc[HP][D], m[HP], top[HP], l[HP];
#pragma unroll
        for (int hh = 0; hh < HP; ++hh) {
            qv[hh].load(gq + static_cast<int64_t>(own_row) * a.row_stride + (h + hh) * D);
#pragma unroll
            for (int c = 0; c < D; ++c) acc[hh][c] = 0.0f;
            // (the lowest finite number: a key whose logit is minus infinity has no weight, also where a lane sees it first)
            m[hh] = -3.4028234663852886e38f;
            top[hh] = -INFINITY;
            l[hh] = 0.0f;
        }
#pragma unroll
        for (int n = 0; n < ND; ++n) ci[n] = a.n_coords[static_cast<int64_t>(own_pos) * ND + n];

        // kKeys streamed keys per iteration: their loads and dependent chains interleave, which hides the
        // LDS and cache round trips a single chain would wait out one after the other
        int row_next[kKeys], row_now[kKeys];
        Slice<T, D> kv[kKeys][HP];
        float cj[kKeys][ND];
#pragma unroll
        for (int u = 0; u < kKeys; ++u) row_next[u] = kSorted ? 0 : a.n2n[k0 + min((u << gshift) + grp, n_k - 1)];
        auto row_at = [&](int row) { return static_cast<uint64_t>(static_cast<uint32_t>(row)) * static_cast<uint64_t>(a.row_stride); };
        // the keys of an iteration and their signals
        auto fetch_keys = [&](int it) {
#pragma unroll
            for (int u = 0; u < kKeys; ++u) {
                const int st = ((it + u) << gshift) + grp;
                const int st_pos = k0 + min(st, n_k - 1);
                row_now[u] = kSorted ? st_pos : row_next[u];
                if (!kSorted) row_next[u] = a.n2n[k0 + min(st + (kKeys << gshift), n_k - 1)];
#pragma unroll
                for (int n = 0; n < ND; ++n) cj[u][n] = a.n_coords[static_cast<uint64_t>(static_cast<uint32_t>(st_pos)) * ND + n];
#pragma unroll
                for (int hh = 0; hh < HP; ++hh) kv[u][hh].load(gk + (row_at(row_now[u]) + static_cast<uint32_t>((h + hh) * D)));
            }
        };
        if constexpr (kAhead) fetch_keys(0);
        for (int it = 0; it < max_steps; it += kKeys) {
            // the next unit's ticket is drawn during the last iteration: the atomic's round trip overlaps that
            // work, and a unit is not held back (out of reach of idle wavefronts) for longer than one step
            if (it + kKeys >= max_steps) queues.draw();
            Slice<T, D> v_in[kKeys][HP];
            float logit[kKeys][HP];
            uint32_t off[kKeys][ND];
            bool valid[kKeys];
            auto load_values = [&](int u) {
#pragma unroll
                for (int hh = 0; hh < HP; ++hh) v_in[u][hh].load(gv + (row_at(row_now[u]) + static_cast<uint32_t>((h + hh) * D)));
            };
            if constexpr (!kAhead) fetch_keys(it);
#pragma unroll
            for (int u = 0; u < kKeys; ++u) {
                valid[u] = ((it + u) << gshift) + grp < n_k;
                if constexpr (!kAhead) load_values(u);
#pragma unroll
                for (int n = 0; n < ND; ++n)
                    off[u][n] = mad_u24(static_cast<uint32_t>(crse_row(ci[n], cj[u][n], half_rows[n], upper[n])), row_bytes, base_off[n]);
            }
            if constexpr (kAhead) {
                // rows of the q-side table and of the k-side table in turn, of all heads, the next ones on their way; the values
                // of the keys are asked for once the registers of the first rows are free
                constexpr int kItems = 2 * ND, kAskForValues = 4;
                Slice<T, D> rows[2][HP];
                float of_axis[HP];
                auto read = [&](int i) {
#pragma unroll
                    for (int hh = 0; hh < HP; ++hh) rows[i % 2][hh].load_lds(off[0][i / 2] + hh * kHeadBytes + (i % 2) * D * sizeof(T));
                };
                read(0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int hh = 0; hh < HP; ++hh) logit[0][hh] = qv[hh].dot(kv[0][hh], 0.0f);
#pragma unroll
                for (int i = 0; i < kItems; ++i) {
                    if (i == kAskForValues) load_values(0);
                    if (i + 1 < kItems) read(i + 1);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int hh = 0; hh < HP; ++hh) {
                        const Slice<T, D> &mine = i % 2 ? kv[0][hh] : qv[hh];
                        if constexpr (Slice<T, D>::kChainLogit) {
                            logit[0][hh] = mine.dot(rows[i % 2][hh], logit[0][hh]);
                        } else {
                            of_axis[hh] = mine.dot(rows[i % 2][hh], i % 2 ? of_axis[hh] : 0.0f);
                            if (i % 2) logit[0][hh] += of_axis[hh];
                        }
                    }
                }
                // (or the compiler moves the products below `valid`, away from their rows)
#pragma unroll
                for (int hh = 0; hh < HP; ++hh) asm volatile("" : "+v"(logit[0][hh]));
            } else {
#pragma unroll
                for (int u = 0; u < kKeys; ++u) {
#pragma unroll
                    for (int hh = 0; hh < HP; ++hh) logit[u][hh] = qv[hh].dot(kv[u][hh], 0.0f);
#pragma unroll
                    for (int n = 0; n < ND; ++n) {
#pragma unroll
                        for (int hh = 0; hh < HP; ++hh) {
                            Slice<T, D> tq_r, tk_r;
                            tq_r.load_lds(off[u][n] + hh * kHeadBytes);
                            tk_r.load_lds(off[u][n] + hh * kHeadBytes + D * sizeof(T));
                            if (Slice<T, D>::kChainLogit) logit[u][hh] = kv[u][hh].dot(tk_r, qv[hh].dot(tq_r, logit[u][hh]));
                            else logit[u][hh] += kv[u][hh].dot(tk_r, qv[hh].dot(tq_r, 0.0f));
                        }
                    }
                }
            }
            // (the value rows, two of them on their way)
            constexpr int kRows = HP * ND, kOnWay = 2;
            Slice<T, D> rows[kOnWay + 1];
            auto read = [&](int r) { rows[r % (kOnWay + 1)].load_lds(off[0][r % ND] + r / ND * kHeadBytes + 2 * D * sizeof(T)); };
            if constexpr (kAhead) {
#pragma unroll
                for (int r = 0; r < kOnWay; ++r) read(r);
                fetch_keys(it + kKeys);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (!kLazy) {
                // online softmax: the running maximum moves with every key that raises it
                if (valid[0]) {   // the lowest key of the iteration; lanes whose block has ended sit the step out
#pragma unroll
                    for (int hh = 0; hh < HP; ++hh) {
                        float m_new = fmaxf(m[hh], logit[0][hh]);
#pragma unroll
                        for (int u = 1; u < kKeys; ++u) {
                            logit[u][hh] = valid[u] ? logit[u][hh] : -INFINITY;
                            m_new = fmaxf(m_new, logit[u][hh]);
                        }
                        const float scale = __expf(m[hh] - m_new);   // 0 on the first key
                        l[hh] *= scale;
#pragma unroll
                        for (int c = 0; c < D; ++c) acc[hh][c] *= scale;
#pragma unroll
                        for (int u = 0; u < kKeys; ++u) {
                            const float p = __expf(logit[u][hh] - m_new);
                            l[hh] += p;
                            if constexpr (!kSumFirst) v_in[u][hh].fma_to(acc[hh], p);
                            if constexpr (kAhead) {
#pragma unroll
                                for (int n = 0; n < ND; ++n) {
                                    const int r = hh * ND + n;
                                    if (r + kOnWay < kRows) read(r + kOnWay);
                                    __builtin_amdgcn_sched_barrier(0);
                                    if constexpr (kSumFirst) v_in[u][hh].add(rows[r % (kOnWay + 1)]);
                                    else rows[r % (kOnWay + 1)].fma_to(acc[hh], p);
                                }
                                if constexpr (kSumFirst) v_in[u][hh].fma_to(acc[hh], p);
                            } else
#pragma unroll
                            for (int n = 0; n < ND; ++n) {
                                Slice<T, D> tv_r;
                                tv_r.load_lds(off[u][n] + hh * kHeadBytes + 2 * D * sizeof(T));
                                tv_r.fma_to(acc[hh], p);
                            }
                        }
                        m[hh] = m_new;
                    }
                }
            } else {
                // Online softmax against a reference exponent m that follows the running maximum lazily: it moves
                // (and the sums are rescaled) only when the lane's logit exceeds it by more than kSlack, which
                // after the first keys of a unit is rare, so most steps skip the rescaling of l and the D outputs;
                // weights stay below e^kSlack.  `top` is the true running maximum.
                float hi[HP];
                bool moved = false;
#pragma unroll
                for (int hh = 0; hh < HP; ++hh) {
                    hi[hh] = logit[0][hh];
#pragma unroll
                    for (int u = 1; u < kKeys; ++u) {
                        logit[u][hh] = valid[u] ? logit[u][hh] : -INFINITY;
                        hi[hh] = fmaxf(hi[hh], logit[u][hh]);
                    }
                    moved = moved || hi[hh] > m[hh] + kSlack;
                }
                // each lane decides for itself, so the bits of a query's result do not depend on which other queries
                // share its wavefront
                if (valid[0] && moved) {
#pragma unroll
                    for (int hh = 0; hh < HP; ++hh) {
                        const float m_new = fmaxf(m[hh], hi[hh]);
                        const float scale = __expf(m[hh] - m_new);   // 0 on the first key
                        l[hh] *= scale;
#pragma unroll
                        for (int c = 0; c < D; ++c) acc[hh][c] *= scale;
                        m[hh] = m_new;
                    }
                }
                if (valid[0]) {   // the lowest key of the iteration; lanes whose block has ended sit the step out
#pragma unroll
                    for (int hh = 0; hh < HP; ++hh) {
                        top[hh] = fmaxf(top[hh], hi[hh]);
#pragma unroll
                        for (int u = 0; u < kKeys; ++u) {
                            const float p = __expf(logit[u][hh] - m[hh]);
                            l[hh] += p;
                            v_in[u][hh].fma_to(acc[hh], p);
                            // The pair's value-table rows are added three at a time in packed fp16, two channels per
                            // instruction, before they enter the fp32 sums: 56 instructions per pair and head at
                            // head_dim 8 instead of 80 mixed-precision FMAs.  Groups of three keep the fp16 roundings
                            // at two per element, on sums of three rows (one chain over all nine rows saves eight
                            // more instructions, measured 13 % slower - eight dependent adds - and used up the 2e-3
                            // error budget on tables of magnitude 0.1); adding the value here as well measured -4 %
                            // for the same reason not to.  The reference's half path adds all rows and the value in
                            // half2 (self_attn_aio_fwd.cu:147).
                            constexpr int kGroup = 3;
                            Slice<T, D> sum_of_rows;
                            if constexpr (kAhead) {
#pragma unroll
                                for (int n = 0; n < ND; ++n) {
                                    const int r = hh * ND + n;
                                    if (r + kOnWay < kRows) read(r + kOnWay);
                                    __builtin_amdgcn_sched_barrier(0);
                                    if (n % kGroup == 0) sum_of_rows = rows[r % (kOnWay + 1)];
                                    else sum_of_rows.add(rows[r % (kOnWay + 1)]);
                                    if (n % kGroup == kGroup - 1 || n == ND - 1) sum_of_rows.fma_to(acc[hh], p);
                                }
                            } else
#pragma unroll
                            for (int n0 = 0; n0 < ND; n0 += kGroup) {
                                Slice<T, D> tv_sum;
                                tv_sum.load_lds(off[u][n0] + hh * kHeadBytes + 2 * D * sizeof(T));
#pragma unroll
                                for (int g = 1; g < kGroup && n0 + g < ND; ++g) {
                                    Slice<T, D> tv_r;
                                    tv_r.load_lds(off[u][n0 + g] + hh * kHeadBytes + 2 * D * sizeof(T));
                                    tv_sum.add(tv_r);
                                }
                                tv_sum.fma_to(acc[hh], p);
                            }
                        }
                    }
                }
            }
        }
        // from the reference exponent to the true maximum (lanes that saw no key with a weight: that is -inf, nothing to scale)
        if constexpr (!kLazy) {
#pragma unroll
            for (int hh = 0; hh < HP; ++hh) m[hh] = l[hh] == 0.0f ? -INFINITY : m[hh];
        } else {
#pragma unroll
            for (int hh = 0; hh < HP; ++hh) {
                const float scale = top[hh] == -INFINITY ? 1.0f : __expf(m[hh] - top[hh]);
                l[hh] *= scale;
#pragma unroll
                for (int c = 0; c < D; ++c) acc[hh][c] *= scale;
                m[hh] = top[hh];
            }
        }
#pragma unroll
        for (int hh = 0; hh < HP; ++hh) {
            // lanes that share a query saw alternate keys: merge their softmax states
            for (int other = 1; other < (1 << gshift); other <<= 1) {
                const float m_o = __shfl_xor(m[hh], other), l_o = __shfl_xor(l[hh], other);
                const float m_all = fmaxf(m[hh], m_o);
                const float w_me = (m[hh] == -INFINITY) ? 0.0f : __expf(m[hh] - m_all);
                const float w_ot = (m_o == -INFINITY) ? 0.0f : __expf(m_o - m_all);
                l[hh] = l[hh] * w_me + l_o * w_ot;
#pragma unroll
                for (int c = 0; c < D; ++c) acc[hh][c] = acc[hh][c] * w_me + __shfl_xor(acc[hh][c], other) * w_ot;
                m[hh] = m_all;
            }
            if (own_valid && sub == 0) {
                const float inv = 1.0f / l[hh];
#pragma unroll
                for (int c = 0; c < D; ++c) acc[hh][c] *= inv;
                store_row<D>(static_cast<T *>(a.out) + static_cast<int64_t>(own_row) * HD + (h + hh) * D, acc[hh]);
                if (a.out_max) a.out_max[static_cast<int64_t>(own_row) * H + h + hh] = m[hh];
                if (a.out_sum) a.out_sum[static_cast<int64_t>(own_row) * H + h + hh] = l[hh];
            }
        }
    }
    // The work list can serve further launches (a plan kept by the caller): the last wavefront of the launch to
    // leave its loop - by then no wavefront draws tickets any more - puts every queue counter back to zero.  The
    // exits are counted in three levels (workgroup in LDS, one of kQueues cache lines, all lines), so that no
    // cache line sees more than a few hundred of these atomics.
    if (lane == 0 && atomicAdd(&group_exited, 1) == kThreads / 64 - 1) {
        __threadfence();
        int *total = static_cast<int *>(a.workspace) + ws_total_offset(H) / sizeof(int);
        const int groups = static_cast<int>(gridDim.x), line = static_cast<int>(blockIdx.x) % kQueues;
        const int on_line = (groups - line + kQueues - 1) / kQueues;
        int *line_counter = total + (1 + line) * kCounterStride;
        if (atomicAdd(line_counter, 1) == on_line - 1) {
            *line_counter = 0;
            if (atomicAdd(total + 1, 1) == min(groups, kQueues) - 1) {
                total[1] = 0;
                int *all_counters = static_cast<int *>(a.workspace);
                for (int t = 0; t < H * kQueues; ++t) all_counters[t * kCounterStride] = 0;
                __threadfence();
            }
        }
    }
}

// ---- backward: the pair sweeps ------------------------------------------------------------------------------
// dq, dk, dv of the attention backward (Swin3D/src/attn/self_attn_aio_bwd.cu:197-509 adds every term with a global
// atomic) on the forward's work list: a lane owns one voxel of some window and streams the window's other side,
//   kKeyOwned = false: lane = query i, streams the keys j:    dq_i += dL (k_j + Tq(i,j))
//   kKeyOwned = true:  lane = key j, streams the queries i:   dk_j += dL (q_i + Tk(i,j)),  dv_j += P dout_i
// with P = exp(L - max_i) / sum_i from the forward's saved statistics, dP = dout_i . (v_j + Tv(i,j)) and
// dL = P (dP - dout_i . o_i).  Every gradient row has one owner and is stored once.  The query-owned sweep leaves (dL, P) of
// every (pair, head) at [head][pairs before the window + j n + i], where the lanes of a window write consecutive addresses;
// the key-owned sweep and the table-gradient kernels read them there.
//
// The query-owned sweep is bound by VALU issue, the key-owned one by its records' lines.  199,327 voxels in windows of 26,
// 6 heads of 8, 9 axes, fp16: 338 + 269 us.  When the key-owned sweep made dL and P again (125 of its 280 instructions a pair)
// and left them in a second order for the table gradients, 326 + 374, with a store of 12 bytes a (pair, head) for 8.
template <typename T, int D, int HP> __host__ __device__ constexpr int bwd_pair_threads() { return 256; }
// The sweep that leaves records only: one workgroup of twelve wavefronts a CU, three per SIMD.
constexpr int kRecordThreads = 768, kRecordWaves = 3;
// elements between rows of Tk in the key-owned sweep's LDS (padded as the other's)
template <typename T, int D, int HP> __host__ __device__ constexpr int key_row_stride()
{
    return HP * D + ((HP * D * static_cast<int>(sizeof(T)) / 4) % 8 == 0 ? 16 / static_cast<int>(sizeof(T)) : 0);
}

// TF is the type the feature rows are stored in (q, k, v, dout and the gradients dq, dk, dv); T the type of the
// tables and of the arithmetic.  TF = __half with T = float serves an fp16 forward whose backward runs in fp32: the
// rows are widened as they are loaded and the gradients rounded as they are stored, the arithmetic is that of T = TF
// = float on widened copies.
template <typename T, typename TF, int D, int ND, int HP, bool kKeyOwned, bool kOnlyRecords = false>
// Wavefronts per SIMD, by register cap: fp16 four at head_dim 8, three at 16; fp32 three and two.  The key-owned sweep stays
// below all of them (113 to 167 registers); of the query-owned one nine axes spill 9 (fp16, 16), 1 (fp32, 8), 21 and, beside
// fp16 rows, 13 (fp32, 16).  us of the query-owned and the key-owned sweep with one wavefront more, as it is, one less:
//   head_dim 8, 199,327 voxels in windows of 26, 6 heads: fp16 495 + 383, 336 + 270, 332 + 266 (the cap binds neither);
//     fp32 1440 + 372, 431 + 366, 574 + 370; beside fp16 rows 1203 + 303, 426 + 303, 551 + 302
//   head_dim 16, 49,682 voxels, windows of ten a side, whose tables are too long for strips: fp16 2123 + 939, 939 + 589,
//     953 + 587; fp32 14266 + 1066, 3564 + 1038, 2526 + 1014; beside fp16 rows 12006 + 738, 2864 + 715, 2538 + 714
// (in the last two LDS holds one workgroup a CU, with tables of 432 rows; it holds two below 394, with six axes too, which spill
// nothing).
__global__ __launch_bounds__((kOnlyRecords ? kRecordThreads : bwd_pair_threads<T, D, HP>()), (kOnlyRecords ? kRecordWaves : sizeof(T) == 2 ? (D == 8 ? 4 : 3) : (D == 8 ? 3 : 2))) void attn_bwd_pairs_kernel(BwdPairArgs b)
{
    const AttnArgs &a = b.f;
    constexpr int kThreads = kOnlyRecords ? kRecordThreads : bwd_pair_threads<T, D, HP>();
    constexpr int kSlices = kKeyOwned ? 1 : 3;      // the key-owned sweep needs Tk only
    extern __shared__ __align__(16) float smem[];
    __shared__ __align__(16) int group_exit_counter[4];
    int &group_exited = group_exit_counter[0];
    if (threadIdx.x == 0) group_exited = 0;
    const int H = a.H;
    const int HD = H * D;
    const GroupPlace place(a, H / HP);
    const int hg = place.head_group;
    const int h = hg * HP;
    constexpr int kRowStride = kKeyOwned ? key_row_stride<T, D, HP>() : table_row_stride_heads<T, D, HP>();
    T *tab = reinterpret_cast<T *>(smem);
    {
        const T *gq = static_cast<const T *>(a.table_q);
        const T *gk = static_cast<const T *>(a.table_k);
        const T *gv = static_cast<const T *>(a.table_v);
        constexpr int kPieces = D * static_cast<int>(sizeof(T)) / 16;
        constexpr int kPerPiece = 16 / static_cast<int>(sizeof(T));
        for (int t = threadIdx.x; t < a.total_rows * HP * kPieces; t += kThreads) {
            const int r = t / (HP * kPieces), hp = t - r * (HP * kPieces);
            const int hh = hp / kPieces, c = (hp - hh * kPieces) * kPerPiece;
            const int64_t g = static_cast<int64_t>(r) * HD + (h + hh) * D + c;
            T *row = tab + r * kRowStride + hh * kSlices * D + c;
            if constexpr (kKeyOwned) {
                *reinterpret_cast<uint4 *>(row) = *reinterpret_cast<const uint4 *>(gk + g);
            } else {
                *reinterpret_cast<uint4 *>(row) = *reinterpret_cast<const uint4 *>(gq + g);
                *reinterpret_cast<uint4 *>(row + D) = *reinterpret_cast<const uint4 *>(gk + g);
                *reinterpret_cast<uint4 *>(row + 2 * D) = *reinterpret_cast<const uint4 *>(gv + g);
            }
        }
    }
    __syncthreads();   // the only workgroup barrier

    const int lane = threadIdx.x & 63;
    const TF *gq = static_cast<const TF *>(a.q);
    const TF *gk = static_cast<const TF *>(a.k);
    const TF *gv = static_cast<const TF *>(a.v);
    const TF *ggo = static_cast<const TF *>(b.dout);
    const char *ws = static_cast<const char *>(a.workspace);
    const int4 *unit_info = reinterpret_cast<const int4 *>(ws + ws_units_offset(H));
    const int4 *entries = reinterpret_cast<const int4 *>(ws + ws_entries_offset(H, a.N));
    const int total_units = __builtin_amdgcn_readfirstlane(reinterpret_cast<const int *>(ws + ws_total_offset(H))[0]);
    int *counters = static_cast<int *>(a.workspace) + hg * kQueues * kCounterStride;
    constexpr int kRowBytes = kRowStride * static_cast<int>(sizeof(T));
    constexpr uint32_t kHeadBytes = kSlices * D * sizeof(T);
    const uint32_t tab_addr = __builtin_amdgcn_readfirstlane(lds_address(tab));
    const uint32_t row_bytes = kRowBytes;
    float half_rows[ND], upper[ND];
    uint32_t base_off[ND];
#pragma unroll
    for (int n = 0; n < ND; ++n) {
        half_rows[n] = static_cast<float>(a.rows[n] / 2);
        upper[n] = crse_upper(a.rows[n]);
        base_off[n] = __builtin_amdgcn_readfirstlane(tab_addr + a.base[n] * kRowBytes);
    }
    UnitQueues<kThreads / 64> queues(counters, place, total_units);
    for (;;) {
        const int unit = queues.unit();
        if (unit < 0) break;
        // the unit, as in the forward sweep: 64 >> gshift owned voxels, each on 2^gshift adjacent lanes that take
        // alternate elements of the streamed side
        const int4 info = unit_info[unit];
        const int first = __builtin_amdgcn_readfirstlane(info.x);
        const int gshift = __builtin_amdgcn_readfirstlane(info.y);
        const int owners = __builtin_amdgcn_readfirstlane(info.w);
        const int sub = lane & ((1 << gshift) - 1);
        const bool own_valid = (lane >> gshift) < owners;
        const int slot = __builtin_amdgcn_readfirstlane(info.z) + min(lane >> gshift, owners - 1);
        const int4 seen = entries[first + lane];
        const int seen_from = seen.w == __builtin_amdgcn_readfirstlane(seen.w) ? seen.x : 0x7fffffff;
        int at = 0;
#pragma unroll
        for (int half = 32; half > 0; half >>= 1)
            if (__shfl(seen_from, at + half) <= slot) at += half;
        const int n_w = __shfl(seen.y, at), s0 = __shfl(seen.z, at);
        const int own_in = slot - __shfl(seen.x, at);     // position inside the window
        const int own_pos = s0 + own_in;
        const int own_row = a.n2n[own_pos];
        int max_steps = (n_w + (1 << gshift) - 1) >> gshift;
#pragma unroll
        for (int other = 32; other > 0; other >>= 1) max_steps = max(max_steps, __shfl_xor(max_steps, other));
        max_steps = __builtin_amdgcn_readfirstlane(max_steps);
        // pairs before the window; a window that does not fit the caller's pair store is skipped as a whole
        const int64_t pair_base = b.pos_base[s0];
        const bool fits = pair_base + static_cast<int64_t>(n_w) * n_w <= b.pairs;

        Slice<T, D> own_x[HP], own_y[HP];     // q_i, dout_i
        float own_m[HP], own_inv[HP], own_delta[HP], own_none[HP];
        float ci[ND], res_x[HP][D], res_y[kKeyOwned ? HP : 1][D];
#pragma unroll
        for (int hh = 0; hh < HP; ++hh) {
            const int64_t at_row = static_cast<int64_t>(own_row) * a.row_stride + (h + hh) * D;
            if constexpr (!kKeyOwned) {
                own_x[hh].load(gq + at_row);
                own_y[hh].load(ggo + static_cast<int64_t>(own_row) * HD + (h + hh) * D);
                own_m[hh] = b.stat_max[static_cast<int64_t>(own_row) * H + h + hh];
                own_inv[hh] = 1.0f / b.stat_sum[static_cast<int64_t>(own_row) * H + h + hh];
                if constexpr (!kOnlyRecords) {
                    own_delta[hh] = b.delta[static_cast<int64_t>(own_row) * H + h + hh];
                } else {
                    float x[D], y[D];
                    const int64_t at_out = static_cast<int64_t>(own_row) * HD + (h + hh) * D;
                    load_row<D>(ggo + at_out, x);
                    load_row<D>(static_cast<const TF *>(b.out) + at_out, y);
                    own_delta[hh] = 0.0f;
                    bool some = false;
#pragma unroll
                    for (int c = 0; c < D; ++c) {
                        own_delta[hh] += x[c] * y[c];
                        some = some || fabsf(x[c]) < INFINITY;
                    }
                    own_none[hh] = some ? 0.0f : __int_as_float(0x7fc00000);
                }
            }
#pragma unroll
            for (int c = 0; c < D; ++c) res_x[hh][c] = 0.0f;
            if constexpr (kKeyOwned) {
#pragma unroll
                for (int c = 0; c < D; ++c) res_y[hh][c] = 0.0f;
            }
        }
#pragma unroll
        for (int n = 0; n < ND; ++n) ci[n] = a.n_coords[static_cast<int64_t>(own_pos) * ND + n];

        // Lanes that share an owned voxel take alternate elements of the stream; of keys, runs of it: a lane's records are then
        // one after the other.  It reads four of them at a time, four steps ahead: the lanes' records are n_w apart, and a
        // line fetched for one record would be gone before the next (308 us instead of 269 at the layer below).
        const int run = (n_w + (1 << gshift) - 1) >> gshift;
        auto streamed = [&](int it) { return kKeyOwned ? sub * run + it : (it << gshift) + sub; };
        int row_next = a.n2n[s0 + min(streamed(0), n_w - 1)];
        constexpr int kRecords = kPairSpare;
        typedef float f32x4_2 __attribute__((ext_vector_type(4), aligned(8)));
        float2 rec_now[HP][kRecords], rec_ahead[HP][kRecords];
        auto records = [&](int it, float2 (&into)[HP][kRecords]) {
#pragma unroll
            for (int hh = 0; hh < HP; ++hh) {
                // (behind the last one of a lane lie others, or what the store has spare: they are not used)
                const float2 *from = b.pd + static_cast<int64_t>(h + hh) * b.pairs +
                                     (fits ? pair_base + static_cast<int64_t>(own_in) * n_w + min(streamed(it), n_w - 1) : 0);
#pragma unroll
                for (int e = 0; e < kRecords; e += 2) {
                    const f32x4_2 two = *reinterpret_cast<const f32x4_2 *>(from + e);
                    into[hh][e] = make_float2(two[0], two[1]);
                    into[hh][e + 1] = make_float2(two[2], two[3]);
                }
            }
        };
        if constexpr (kKeyOwned) {
            records(0, rec_now);
            records(kRecords, rec_ahead);
        }
        if constexpr (kOnlyRecords) {
            // As in the forward, the next table rows and the next key are on their way; the same sums in the same order.
            Slice<TF, D> next_k[HP], next_v[HP];
            float cj[ND];
            auto fetch = [&](int it) {
                const int pos = s0 + min(streamed(it), n_w - 1);
                const uint64_t at_row = static_cast<uint64_t>(static_cast<uint32_t>(row_next)) * static_cast<uint64_t>(a.row_stride);
                row_next = a.n2n[s0 + min(streamed(it + 1), n_w - 1)];
#pragma unroll
                for (int n = 0; n < ND; ++n) cj[n] = a.n_coords[static_cast<uint64_t>(static_cast<uint32_t>(pos)) * ND + n];
#pragma unroll
                for (int hh = 0; hh < HP; ++hh) {
                    next_k[hh].load(gk + (at_row + static_cast<uint32_t>((h + hh) * D)));
                    next_v[hh].load(gv + (at_row + static_cast<uint32_t>((h + hh) * D)));
                }
            };
            fetch(0);
            for (int it = 0; it < max_steps; ++it) {
                if (it + 1 >= max_steps) queues.draw();
                const int st = streamed(it);
                const bool valid = st < n_w && own_valid && fits;
                uint32_t off[ND];
#pragma unroll
                for (int n = 0; n < ND; ++n) off[n] = mad_u24(static_cast<uint32_t>(crse_row(ci[n], cj[n], half_rows[n], upper[n])), row_bytes, base_off[n]);
                // rows of the three tables in turn, of all heads
                constexpr int kItems = 3 * ND, kAskAt = 3;
                Slice<T, D> rows[2][HP], key[HP];
                auto read = [&](int i) {
#pragma unroll
                    for (int hh = 0; hh < HP; ++hh) rows[i % 2][hh].load_lds(off[i / 3] + hh * kHeadBytes + (i % 3) * D * sizeof(T));
                };
                read(0);
                __builtin_amdgcn_sched_barrier(0);
                float logit[HP], dp[HP], part[HP];
#pragma unroll
                for (int hh = 0; hh < HP; ++hh) {
                    key[hh].widen(next_k[hh]);
                    Slice<T, D> value;
                    value.widen(next_v[hh]);
                    logit[hh] = own_x[hh].dot(key[hh], 0.0f);
                    dp[hh] = own_y[hh].dot(value, 0.0f);
                }
#pragma unroll
                for (int i = 0; i < kItems; ++i) {
                    if (i + 1 < kItems) read(i + 1);
                    if (i == kAskAt) fetch(it + 1);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int hh = 0; hh < HP; ++hh) {
                        const Slice<T, D> &row = rows[i % 2][hh];
                        constexpr bool kChain = Slice<T, D>::kChainLogit;
                        if (i % 3 == 0) part[hh] = own_x[hh].dot(row, kChain ? logit[hh] : 0.0f);
                        else if (i % 3 == 1) part[hh] = key[hh].dot(row, part[hh]), logit[hh] = kChain ? part[hh] : logit[hh] + part[hh];
                        else if (kChain) dp[hh] = own_y[hh].dot(row, dp[hh]);
                        else dp[hh] += own_y[hh].dot(row, 0.0f);
                    }
                }
                // (or the compiler moves the products below `valid`, away from their rows)
#pragma unroll
                for (int hh = 0; hh < HP; ++hh) asm volatile("" : "+v"(logit[hh]), "+v"(dp[hh]));
#pragma unroll
                for (int hh = 0; hh < HP; ++hh) {
                    // (a logit of minus infinity has no weight, but its dL meets an infinite key or table row in dq; a query
                    // whose dout has no finite channel has no weights either: all channels of what they make are NaN)
                    const int64_t head_at = static_cast<int64_t>(h + hh) * b.pairs + pair_base;
                    const float p = __expf(logit[hh] - own_m[hh]) * own_inv[hh];
                    const float dl = fabsf(logit[hh]) < INFINITY ? p * (dp[hh] - own_delta[hh]) : __int_as_float(0x7fc00000);
                    if (valid) b.pd[head_at + static_cast<int64_t>(min(st, n_w - 1)) * n_w + own_in] = make_float2(dl, p + own_none[hh]);
                }
            }
        } else {
            for (int it = 0; it < max_steps; ++it) {
                if (it + 1 >= max_steps) queues.draw();
                const int st = streamed(it);
                const bool valid = st < n_w && (!kKeyOwned || it < run) && own_valid && fits;
                const int st_in = min(st, n_w - 1);
                const int st_pos = s0 + st_in;
                const int st_row = row_next;
                row_next = a.n2n[s0 + min(streamed(it + 1), n_w - 1)];
                Slice<T, D> st_x[HP], st_y[HP];   // k_j, v_j  or  q_i, dout_i
#pragma unroll
                for (int hh = 0; hh < HP; ++hh) {
                    const int64_t at_row = static_cast<int64_t>(st_row) * a.row_stride + (h + hh) * D;
                    const int64_t at_grad = static_cast<int64_t>(st_row) * HD + (h + hh) * D;
                    if constexpr (kKeyOwned) {
                        st_x[hh].load(gq + at_row);
                        st_y[hh].load(ggo + at_grad);
                    } else {
                        st_x[hh].load(gk + at_row);
                        st_y[hh].load(gv + at_row);
                    }
                }
                float2 rec[HP];
                if constexpr (kKeyOwned) {
#pragma unroll
                    for (int hh = 0; hh < HP; ++hh) {
                        rec[hh] = rec_now[hh][0];
#pragma unroll
                        for (int e = 0; e + 1 < kRecords; ++e) rec_now[hh][e] = rec_now[hh][e + 1];
                    }
                    if (it % kRecords == kRecords - 1) {
#pragma unroll
                        for (int hh = 0; hh < HP; ++hh)
#pragma unroll
                            for (int e = 0; e < kRecords; ++e) rec_now[hh][e] = rec_ahead[hh][e];
                        records(it + 1 + kRecords, rec_ahead);
                    }
                }
                uint32_t off[ND];
                {
                    float cj[ND];
#pragma unroll
                    for (int n = 0; n < ND; ++n) cj[n] = a.n_coords[static_cast<int64_t>(st_pos) * ND + n];
#pragma unroll
                    for (int n = 0; n < ND; ++n) {
                        // row_n(i, j): the query's coordinate first
                        const float c_i = kKeyOwned ? cj[n] : ci[n], c_j = kKeyOwned ? ci[n] : cj[n];
                        off[n] = mad_u24(static_cast<uint32_t>(crse_row(c_i, c_j, half_rows[n], upper[n])), row_bytes, base_off[n]);
                    }
                }
#pragma unroll
                for (int hh = 0; hh < HP; ++hh) {
                    const int64_t head_at = static_cast<int64_t>(h + hh) * b.pairs + pair_base;
                    float logit = 0.0f, dp = 0.0f;
                    if constexpr (!kKeyOwned) {
                        logit = own_x[hh].dot(st_x[hh], 0.0f);
                        dp = own_y[hh].dot(st_y[hh], 0.0f);
                    }
                    // sums of three rows of the table that enters the owned gradient as a vector (packed fp16 adds for
                    // fp16 I/O, as the forward adds its value-table rows)
                    // (fp32: one sum of all rows - plain adds, no packing to gain, and two sums fewer to hold)
                    constexpr int kGroup = sizeof(T) == 4 ? ND : 3;
                    Slice<T, D> vec_sum[(ND + kGroup - 1) / kGroup];
#pragma unroll
                    for (int n = 0; n < ND; ++n) {
                        Slice<T, D> vec_r;       // Tk, or Tq
                        vec_r.load_lds(off[n] + hh * kHeadBytes);
                        if constexpr (!kKeyOwned) {
                            Slice<T, D> tk_r, tv_r;
                            tk_r.load_lds(off[n] + hh * kHeadBytes + D * sizeof(T));
                            tv_r.load_lds(off[n] + hh * kHeadBytes + 2 * D * sizeof(T));
                            if (Slice<T, D>::kChainLogit) logit = st_x[hh].dot(tk_r, own_x[hh].dot(vec_r, logit));
                            else logit += st_x[hh].dot(tk_r, own_x[hh].dot(vec_r, 0.0f));
                            if (Slice<T, D>::kChainLogit) dp = own_y[hh].dot(tv_r, dp);
                            else dp += own_y[hh].dot(tv_r, 0.0f);
                        }
                        if (n % kGroup == 0) vec_sum[n / kGroup] = vec_r;
                        else vec_sum[n / kGroup].add(vec_r);
                    }
                    float p, dl;
                    if constexpr (kKeyOwned) {
                        p = valid ? rec[hh].y : 0.0f;
                        dl = valid ? rec[hh].x : 0.0f;
                    } else {
                        p = valid ? __expf(logit - own_m[hh]) * own_inv[hh] : 0.0f;
                        dl = p * (dp - own_delta[hh]);
                    }
                    // dq_i += dL (k_j + Tq)   or   dk_j += dL (q_i + Tk)
                    st_x[hh].fma_to(res_x[hh], dl);
#pragma unroll
                    for (int g = 0; g < (ND + kGroup - 1) / kGroup; ++g) vec_sum[g].fma_to(res_x[hh], dl);
                    if constexpr (kKeyOwned) st_y[hh].fma_to(res_y[hh], p);     // dv_j += P dout_i
                    if constexpr (!kKeyOwned) {
                        if (valid) b.pd[head_at + static_cast<int64_t>(st_in) * n_w + own_in] = make_float2(dl, p);
                    }
                }
            }
#pragma unroll
            for (int hh = 0; hh < HP; ++hh) {
                // lanes that share an owned voxel saw alternate elements of the stream
                for (int other = 1; other < (1 << gshift); other <<= 1) {
#pragma unroll
                    for (int c = 0; c < D; ++c) res_x[hh][c] += __shfl_xor(res_x[hh][c], other);
                    if constexpr (kKeyOwned) {
#pragma unroll
                        for (int c = 0; c < D; ++c) res_y[hh][c] += __shfl_xor(res_y[hh][c], other);
                    }
                }
                if (own_valid && sub == 0) {
                    // a window beyond the caller's pair store was skipped: its rows say so
                    if (!fits) {
#pragma unroll
                        for (int c = 0; c < D; ++c) res_x[hh][c] = __int_as_float(0x7fc00000);
                        if constexpr (kKeyOwned) {
#pragma unroll
                            for (int c = 0; c < D; ++c) res_y[hh][c] = __int_as_float(0x7fc00000);
                        }
                    }
                    const int64_t at_row = static_cast<int64_t>(own_row) * b.grad_stride + (h + hh) * D;
                    if constexpr (kKeyOwned) {
                        store_row<D>(static_cast<TF *>(b.dk) + at_row, res_x[hh]);
                        store_row<D>(static_cast<TF *>(b.dv) + at_row, res_y[hh]);
                    } else {
                        store_row<D>(static_cast<TF *>(b.dq) + at_row, res_x[hh]);
                    }
                }
            }
        }
    }
    // the last wavefront of the launch to leave puts the queue counters back to zero (as in the forward sweep):
    // the next sweep runs on the same list
    if (lane == 0 && atomicAdd(&group_exited, 1) == kThreads / 64 - 1) {
        __threadfence();
        int *total = static_cast<int *>(a.workspace) + ws_total_offset(H) / sizeof(int);
        const int groups = static_cast<int>(gridDim.x), line = static_cast<int>(blockIdx.x) % kQueues;
        const int on_line = (groups - line + kQueues - 1) / kQueues;
        int *line_counter = total + (1 + line) * kCounterStride;
        if (atomicAdd(line_counter, 1) == on_line - 1) {
            *line_counter = 0;
            if (atomicAdd(total + 1, 1) == min(groups, kQueues) - 1) {
                total[1] = 0;
                int *all_counters = static_cast<int *>(a.workspace);
                for (int t = 0; t < H * kQueues; ++t) all_counters[t * kCounterStride] = 0;
                __threadfence();
            }
        }
    }
}

template <typename T, int D, int ND, int HP, bool kSorted>
int launch_sweep_heads(const AttnArgs &a, hipStream_t stream, int what)
{
    const size_t lds = align_up(sizeof(T) * static_cast<size_t>(a.total_rows) * table_row_stride_heads<T, D, HP>(), 16);
    if (lds > 160 * 1024)
        return fail(S3D_ERR_UNSUPPORTED, "s3d_attn_fwd: %d table rows x D=%d need %zu B of LDS (> 160 KiB)",
                    a.total_rows, D, lds);
    auto kernel = attn_fwd_sweep_kernel<T, D, ND, HP, kSorted>;
    if (int rc = allow_dynamic_lds(reinterpret_cast<const void *>(kernel), lds)) return rc;
    // A workgroup serves one head group for its whole life: as many workgroups per CU as registers and LDS allow.
    int per_cu = groups_per_cu<T, D>();
    while (per_cu > 1 && per_cu * lds > 160 * 1024) --per_cu;
    AttnArgs b = a;
    constexpr int kThreads = group_threads<T, D>();
    const int grid = place_groups(b, per_cu * device_cus(), a.H / HP, kThreads);
    if constexpr (D == 8 && HP < 3) {
        // The list is cut as for sixteen wavefronts a CU: chains of additions no longer than four workgroups of four (in fp32 two of eight)
        // had them.  Cut for twelve, 60,001 voxels x 10 heads in fp32 were 2.55e-7 from 64 bits for 2.51e-7, in 145.1 us for 146.7; fp16
        // 100,003 x 10 196.5 for 200.5, 595,677 x 10 879 for 884.
        constexpr int kWaves = sizeof(T) == 4 && HP == 2 ? 8 : 4;
        int held = 16 / kWaves;
        while (held > 1 && held * lds > 160 * 1024) --held;
        AttnArgs cut = a;
        place_groups(cut, held * device_cus(), a.H / HP, 64 * kWaves);
        b.target_items = cut.target_items;
    }
    b.block_shift = target_shift_for(a.N, a.W, b.target_items);
    if (what & kAttnBuildList) {
        launch_work_list(b, stream, what & kAttnStripList);
        S3D_HIP_CHECK(hipGetLastError());
    }
    if (what & kAttnSweep) {
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(kThreads), lds, stream, b);
        S3D_HIP_CHECK(hipGetLastError());
    }
    return S3D_OK;
}

template <typename T, int D, int ND>
int launch_sweep(const AttnArgs &a, hipStream_t stream, int what)
{
    // Two heads per wavefront where the registers allow it (fp16) and the heads pair up: the cRSE rows and LDS
    // addresses of a pair are spent once for both.  At head_dim 16 that means one workgroup of twelve wavefronts per
    // CU (75 KB of tables): it measured -10 % at 6 heads.
    if constexpr (sizeof(T) == 2 && D <= 16) {
        // three heads where they go in threes and fit (head_dim 8: 168 registers, one workgroup with 45 KB of
        // tables per CU): -2 % against pairs at 6 and 12 heads
        if constexpr (D == 8) {
            if (a.H % 3 == 0)
                return a.n2n ? launch_sweep_heads<T, D, ND, 3, false>(a, stream, what)
                             : launch_sweep_heads<T, D, ND, 3, true>(a, stream, what);
        }
        if (a.H % 2 == 0)
            return a.n2n ? launch_sweep_heads<T, D, ND, 2, false>(a, stream, what)
                         : launch_sweep_heads<T, D, ND, 2, true>(a, stream, what);
    }
    // fp32 at head_dim 8: pairs of heads as well
    if constexpr (sizeof(T) == 4 && D == 8) {
        if (a.H % 2 == 0)
            return a.n2n ? launch_sweep_heads<T, D, ND, 2, false>(a, stream, what)
                         : launch_sweep_heads<T, D, ND, 2, true>(a, stream, what);
    }
    return a.n2n ? launch_sweep_heads<T, D, ND, 1, false>(a, stream, what)
                 : launch_sweep_heads<T, D, ND, 1, true>(a, stream, what);
}

template <typename T>
int dispatch_shape(const AttnArgs &a, hipStream_t stream, int what)
{
#define S3D_CASE(DD, NN) \
    if (a.D == DD && a.nd == NN) return launch_sweep<T, DD, NN>(a, stream, what);
    S3D_CASE(8, 3) S3D_CASE(8, 6) S3D_CASE(8, 9)
    S3D_CASE(16, 3) S3D_CASE(16, 6) S3D_CASE(16, 9)
    S3D_CASE(32, 3) S3D_CASE(32, 6) S3D_CASE(32, 9)
#undef S3D_CASE
    return fail(S3D_ERR_UNSUPPORTED, "s3d_attn_fwd: unsupported head_dim %d / cRSE axes %d "
                "(head_dim in {8,16,32}, axes in {3,6,9})", a.D, a.nd);
}

}  // namespace

namespace {

template <typename T, typename TF, int D, int ND>
int launch_bwd_pairs(const BwdPairArgs &b0, hipStream_t stream)
{
    // one head per wavefront: with two (fp16, head_dim 8) the pair of sweeps measured 0.3 ms slower at the 6-head layer
    constexpr int HP = 1;
    const AttnArgs &a = b0.f;
    // the query-owned sweep keeps a head's slices of the three tables, the key-owned one those of Tk
    const size_t q_lds = align_up(sizeof(T) * static_cast<size_t>(a.total_rows) * table_row_stride_heads<T, D, HP>(), 16);
    const size_t k_lds = align_up(sizeof(T) * static_cast<size_t>(a.total_rows) * key_row_stride<T, D, HP>(), 16);
    if (q_lds > 160 * 1024)
        return fail(S3D_ERR_UNSUPPORTED, "s3d_attn_bwd: %d table rows x D=%d need %zu B of LDS (> 160 KiB)",
                    a.total_rows, D, q_lds);
    auto q_sweep = attn_bwd_pairs_kernel<T, TF, D, ND, HP, false>;
    auto k_sweep = attn_bwd_pairs_kernel<T, TF, D, ND, HP, true>;
    constexpr int kThreads = bwd_pair_threads<T, D, HP>();
    if (int rc = allow_dynamic_lds(reinterpret_cast<const void *>(q_sweep), q_lds)) return rc;
    if (int rc = allow_dynamic_lds(reinterpret_cast<const void *>(k_sweep), k_lds)) return rc;
    const int groups = a.H / HP;
    // workgroups: as many as registers and the tables in LDS allow, the query-owned sweep's placed as the forward's, the key-owned
    // one's in whole sets
    auto with_grid = [&](BwdPairArgs &b, const void *kernel, size_t lds, int &grid, bool whole_sets) {
        int per_cu = 0;
        S3D_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kThreads, lds));
        if (per_cu < 1) per_cu = 1;
        grid = place_groups(b.f, per_cu * device_cus(), groups, kThreads, whole_sets);
        return static_cast<int>(S3D_OK);
    };
    BwdPairArgs b = b0, by_key = b0;
    int grid = 0, key_grid = 0;
    if (int rc = with_grid(b, reinterpret_cast<const void *>(q_sweep), q_lds, grid, false)) return rc;
    if (int rc = with_grid(by_key, reinterpret_cast<const void *>(k_sweep), k_lds, key_grid, true)) return rc;
    // (one work list, cut for the query-owned sweep, which takes longer)
    b.f.block_shift = target_shift_for(a.N, a.W, b.f.target_items);
    launch_work_list(b.f, stream);
    S3D_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(q_sweep, dim3(static_cast<unsigned>(grid)), dim3(kThreads), q_lds, stream, b);
    hipLaunchKernelGGL(k_sweep, dim3(static_cast<unsigned>(key_grid)), dim3(kThreads), k_lds, stream, by_key);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

template <typename T, typename TF, int ND, int HP>
int launch_bwd_records(const BwdPairArgs &b0, const tile::StripSetup &strips, hipStream_t stream)
{
    constexpr int D = 8;
    const AttnArgs &a = b0.f;
    const size_t lds = align_up(sizeof(T) * static_cast<size_t>(a.total_rows) * table_row_stride_heads<T, D, HP>(), 16);
    auto kernel = attn_bwd_pairs_kernel<T, TF, D, ND, HP, false, true>;
    constexpr int kThreads = kRecordThreads;
    if (int rc = allow_dynamic_lds(reinterpret_cast<const void *>(kernel), lds)) return rc;
    int per_cu = 0;
    S3D_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void *>(kernel), kThreads, lds));
    if (per_cu < 1) per_cu = 1;
    BwdPairArgs b = b0;
    const int grid = place_groups(b.f, per_cu * device_cus(), a.H / HP, kThreads);
    b.f.block_shift = target_shift_for(a.N, a.W, b.f.target_items);
    if (int rc = launch_records_lists(strips, b.f, sizeof(T) != sizeof(TF), stream)) return rc;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(kThreads), lds, stream, b);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

// Records alone, for the strips of attn_strip_bwd.hip (head_dim 8).  Bound by VALU issue, some 320 instructions a step of two
// heads.  A call, forward included, us: 199,327 voxels in windows of 26, 6 heads, 9 axes, fp16 1475 with pairs of heads, 1465 with
// three (6 axes, 60,001 voxels, 467 and 469.5); beside fp16 rows 1570, fp32 tables.  As one workgroup of 256 for each wavefront of a
// SIMD 1482 and 1604, of 384 1551 and 1684; before rows and keys were read ahead, 1520 and 1700.  fp32, one head / two, 9 axes 40,001 x
// 6 560 / 602, 20,001 x 6 338 / 385, windows of 57 60,001 x 10 1930 / 2079; 6 axes (two spill two registers) 485 / 473, 290 / 297,
// 1633 / 1571; 3 axes 20,001 x 6 266 / 265, windows of 57 60,001 x 10 1368 / 1331.
template <typename T, typename TF, int ND>
int dispatch_bwd_records(const BwdPairArgs &b, const tile::StripSetup &strips, hipStream_t stream)
{
    if constexpr (sizeof(T) == 2 && ND == 9) {
        if (b.f.H % 3 == 0) return launch_bwd_records<T, TF, ND, 3>(b, strips, stream);
    }
    if constexpr (sizeof(TF) == 2 || ND < 9) {
        if (b.f.H % 2 == 0) return launch_bwd_records<T, TF, ND, 2>(b, strips, stream);
    }
    return launch_bwd_records<T, TF, ND, 1>(b, strips, stream);
}

template <typename T, typename TF>
int dispatch_bwd_pairs(const BwdPairArgs &b, hipStream_t stream)
{
#define S3D_CASE(DD, NN) \
    if (b.f.D == DD && b.f.nd == NN) return launch_bwd_pairs<T, TF, DD, NN>(b, stream);
    S3D_CASE(8, 3) S3D_CASE(8, 6) S3D_CASE(8, 9)
    S3D_CASE(16, 3) S3D_CASE(16, 6) S3D_CASE(16, 9)
#undef S3D_CASE
    return fail(S3D_ERR_UNSUPPORTED, "s3d_attn_bwd: unsupported head_dim %d / cRSE axes %d", b.f.D, b.f.nd);
}

}  // namespace

int launch_attn_bwd_pairs(const BwdPairArgs &b, int dtype, hipStream_t stream)
{
    switch (dtype) {
    case S3D_DTYPE_F32: return dispatch_bwd_pairs<float, float>(b, stream);
    case S3D_DTYPE_F16: return dispatch_bwd_pairs<__half, __half>(b, stream);
    case S3D_DTYPE_F32_F16_ROWS: return dispatch_bwd_pairs<float, __half>(b, stream);
    default: return fail(S3D_ERR_BAD_DTYPE, "s3d_attn_bwd: dtype %d (0 = fp32, 1 = fp16, 2 = fp32 on fp16 rows)", dtype);
    }
}

int launch_attn_bwd_records(const BwdPairArgs &b, const tile::StripSetup &strips, int dtype, hipStream_t stream)
{
#define S3D_CASE(NN)                                                                                       \
    if (b.f.D == 8 && b.f.nd == NN)                                                                        \
        return dtype == S3D_DTYPE_F32   ? dispatch_bwd_records<float, float, NN>(b, strips, stream)                \
               : dtype == S3D_DTYPE_F16 ? dispatch_bwd_records<__half, __half, NN>(b, strips, stream)              \
                                        : dispatch_bwd_records<float, __half, NN>(b, strips, stream);
    S3D_CASE(3) S3D_CASE(6) S3D_CASE(9)
#undef S3D_CASE
    return fail(S3D_ERR_UNSUPPORTED, "s3d_attn_bwd: head_dim %d, %d axes in the records sweep", b.f.D, b.f.nd);
}

size_t attn_sweep_workspace_bytes(int H, int64_t W, int64_t N)
{
    // queue counters, the totals, one record per unit, the sorted window list and the list builder's notes
    return ws_end_offset(H, W, N);
}

void *attn_sweep_notes(const AttnArgs &a)
{
    static_assert(sizeof(unsigned long long) * kListGroups * (kListThreads / 64 + 1) * kBins == kSweepNotesBytes, "the bins");
    // (one workgroup: its wavefronts' bins in front, and its own behind all that 32 would have)
    static_assert(sizeof(unsigned long long) * (kListThreads / 64) * kBins <= kSweepNotesKept, "the bins of one workgroup");
    return static_cast<char *>(a.workspace) + ws_bins_offset(a.H, a.W, a.N);
}

int launch_attn_sweep(const AttnArgs &a, int dtype, hipStream_t stream, int what)
{
    switch (dtype) {
    case S3D_DTYPE_F32: return dispatch_shape<float>(a, stream, what);
    case S3D_DTYPE_F16: return dispatch_shape<__half>(a, stream, what);
    default: return fail(S3D_ERR_BAD_DTYPE, "s3d_attn_fwd: dtype %d (0 = fp32, 1 = fp16)", dtype);
    }
}

}  // namespace s3d
