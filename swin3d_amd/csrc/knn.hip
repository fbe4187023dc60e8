// Grid-bucketed exact K nearest neighbours inside batch segments (gfx950).
//
// Replaces the brute-force kernel of Swin3D/src/knn/knn_cuda_kernel.cu:139-204
// (one thread streaming every source of the batch through a 64-slot heap).
// Sources are bucketed into a uniform grid (one counting sort); a small group of
// lanes per query walks cubic shells of cells around the query's cell and keeps
// the K best candidates, ordered by (squared distance, source row).  A shell
// walk stops once the K-th best distance is provably smaller than the distance
// to anything outside the visited cube, so the result is exact and independent
// of the visiting order: ties go to the lower source row.
//
// Distance arithmetic: d = src - query per axis, ((dx*dx) + (dy*dy)) + (dz*dz),
// every operation individually rounded to fp32 (no fused multiply-add).
#include "attn_kernels.h"

#include <type_traits>

namespace s3d {
namespace {

constexpr int kThreads = 256;
constexpr int kMaxBatch = 4096;
constexpr int kBboxBlocks = 128;   // workgroups of the bounding-box pass = partial boxes the count pass reduces

struct KnnPlan {
    // bounding box of all sources as order-preserving integer images of the floats
    int lo[3], hi[3];
    float origin[3];
    float cell, inv_cell, slack;
    int dim[3];
    int pitch;            // dim[0] + 1: an x-row of cells has one more in memory, whose start is the row's end
    int cells_per_batch;  // in memory: pitch dim[1] dim[2]
    int src_end;  // sources at or beyond this row belong to no batch segment
};

struct Layout {
    size_t plan, partials, counts, starts, src_place, sorted, total;
    int64_t cells_cap;
};

int64_t cells_cap_for(int64_t Ns)
{
    int64_t cap = 4 * Ns;
    if (cap < 2 * kMaxBatch) cap = 2 * kMaxBatch;      // (a batch segment takes two at least: one cell and the row's end)
    if (cap > (1LL << 24)) cap = 1LL << 24;
    return cap;
}

Layout make_layout(int64_t Ns)
{
    Layout L{};
    L.cells_cap = cells_cap_for(Ns);
    const size_t ns = static_cast<size_t>(Ns > 0 ? Ns : 1);
    const size_t cells = static_cast<size_t>(L.cells_cap);
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t at = off;
        off = align_up(off + bytes, 256);
        return at;
    };
    L.plan = take(sizeof(KnnPlan));
    L.partials = take(sizeof(int32_t) * (6 * kBboxBlocks + 1));      // ... and how many sources have a place
    L.counts = take(cells * sizeof(int32_t));
    L.starts = take(cells * sizeof(int32_t));
    L.src_place = take(ns * sizeof(int2));
    L.sorted = take(ns * sizeof(float4));
    L.total = off;
    return L;
}

// order-preserving map float -> int (so integer atomicMin/Max work on floats)
__device__ __forceinline__ int float_to_ordered(float f)
{
    const int i = __float_as_int(f);
    return i >= 0 ? i : i ^ 0x7fffffff;
}
__device__ __forceinline__ float ordered_to_float(int i)
{
    return __int_as_float(i >= 0 ? i : i ^ 0x7fffffff);
}

// Bounding box of the sources, one partial box per workgroup (no atomics, nothing to initialise), and the cell
// counters set to zero: a small grid-stride grid.
__global__ __launch_bounds__(kThreads) void knn_bbox_kernel(const float *__restrict__ src, int64_t stride, int64_t Ns,
                                                            int32_t *__restrict__ partials,
                                                            int32_t *__restrict__ counts, int64_t cells)
{
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; i < cells;
         i += static_cast<int64_t>(gridDim.x) * kThreads)
        counts[i] = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) partials[6 * kBboxBlocks] = 0;
    int lo[3] = {0x7fffffff, 0x7fffffff, 0x7fffffff};
    int hi[3] = {static_cast<int>(0x80000000u), static_cast<int>(0x80000000u),
                 static_cast<int>(0x80000000u)};
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; i < Ns;
         i += static_cast<int64_t>(gridDim.x) * kThreads) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const int o = float_to_ordered(src[i * stride + a]);
            lo[a] = min(lo[a], o);
            hi[a] = max(hi[a], o);
        }
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        for (int off = 32; off > 0; off >>= 1) {
            lo[a] = min(lo[a], __shfl_down(lo[a], off));
            hi[a] = max(hi[a], __shfl_down(hi[a], off));
        }
    }
    __shared__ int part[kThreads / 64][6];
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            part[threadIdx.x >> 6][a] = lo[a];
            part[threadIdx.x >> 6][3 + a] = hi[a];
        }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        int v = part[0][threadIdx.x];
        for (int w = 1; w < kThreads / 64; ++w)
            v = threadIdx.x < 3 ? min(v, part[w][threadIdx.x]) : max(v, part[w][threadIdx.x]);
        partials[blockIdx.x * 6 + threadIdx.x] = v;
    }
}

// One wavefront: turn the bounding box (plan->lo / hi) into grid parameters that fit `cells_cap`.  Every workgroup makes the
// same of it.
__device__ void make_plan(KnnPlan *plan, const int32_t *__restrict__ src_offset, int B, int64_t Ns, int K,
                          float cell_hint, int64_t cells_cap)
{
    const int lane = threadIdx.x & 63;
    int src_end = src_offset[B - 1];
    if (src_end > Ns) src_end = static_cast<int>(Ns);
    if (src_end < 0) src_end = 0;
    if (src_end == 0) {  // no candidate anywhere: the query kernel pads every slot
        if (lane == 0) {
            for (int a = 0; a < 3; ++a) {
                plan->origin[a] = 0.0f;
                plan->dim[a] = 1;
            }
            plan->cell = plan->inv_cell = 1.0f;
            plan->slack = 0.0f;
            plan->pitch = plan->cells_per_batch = 2;
            plan->src_end = 0;
        }
        return;
    }
    float ext[3], max_abs = 0.0f;
    for (int a = 0; a < 3; ++a) {
        const float lo = ordered_to_float(plan->lo[a]);
        const float hi = ordered_to_float(plan->hi[a]);
        ext[a] = fmaxf(hi - lo, 0.0f);
        max_abs = fmaxf(max_abs, fmaxf(fabsf(lo), fabsf(hi)));
    }
    const int64_t per_batch_cap = cells_cap / B;  // B <= kMaxBatch <= cells_cap / 2
    float cell = cell_hint;
    if (!(cell > 0.0f)) {
        // no hint: about K / 32 sources per cell if the sources filled their box (scans of surfaces fill a small part
        // of the box, so the occupied cells hold more and most cells of a shell are empty, which the query kernel
        // skips cheaply; measured at K = 16 on a room scan, 200k sources, 50k queries: divisor 8, 16, 24, 32, 48, 64
        // -> 0.109, 0.113, 0.107, 0.106, 0.105, 0.111 ms per call), and never more cells than the cell array has
        const float floor_ext = fmaxf(fmaxf(ext[0], ext[1]), ext[2]) * 1e-3f + 1e-12f;
        const float vol = fmaxf(ext[0], floor_ext) * fmaxf(ext[1], floor_ext) * fmaxf(ext[2], floor_ext);
        cell = cbrtf(vol / static_cast<float>(src_end > 0 ? src_end : 1) * static_cast<float>(K) * (1.0f / 32.0f));
        cell = fmaxf(cell, cbrtf(vol / static_cast<float>(per_batch_cap > 0 ? per_batch_cap : 1)));
    }
    if (!(cell > 1e-20f)) cell = 1.0f;
    // the first that fits of a ladder of cell edges (forty steps of 3 %, then of 25 %), a lane each: 64 at a time
    int dim[3];
    bool fits = false;
    for (int first = 0; first < 448 && !fits; first += 64) {
        const int step = first + lane;
        const float edge = cell * exp2f(static_cast<float>(min(step, 40)) * 0.04264434f + static_cast<float>(max(step - 40, 0)) * 0.32192809f);
        double total = 1.0;
        int d[3];
        for (int a = 0; a < 3; ++a) {
            const float cells_f = floorf(ext[a] / edge) + 1.0f;
            d[a] = cells_f < 2.0e9f ? static_cast<int>(cells_f) : 2000000000;
            total *= static_cast<double>(d[a]) + (a == 0 ? 1.0 : 0.0);
        }
        const unsigned long long good = __ballot(total <= static_cast<double>(per_batch_cap));
        if (good) {
            const int which = __ffsll(static_cast<long long>(good)) - 1;
            for (int a = 0; a < 3; ++a) dim[a] = __shfl(d[a], which);
            cell = __shfl(edge, which);
            fits = true;
        }
    }
    if (!fits) {  // degenerate input: single cell
        dim[0] = dim[1] = dim[2] = 1;
        cell = fmaxf(fmaxf(ext[0], ext[1]), ext[2]) * 2.0f + 1.0f;
    }
    if (lane != 0) return;
    plan->src_end = src_end;
    plan->cell = cell;
    plan->inv_cell = 1.0f / cell;
    // sources within `slack` of a cell face may sit in either neighbour cell
    plan->slack = 1e-3f * cell + 8e-6f * max_abs;
    for (int a = 0; a < 3; ++a) {
        plan->origin[a] = ordered_to_float(plan->lo[a]);
        plan->dim[a] = dim[a];
    }
    plan->pitch = dim[0] + 1;
    plan->cells_per_batch = (dim[0] + 1) * dim[1] * dim[2];
}

// the plan of a call without sources (the query kernel pads every slot)
__global__ void knn_plan_kernel(KnnPlan *plan, const int32_t *__restrict__ src_offset, int B,
                                int64_t Ns, int K, float cell_hint, int64_t cells_cap)
{
    if (threadIdx.x >= 64 || blockIdx.x != 0) return;
    make_plan(plan, src_offset, B, Ns, K, cell_hint, cells_cap);
}

__device__ __forceinline__ int cell_coord(float p, float origin, float inv_cell)
{
    const float t = floorf((p - origin) * inv_cell);
    // keep the conversion defined for far-away queries
    return static_cast<int>(fminf(fmaxf(t, -1.0e9f), 1.0e9f));
}

__device__ __forceinline__ int find_batch(const int32_t *__restrict__ offset, int B, int64_t g)
{
    int b = 0;
    for (; b < B; ++b)
        if (g < offset[b]) break;
    return b;  // == B: beyond the last segment
}

__device__ __forceinline__ int cell_of(const KnnPlan &plan, const float *p, int b)
{
    int c[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        c[a] = cell_coord(p[a], plan.origin[a], plan.inv_cell);
        c[a] = min(max(c[a], 0), plan.dim[a] - 1);
    }
    return b * plan.cells_per_batch + (c[2] * plan.dim[1] + c[1]) * plan.pitch + c[0];
}

// reduce a box of order-preserving integers (lower corner, upper corner) over the workgroup into `box`
template <int kWaves> __device__ __forceinline__ void reduce_box(int *v, int (*part)[6], int *box)
{
#pragma unroll
    for (int a = 0; a < 6; ++a)
        for (int off = 32; off > 0; off >>= 1) {
            const int o = __shfl_down(v[a], off);
            v[a] = a < 3 ? min(v[a], o) : max(v[a], o);
        }
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int a = 0; a < 6; ++a) part[threadIdx.x >> 6][a] = v[a];
    __syncthreads();
    if (threadIdx.x < 6) {
        int r = part[0][threadIdx.x];
        for (int w = 1; w < kWaves; ++w)
            r = threadIdx.x < 3 ? min(r, part[w][threadIdx.x]) : max(r, part[w][threadIdx.x]);
        box[threadIdx.x] = r;
    }
    __syncthreads();
}

// Every workgroup first reduces the partial boxes and derives the grid from them (the same arithmetic in every
// workgroup; workgroup 0 leaves the plan for the kernels that follow), then its sources take their places: a
// source's cell and its slot there, drawn from the cell's counter.  Neighbouring lanes that fall into the same
// cell (sources usually arrive in lattice order) draw one run of slots with one atomic.
__global__ __launch_bounds__(kThreads) void knn_count_kernel(
    const float *__restrict__ src, int64_t stride, int64_t Ns, const int32_t *__restrict__ src_offset, int B,
    const int32_t *__restrict__ partials, int boxes, int K, float cell_hint, int64_t cells_cap,
    KnnPlan *__restrict__ plan_out,
    int32_t *__restrict__ counts, int2 *__restrict__ src_place)
{
    __shared__ KnnPlan plan;
    __shared__ int part[kThreads / 64][6];
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    float own[3] = {0.0f, 0.0f, 0.0f};
    if (i < Ns)
#pragma unroll
        for (int a = 0; a < 3; ++a) own[a] = src[i * stride + a];
    {
        int v[6];
#pragma unroll
        for (int a = 0; a < 6; ++a) v[a] = a < 3 ? 0x7fffffff : static_cast<int>(0x80000000u);
        for (int t = threadIdx.x; t < boxes; t += kThreads)
#pragma unroll
            for (int a = 0; a < 6; ++a) v[a] = a < 3 ? min(v[a], partials[t * 6 + a]) : max(v[a], partials[t * 6 + a]);
        reduce_box<kThreads / 64>(v, part, plan.lo);      // (lo and hi lie side by side)
        if (threadIdx.x < 64) {
            make_plan(&plan, src_offset, B, Ns, K, cell_hint, cells_cap);
            if (blockIdx.x == 0 && threadIdx.x == 0) *plan_out = plan;
        }
        __syncthreads();
    }
    const int lane = threadIdx.x & 63;
    int cell = -2;                       // beyond the array
    if (i < Ns) {
        const int b = find_batch(src_offset, B, i);
        cell = b < B ? cell_of(plan, own, b) : -1;      // (-1: in no batch segment)
    }
    // runs of equal cells along the lanes: the first lane of a run draws the run's slots
    const int before = __shfl_up(cell, 1);
    const bool head = lane == 0 || before != cell;
    const unsigned long long heads = __ballot(head);
    const unsigned long long upto = heads & (lane == 63 ? ~0ull : ((2ull << lane) - 1));
    const int my_head = 63 - __clzll(static_cast<long long>(upto));
    const unsigned long long above = lane == 63 ? 0ull : heads & ~((2ull << lane) - 1);
    const int next = above ? __ffsll(static_cast<long long>(above)) - 1 : 64;
    int base = 0;
    if (head && cell >= 0) base = atomicAdd(&counts[cell], next - lane);
    base = __shfl(base, my_head);
    if (i < Ns) src_place[i] = make_int2(cell, base + (lane - my_head));
}

// inclusive sum over the lanes of a wavefront, by DPP moves
__device__ __forceinline__ int wave_scan(int x)
{
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);      // row_shr 1, 2, 4, 8
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, true);      // row_bcast15 into rows 1, 3
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, true);      // row_bcast31 into rows 2, 3
    return x;
}

// Where every cell's sources start.  The sources of an x-row of cells lie one after the other (a query reads runs of cells),
// the rows in any order: a workgroup takes whole rows, adds their counts up and draws the room for them with one atomic.
// (One launch and no state to prepare, where a scan over all cells took two: 10.5 -> 6 us for 199,327 sources.)
constexpr int kStartThreads = 1024, kStartCells = 4 * kStartThreads;
__global__ __launch_bounds__(kStartThreads) void knn_starts_kernel(const KnnPlan *__restrict__ plan_ptr, int B,
                                                                   const int32_t *__restrict__ counts, int32_t *__restrict__ starts,
                                                                   int32_t *__restrict__ placed)
{
    __shared__ int wave_sum[kStartThreads / 64];
    __shared__ int base_s;
    const int pitch = plan_ptr->pitch;
    const int64_t rows = static_cast<int64_t>(B) * (plan_ptr->cells_per_batch / pitch);
    const int64_t rows_here = max(1, kStartCells / pitch);
    const int64_t first = static_cast<int64_t>(blockIdx.x) * rows_here;
    if (first >= rows) return;
    const int64_t cells0 = first * pitch, cells1 = min(first + rows_here, rows) * pitch;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // sum of a thread's four neighbouring cells before it, in the piece from `at` on, and the piece's sum
    int v[4];
    auto piece = [&](int64_t at, int &all) {
        const int64_t mine = at + 4 * static_cast<int>(threadIdx.x);
        int own = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = mine + e < cells1 ? counts[mine + e] : 0;
            own += v[e];
        }
        const int incl = wave_scan(own);
        if (lane == 63) wave_sum[wave] = incl;
        __syncthreads();
        int before = incl - own;
        all = 0;
#pragma unroll
        for (int w = 0; w < kStartThreads / 64; ++w) {
            before += w < wave ? wave_sum[w] : 0;
            all += wave_sum[w];
        }
        __syncthreads();
        return before;
    };
    auto write = [&](int64_t at, int run) {
        const int64_t mine = at + 4 * static_cast<int>(threadIdx.x);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (mine + e < cells1) starts[mine + e] = run;
            run += v[e];
        }
    };
    int all = 0, before = piece(cells0, all), total = all;
    // (a row of more cells than the workgroup takes at a time: twice through it)
    for (int64_t at = cells0 + kStartCells; at < cells1; at += kStartCells) {
        int more;
        piece(at, more);
        total += more;
    }
    if (threadIdx.x == 0) base_s = total > 0 ? atomicAdd(placed, total) : 0;
    __syncthreads();
    int base = base_s;
    if (cells1 - cells0 <= kStartCells) {
        write(cells0, base + before);
        return;
    }
    for (int64_t at = cells0; at < cells1; at += kStartCells) {
        before = piece(at, all);
        write(at, base + before);
        base += all;
    }
}

// The whole grid of up to kSmallSources sources by one workgroup, with the counters in LDS: box, plan, places, starts and
// sorted sources in one launch of 12 us instead of four that take 16 (2,951 sources).  Whole calls, one workgroup and several
// kernels: 1,500 sources 23.4 and 29.7 us, 3,000 27.6 and 32.7, 5,000 29.6 and 30.1, 8,100 36.1 and 32.5.
constexpr int kSmallThreads = 1024, kSmallEach = 4, kSmallSources = kSmallThreads * kSmallEach;
constexpr size_t small_lds(int64_t cells_cap) { return sizeof(int32_t) * static_cast<size_t>(cells_cap); }
__global__ __launch_bounds__(kSmallThreads) void knn_small_grid_kernel(
    const float *__restrict__ src, int64_t stride, int Ns, const int32_t *__restrict__ src_offset, int B, int K, float cell_hint, int cells_cap,
    KnnPlan *__restrict__ plan_out, int32_t *__restrict__ starts, float4 *__restrict__ sorted)
{
    extern __shared__ int counts[];
    __shared__ KnnPlan plan;
    __shared__ int part[kSmallThreads / 64][6], wave_sum[kSmallThreads / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float p[kSmallEach][3];
    int v[6];
#pragma unroll
    for (int a = 0; a < 6; ++a) v[a] = a < 3 ? 0x7fffffff : static_cast<int>(0x80000000u);
#pragma unroll
    for (int k = 0; k < kSmallEach; ++k) {
        const int i = k * kSmallThreads + static_cast<int>(threadIdx.x);
        if (k * kSmallThreads >= Ns) break;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            p[k][a] = i < Ns ? src[i * stride + a] : 0.0f;
            const int o = float_to_ordered(p[k][a]);
            v[a] = i < Ns ? min(v[a], o) : v[a];
            v[3 + a] = i < Ns ? max(v[3 + a], o) : v[3 + a];
        }
    }
    reduce_box<kSmallThreads / 64>(v, part, plan.lo);
    if (wave == 0) {
        make_plan(&plan, src_offset, B, Ns, K, cell_hint, cells_cap);
        if (lane == 0) *plan_out = plan;
    }
    __syncthreads();
    const int cells = B * plan.cells_per_batch;
    for (int c = threadIdx.x; c < cells; c += kSmallThreads) counts[c] = 0;
    __syncthreads();
    int cell[kSmallEach], slot[kSmallEach];
#pragma unroll
    for (int k = 0; k < kSmallEach; ++k) {
        const int i = k * kSmallThreads + static_cast<int>(threadIdx.x);
        if (k * kSmallThreads >= Ns) break;
        const int b = i < Ns ? find_batch(src_offset, B, i) : B;
        cell[k] = b < B ? cell_of(plan, p[k], b) : -1;
        slot[k] = cell[k] >= 0 ? atomicAdd(&counts[cell[k]], 1) : 0;
    }
    __syncthreads();
    // exclusive sum over the cells, a share of them per wavefront, four neighbours a lane
    const int share = ((cells + 16 * 256 - 1) / (16 * 256)) * 256;
    const int c0 = wave * share, c1 = min(c0 + share, cells);
    int sum = 0;
    for (int c = c0 + lane; c < c1; c += 64) sum += counts[c];
    sum = wave_scan(sum);
    if (lane == 63) wave_sum[wave] = sum;
    __syncthreads();
    int run = 0;
#pragma unroll
    for (int w = 0; w < kSmallThreads / 64; ++w) run += w < wave ? wave_sum[w] : 0;
    for (int c = c0; c < c1; c += 256) {
        int own[4], all = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            own[e] = c + 4 * lane + e < c1 ? counts[c + 4 * lane + e] : 0;
            all += own[e];
        }
        const int incl = wave_scan(all);
        int at = run + incl - all;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (c + 4 * lane + e < c1) {
                counts[c + 4 * lane + e] = at;
                starts[c + 4 * lane + e] = at;
            }
            at += own[e];
        }
        run += __builtin_amdgcn_readlane(incl, 63);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kSmallEach; ++k) {
        const int i = k * kSmallThreads + static_cast<int>(threadIdx.x);
        if (k * kSmallThreads >= Ns) break;
        if (cell[k] >= 0) sorted[counts[cell[k]] + slot[k]] = make_float4(p[k][0], p[k][1], p[k][2], __int_as_float(i));
    }
}

__global__ __launch_bounds__(kThreads) void knn_scatter_kernel(
    const float *__restrict__ src, int64_t stride, int64_t Ns, const int2 *__restrict__ src_place,
    const int32_t *__restrict__ starts, float4 *__restrict__ sorted)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= Ns) return;
    const int2 place = src_place[i];
    if (place.x < 0) return;
    sorted[starts[place.x] + place.y] = make_float4(src[i * stride], src[i * stride + 1], src[i * stride + 2],
                                                    __int_as_float(static_cast<int>(i)));
}

// ((dx*dx) + (dy*dy)) + (dz*dz) with d = src - query and every operation rounded to fp32 on
// its own: contraction into fused multiply-adds is switched off for this function (the
// compiler's default for device code is to fuse).
__device__ __forceinline__ float dist2_unfused(float sx, float sy, float sz, float qx, float qy,
                                               float qz)
{
#pragma clang fp contract(off)
    const float dx = sx - qx, dy = sy - qy, dz = sz - qz;
    const float xx = dx * dx, yy = dy * dy, zz = dz * dz;
    const float xy = xx + yy;
    return xy + zz;
}

// x of lane (this ^ MASK): within a row of 16 lanes by DPP (no LDS), beyond it through LDS
template <int CTRL> __device__ __forceinline__ uint64_t dpp(uint64_t x)
{
    const int lo = static_cast<int>(x), hi = static_cast<int>(x >> 32);
    return (static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, hi, CTRL, 0xf, 0xf, true))) << 32) |
           static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, lo, CTRL, 0xf, 0xf, true));
}
template <int MASK> __device__ __forceinline__ uint64_t lane_xor(uint64_t x)
{
    constexpr int kQuadReverse = 0x1b, kRowHalfMirror = 0x141, kRowMirror = 0x140, kRowRotate8 = 0x128;
    if constexpr (MASK == 1) return dpp<0xb1>(x);
    else if constexpr (MASK == 2) return dpp<0x4e>(x);
    else if constexpr (MASK == 3) return dpp<kQuadReverse>(x);
    else if constexpr (MASK == 7) return dpp<kRowHalfMirror>(x);
    else if constexpr (MASK == 4) return dpp<kQuadReverse>(dpp<kRowHalfMirror>(x));
    else if constexpr (MASK == 15) return dpp<kRowMirror>(x);
    else if constexpr (MASK == 8) return dpp<kRowRotate8>(x);
    else return __shfl_xor(x, MASK);
}

// Candidates are ordered as doubles, whose order the words' is: positive and finite (a distance is no NaN, see the kernel; that of a
// source at the query is a denormal number, which the instruction keeps).  One instruction in place of a comparison and two choices.
__device__ __forceinline__ uint64_t least(uint64_t a, uint64_t b)
{
    uint64_t r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// the smaller of two lanes' values to the lane without HIGH in its number, the larger one to the other: that one takes the least of
// the negated values
template <int MASK, int HIGH> __device__ __forceinline__ void exchange(uint64_t &x, int t)
{
    static_assert((MASK & HIGH) != 0, "one lane of the two");
    if constexpr (MASK > 15) {
        // (a move through LDS, where the comparison is shorter than a change of sign on either side of it: 33 neighbours in one launch,
        // queries a voxel, 595,677 voxels 984 us, 1029 with the minimum, 946 with the minimum within rows of sixteen lanes only; 64
        // neighbours 1296, 1297 and 1204, 199,327 voxels 538, 524 and 490)
        const uint64_t other = lane_xor<MASK>(x);
        x = (other < x) != ((t & HIGH) != 0) ? other : x;
        return;
    }
    const uint64_t sign = (t & HIGH) != 0 ? uint64_t(1) << 63 : 0, own = x ^ sign, other = lane_xor<MASK>(own);
    uint64_t r;
    asm("v_min_f64 %0, %1, -%2" : "=v"(r) : "v"(own), "v"(other));
    x = r ^ sign;
}
// ascending order of a bitonic sequence over SIZE lanes, and of any sequence (bitonic sort whose first step of a size
// compares mirrored lanes, so that every run is ascending)
template <int SIZE> __device__ __forceinline__ void order_bitonic(uint64_t &x, int t)
{
    if constexpr (SIZE > 1) {
        exchange<SIZE / 2, SIZE / 2>(x, t);
        order_bitonic<SIZE / 2>(x, t);
    }
}
template <int SIZE> __device__ __forceinline__ void order(uint64_t &x, int t)
{
    if constexpr (SIZE > 1) {
        order<SIZE / 2>(x, t);
        exchange<SIZE - 1, SIZE / 2>(x, t);
        order_bitonic<SIZE / 2>(x, t);
    }
}

// One query per group of G lanes (G = 4, 8, 16 or 64 >= K).  The group keeps its G best candidates as one sorted list, a
// candidate per lane: a word of (squared distance, source row), whose order is the result's.  The sources of a run of
// cells are read G at a time (the next ones while these are worked on), sorted across the lanes and merged: every step
// is a DPP move and a minimum on all lanes, no candidate waits for another.  At K = 16, 199,327 sources, a query for every
// cell of two voxels: 30 us (33 with a 64-bit comparison and two choices a step, and moves with a copy of their target ahead), and
// with those 43 us with each run of cells read by itself, most of a group's lanes idle in its last step; 73 us with candidates
// inserted one by one.  Bound by VALU issue (65 % of the time), most of it the sorting steps.
//
// A walk starts with the cube of 3 x 3 x 3 cells: the query's own cell alone never proves its K best.
// Groups of sixteen for up to eight neighbours, too, where there are few queries: a group then looks up the nine rows of cells
// in one step.  K = 3, groups of four / of sixteen, us a call (with its interpolation for the first): points within their
// voxels among means of cells, 12,000 queries 41 / 28, 50,000 53 / 40, 100,000 53 / 46, 199,000 65 / 70; centres of voxels among
// centres of cells, whose first cube always holds what they look for, 59,720 queries 31 / 33, 99,239 32 / 36, 199,185 41 / 55.
constexpr int64_t kFewQueries = 65536;
template <int G, int KMAX>
__global__ __launch_bounds__(kThreads) void knn_query_kernel(
    int K, const float *__restrict__ qry, int64_t stride, int64_t Nq, const int32_t *__restrict__ query_offset,
    int B, const KnnPlan *__restrict__ plan_ptr, const int32_t *__restrict__ starts,
    const float4 *__restrict__ sorted, int32_t *__restrict__ ret_idx, float *__restrict__ ret_dist, bool squared)
{
    constexpr uint64_t kNone = 0x7f8000007fffffffULL;      // (infinity, no row)
    const int lane = threadIdx.x & 63;
    const int t = lane % G;                    // position in the group's sorted list
    const int group_shift = lane - t;          // first lane of the group inside the wavefront
    const int64_t g_raw = (static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x) / G;
    const bool live = g_raw < Nq;              // groups past the last query idle along (no early
    const int64_t g = live ? g_raw : Nq - 1;   // exit: their lanes may share a wavefront with live ones)
    const KnnPlan plan = *plan_ptr;
    uint64_t best = kNone;
    const int b = find_batch(query_offset, B, g);
    if (b < B && plan.src_end > 0) {
        const float qx = qry[g * stride], qy = qry[g * stride + 1], qz = qry[g * stride + 2];
        const float qp[3] = {qx, qy, qz};
        int qc[3], r_first = 1, r_last = 0;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            qc[a] = cell_coord(qp[a], plan.origin[a], plan.inv_cell);
            const int below = -qc[a], above = qc[a] - (plan.dim[a] - 1);
            r_first = max(r_first, max(below, above));          // first cube touching the grid
            r_last = max(r_last, max(qc[a], -above));           // shell that covers the whole grid
        }
        r_last = max(r_last, r_first);
        const int32_t *cell_base = starts + static_cast<int64_t>(b) * plan.cells_per_batch;
        auto scan_rows = [&](int begin, int end) {
            // every lane's range of sources: the ranges one after the other, G sources at a time, whatever ranges they
            // belong to (a wall across the rows leaves some seven sources to each of nine ranges)
            const int len = max(end - begin, 0);
            int upto = len;
            if constexpr (G == 16) {
                upto += __builtin_amdgcn_update_dpp(0, upto, 0x111, 0xf, 0xf, true);      // row_shr
                upto += __builtin_amdgcn_update_dpp(0, upto, 0x112, 0xf, 0xf, true);
                upto += __builtin_amdgcn_update_dpp(0, upto, 0x114, 0xf, 0xf, true);
                upto += __builtin_amdgcn_update_dpp(0, upto, 0x118, 0xf, 0xf, true);
            } else {
#pragma unroll
                for (int off = 1; off < G; off <<= 1) {
                    const int up = __shfl_up(upto, off, G);
                    upto += t >= off ? up : 0;
                }
            }
            const int total = __shfl(upto, G - 1, G), ahead = begin - (upto - len);
            if (total == 0) return;
            auto source = [&](int at) {
                at = min(at, total - 1);
                int k = 0;                         // ranges that end at or before it
#pragma unroll
                for (int half = G / 2; half > 0; half >>= 1) k += __shfl(upto, k + half - 1, G) <= at ? half : 0;
                return sorted[at + __shfl(ahead, k, G)];
            };
            float4 p = source(t);
            for (int s = 0; s < total; s += G) {
                const float4 c = p;
                const bool have = s + t < total;
                if (s + G < total) p = source(s + G + t);
                const float d = dist2_unfused(c.x, c.y, c.z, qx, qy, qz);
                uint64_t found = (static_cast<uint64_t>(__float_as_uint(d)) << 32) | __float_as_uint(c.w);
                found = have && d == d ? found : kNone;      // (what is not a number is behind all that is)
                // (a group of sixteen skips sources that are all behind the last that can count)
                if (G == 16 && !__any(found < dpp<0x150 + KMAX - 1>(best))) continue;
                order<G>(found, t);
                found = lane_xor<G - 1>(found);
                best = least(found, best);
                order_bitonic<G>(best, t);
            }
        };
        for (int r = r_first; r <= r_last; ++r) {
            const int z0 = max(qc[2] - r, 0), z1 = min(qc[2] + r, plan.dim[2] - 1);
            const int y0 = max(qc[1] - r, 0), y1 = min(qc[1] + r, plan.dim[1] - 1);
            const int xl = qc[0] - r, xh = qc[0] + r;
            const int ny = y1 - y0 + 1;
            const int n_rows = (z1 - z0 + 1) * ny;   // <= 0 when the shell misses the grid in z or y
            // The rows of the shell, G at a time: every lane of the group looks up the source ranges of one row (the
            // lookups of up to G rows run side by side), then the group scans the rows that have sources - on surface
            // scans most cells of a shell are empty.  A row of a face, or of the first cube, spans the whole x range
            // (one contiguous run of cells), an interior row only its two end cells.
            for (int u0 = 0; u0 < n_rows; u0 += G) {
                int a0 = 0, a1 = 0, b0 = 0, b1 = 0;
                const int u = u0 + t;
                if (u < n_rows) {
                    const int dz = u / ny, z = z0 + dz, y = y0 + u - dz * ny;
                    const bool face = r == r_first || z == qc[2] - r || z == qc[2] + r || y == qc[1] - r || y == qc[1] + r;
                    const int32_t *row = cell_base + (z * plan.dim[1] + y) * plan.pitch;
                    if (face) {
                        const int x0 = max(xl, 0), x1 = min(xh, plan.dim[0] - 1);
                        if (x0 <= x1) {
                            a0 = row[x0];
                            a1 = row[x1 + 1];
                        }
                    } else {
                        if (xl >= 0 && xl < plan.dim[0]) {
                            a0 = row[xl];
                            a1 = row[xl + 1];
                        }
                        if (xh >= 0 && xh < plan.dim[0]) {
                            b0 = row[xh];
                            b1 = row[xh + 1];
                        }
                    }
                }
                scan_rows(a0, a1);
                if (r != r_first) scan_rows(b0, b1);
            }
            const uint64_t kth = __shfl(best, K - 1, G);
            if (static_cast<uint32_t>(kth) != 0x7fffffffu) {
                // everything outside the visited cube is at least `bound` away from the query
                float bound = INFINITY;
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    const float lo_face = plan.origin[a] + static_cast<float>(qc[a] - r) * plan.cell;
                    const float hi_face = plan.origin[a] + static_cast<float>(qc[a] + r + 1) * plan.cell;
                    bound = fminf(bound, fminf(qp[a] - lo_face, hi_face - qp[a]));
                }
                bound -= plan.slack;
                if (bound > 0.0f && __uint_as_float(static_cast<uint32_t>(kth >> 32)) < bound * bound) break;
            }
        }
    }
    if (live && t < K) {
        const int row = static_cast<int>(best & 0xffffffffu);
        const bool filled = row != 0x7fffffff;
        const float d = filled ? __uint_as_float(static_cast<uint32_t>(best >> 32)) : S3D_KNN_PAD_DIST2;
        ret_idx[g * K + t] = filled ? row : -1;
        ret_dist[g * K + t] = squared ? d : sqrtf(d);
    }
}

// Workgroups b, b + 8, .. run on one XCD: a contiguous share of the work each, so that neighbouring queries, which read
// the same sources' rows, find them in that XCD's L2.
__device__ __forceinline__ int64_t share_of_xcd(int64_t items)
{
    const int64_t share = ((items + kThreads - 1) / kThreads + 7) / 8;
    const int64_t block = static_cast<int64_t>(blockIdx.x) % 8 * share + static_cast<int64_t>(blockIdx.x) / 8;
    return block * kThreads + threadIdx.x;
}
inline dim3 xcd_grid(int64_t items) { return dim3(static_cast<unsigned>(ceil_div(ceil_div(items, kThreads), 8) * 8)); }

// Inverse-distance interpolation over the K nearest sources of every query
// (Swin3D/modules/swin3d_layers.py:53-73): weight_i = 1 / (sqrt(dist2_i) + 1e-8), normalised over the K
// neighbours, out = sum_i weight_i * src_feat[idx_i].  One thread per (query, group of VEC channels);
// padded neighbour slots (index -1) carry no weight.  fp32 accumulation, one rounding to the output type.
// kSkip: the result is fp32, added to a row of fp16 features (the projected skip features of an upsample), where the framework
// took a launch to widen src_feat and a sum of two types at a tenth of what memory gives: 25,013 x 96 48 us for the sum alone.
template <typename T, int VEC, bool kSkip>
__global__ __launch_bounds__(kThreads) void knn_interpolate_kernel(const int32_t *__restrict__ idx,
                                                                   const float *__restrict__ dist2, int K,
                                                                   int64_t Nq, const T *__restrict__ feat, int C,
                                                                   const _Float16 *__restrict__ skip,
                                                                   typename std::conditional<kSkip, float, T>::type *__restrict__ out)
{
    using Out = typename std::conditional<kSkip, float, T>::type;
    const int groups = C / VEC;
    const int64_t t = share_of_xcd(Nq * groups);
    if (t >= Nq * groups) return;
    const int64_t qi = t / groups;
    const int c0 = static_cast<int>(t - qi * groups) * VEC;
    // four neighbours at a time: their rows, distances and features are under way together
    constexpr int kAhead = 4;
    auto neighbours = [&](int i0, auto each) {
        int row[kAhead];
        float weight[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const int64_t at = qi * K + min(i0 + i, K - 1);
            row[i] = i0 + i < K ? idx[at] : -1;
            weight[i] = dist2[at];
        }
#pragma unroll
        for (int i = 0; i < kAhead; ++i) weight[i] = 1.0f / (sqrtf(weight[i]) + 1e-8f);
        each(row, weight);
    };
    float norm = 0.0f, acc[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) acc[e] = 0.0f;
    auto sum_weights = [&](const int *row, const float *weight) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i) norm += row[i] >= 0 ? weight[i] : 0.0f;
    };
    auto add_features = [&](const int *row, const float *weight, auto weights_known) {
        T v[kAhead][VEC];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const T *from = feat + static_cast<int64_t>(max(row[i], 0)) * C + c0;
            if (row[i] < 0) continue;
            if constexpr (VEC == 4) {
                if constexpr (sizeof(T) == 4) *reinterpret_cast<float4 *>(v[i]) = *reinterpret_cast<const float4 *>(from);
                else *reinterpret_cast<uint2 *>(v[i]) = *reinterpret_cast<const uint2 *>(from);
            } else {
                v[i][0] = *from;
            }
        }
        weights_known();
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            if (row[i] < 0) continue;
            const float w = weight[i] / norm;
#pragma unroll
            for (int e = 0; e < VEC; ++e) acc[e] += w * static_cast<float>(v[i][e]);
        }
    };
    if (K <= kAhead) {
        // (the features on their way while the weights are added up: 9.5 -> 7 us at 12,421 x 192 fp32, K = 3)
        neighbours(0, [&](const int *row, const float *weight) { add_features(row, weight, [&] { sum_weights(row, weight); }); });
    } else {
        for (int i0 = 0; i0 < K; i0 += kAhead) neighbours(i0, sum_weights);
        for (int i0 = 0; i0 < K; i0 += kAhead)
            neighbours(i0, [&](const int *row, const float *weight) { add_features(row, weight, [] {}); });
    }
    Out o[VEC];
    if constexpr (kSkip) {
        static_assert(VEC == 4, "rows of fours");
        _Float16 beside[VEC];
        *reinterpret_cast<uint2 *>(beside) = *reinterpret_cast<const uint2 *>(skip + qi * C + c0);
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[e] += static_cast<float>(beside[e]);
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) o[e] = static_cast<Out>(acc[e]);
    if constexpr (VEC == 4) {
        if constexpr (sizeof(Out) == 4)
            *reinterpret_cast<float4 *>(out + qi * C + c0) = *reinterpret_cast<const float4 *>(o);
        else
            *reinterpret_cast<uint2 *>(out + qi * C + c0) = *reinterpret_cast<const uint2 *>(o);
    } else {
        out[qi * C + c0] = o[0];
    }
}

// The gradient of that for src_feat, added to dsrc (zeros before), and of the rows beside it: dout in fp16.  A thread has CH channels
// of a query, a CH-th of a row apart, so that the lanes' additions lie side by side.  What bounds it is the pieces of lines that a
// wavefront's additions fall into: a whole row of up to 128 channels in lanes next to each other, half a row beyond, a quarter where
// that is a wavefront's width.  us by CH = 4 / 2 / 1: 199,866 queries of 48 channels 205 / 131 / 124, 50,651 of 96 70 / 60 / 57; of 160
// 103 / 80; 12,652 of 192 34 / 28 / 31; of 256 34.2 / 34.7, of 384 49.0 / 49.5, of 640 79.9 / 79.5; 3,116 of 256 11.6 / 11.7, of 320 13.7 /
// 14.0, of 384 15.4 / 16.2, of 512 19.0 / 19.7, of 640 23.1 / 23.4.
template <int CH>
__global__ __launch_bounds__(kThreads) void knn_interpolate_grad_kernel(const int32_t *__restrict__ idx, const float *__restrict__ dist2, int K,
                                                                        int64_t Nq, const float *__restrict__ dout, int C,
                                                                        float *__restrict__ dsrc, _Float16 *__restrict__ dskip)
{
    const int part = C / CH;
    const int64_t t = share_of_xcd(Nq * part);
    if (t >= Nq * part) return;
    const int64_t qi = t / part;
    const int c = static_cast<int>(t - qi * part);
    float g[CH];
#pragma unroll
    for (int e = 0; e < CH; ++e) g[e] = dout[qi * C + c + e * part];
    if (dskip) {
#pragma unroll
        for (int e = 0; e < CH; ++e) dskip[qi * C + c + e * part] = static_cast<_Float16>(g[e]);
    }
    if (!dsrc) return;
    float norm = 0.0f;
    for (int i = 0; i < K; ++i) norm += idx[qi * K + i] >= 0 ? 1.0f / (sqrtf(dist2[qi * K + i]) + 1e-8f) : 0.0f;
    norm = norm < 1e-30f ? 1e-30f : norm;      // (neighbours at an infinite distance have no share)
    for (int i = 0; i < K; ++i) {
        const int64_t row = idx[qi * K + i];
        if (row < 0) continue;
        const float w = 1.0f / (sqrtf(dist2[qi * K + i]) + 1e-8f) / norm;
#pragma unroll
        for (int e = 0; e < CH; ++e) unsafeAtomicAdd(dsrc + row * C + c + e * part, g[e] * w);
    }
}

template <typename T>
int launch_interpolate(const int32_t *idx, const float *dist2, int K, int64_t Nq, const void *feat, int C, void *out,
                       hipStream_t s)
{
    const T *f = static_cast<const T *>(feat);
    T *o = static_cast<T *>(out);
    if (C % 4 == 0) {
        const int64_t threads = Nq * (C / 4);
        hipLaunchKernelGGL((knn_interpolate_kernel<T, 4, false>), xcd_grid(threads), dim3(kThreads), 0, s, idx, dist2, K, Nq, f, C, nullptr, o);
    } else {
        const int64_t threads = Nq * C;
        hipLaunchKernelGGL((knn_interpolate_kernel<T, 1, false>), xcd_grid(threads), dim3(kThreads), 0, s, idx, dist2, K, Nq, f, C, nullptr, o);
    }
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

// Channel-wise maximum over the K nearest sources of every query (the max-pool of the KNN downsample,
// Swin3D/modules/swin3d_layers.py:292-312: gather [Nq,K,C], then max over K) without the gathered intermediate.
// One thread per (query, 16 bytes of channels).  A padded slot (row -1) reads row 0, as the clamped gather of
// the tensor statement does.  Bound by the gathered rows: with eight of them under way per thread and an XCD's queries next
// to each other 12.8 us at 199,327 x 96 fp16, K = 16, without 29.3.  The next level's rows are fp32: fp16 ones leave widened,
// 14.9 us where they and a cast took 21.8.
template <typename T, int VEC, typename Out>
__global__ __launch_bounds__(kThreads) void knn_max_pool_kernel(const int32_t *__restrict__ idx, int K, int64_t Nq,
                                                                const T *__restrict__ feat, int C,
                                                                Out *__restrict__ out)
{
    const int groups = C / VEC;
    const int64_t t = share_of_xcd(Nq * groups);
    if (t >= Nq * groups) return;
    const int64_t qi = t / groups;
    const int c0 = static_cast<int>(t - qi * groups) * VEC;
    // eight rows at a time, their loads under way together (the slots behind the K-th repeat it)
    constexpr int kAhead = 8;
    T best[VEC];
    for (int i0 = 0; i0 < K; i0 += kAhead) {
        int row[kAhead];
        T v[kAhead][VEC];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) row[i] = max(idx[qi * K + min(i0 + i, K - 1)], 0);
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const T *from = feat + static_cast<int64_t>(row[i]) * C + c0;
            if constexpr (VEC * sizeof(T) == 16) *reinterpret_cast<uint4 *>(v[i]) = *reinterpret_cast<const uint4 *>(from);
            else v[i][0] = *from;
        }
#pragma unroll
        for (int i = 0; i < kAhead; ++i)
#pragma unroll
            for (int e = 0; e < VEC; ++e) best[e] = (i0 + i == 0 || v[i][e] > best[e] || v[i][e] != v[i][e]) ? v[i][e] : best[e];
    }
    if constexpr (VEC * sizeof(T) == 16) {
        constexpr int kPiece = 16 / sizeof(Out);
        Out o[VEC];
#pragma unroll
        for (int e = 0; e < VEC; ++e) o[e] = static_cast<Out>(best[e]);
#pragma unroll
        for (int e = 0; e < VEC; e += kPiece) *reinterpret_cast<uint4 *>(out + qi * C + c0 + e) = *reinterpret_cast<const uint4 *>(o + e);
    } else {
        out[qi * C + c0] = static_cast<Out>(best[0]);
    }
}

template <typename T, typename Out>
int launch_max_pool(const int32_t *idx, int K, int64_t Nq, const void *feat, int C, void *out, hipStream_t s)
{
    const T *f = static_cast<const T *>(feat);
    Out *o = static_cast<Out *>(out);
    constexpr int kVec = 16 / static_cast<int>(sizeof(T));
    if (C % kVec == 0 && reinterpret_cast<uintptr_t>(feat) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0) {
        const int64_t threads = Nq * (C / kVec);
        hipLaunchKernelGGL((knn_max_pool_kernel<T, kVec, Out>), xcd_grid(threads), dim3(kThreads), 0, s, idx, K, Nq, f, C, o);
    } else {
        const int64_t threads = Nq * C;
        hipLaunchKernelGGL((knn_max_pool_kernel<T, 1, Out>), xcd_grid(threads), dim3(kThreads), 0, s, idx, K, Nq, f, C, o);
    }
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

}  // namespace
}  // namespace s3d

namespace s3d {
namespace {

int max_pool(const int32_t *idx, int32_t K, int64_t Nq, const void *src_feat, int64_t Ns, int32_t C, int32_t dtype, bool widened, void *out, void *stream)
{
    if (K < 1 || K > S3D_KNN_KMAX) return fail(S3D_ERR_BAD_SHAPE, "s3d_knn_max_pool: K=%d outside 1..%d", K, S3D_KNN_KMAX);
    if (Nq < 0 || Ns < 0 || C < 1 || Nq * static_cast<int64_t>(C) > 0x3fffffffffLL || (Nq > 0 && Ns < 1))
        return fail(S3D_ERR_BAD_SHAPE, "s3d_knn_max_pool: Nq=%lld Ns=%lld C=%d out of range", (long long)Nq, (long long)Ns,
                    C);
    if (dtype != S3D_DTYPE_F32 && dtype != S3D_DTYPE_F16)
        return fail(S3D_ERR_BAD_DTYPE, "s3d_knn_max_pool: dtype %d (0 = fp32, 1 = fp16)", dtype);
    if (Nq == 0) return S3D_OK;
    if (!idx || !out || !src_feat) return fail(S3D_ERR_NULL_POINTER, "s3d_knn_max_pool: null device pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    return dtype == S3D_DTYPE_F32 ? launch_max_pool<float, float>(idx, K, Nq, src_feat, C, out, s)
           : widened              ? launch_max_pool<_Float16, float>(idx, K, Nq, src_feat, C, out, s)
                                  : launch_max_pool<_Float16, _Float16>(idx, K, Nq, src_feat, C, out, s);
}

}  // namespace
}  // namespace s3d

extern "C" __attribute__((visibility("default"))) int s3d_knn_max_pool(const int32_t *idx, int32_t K, int64_t Nq,
                                                                        const void *src_feat, int64_t Ns, int32_t C,
                                                                        int32_t dtype, void *out, void *stream)
{
    return s3d::max_pool(idx, K, Nq, src_feat, Ns, C, dtype, false, out, stream);
}

extern "C" __attribute__((visibility("default"))) int s3d_knn_max_pool_widened(const int32_t *idx, int32_t K, int64_t Nq, const void *src_feat,
                                                                                int64_t Ns, int32_t C, float *out, void *stream)
{
    return s3d::max_pool(idx, K, Nq, src_feat, Ns, C, S3D_DTYPE_F16, true, out, stream);
}

extern "C" __attribute__((visibility("default"))) size_t s3d_knn_workspace_bytes(int64_t Ns, int64_t Nq, int32_t B)
{
    (void)Nq;
    (void)B;
    return s3d::make_layout(Ns).total;
}

namespace s3d {
namespace {

int knn(int32_t K, const float *src_xyz, int64_t src_stride, int64_t Ns, const float *query_xyz, int64_t query_stride, int64_t Nq,
        const int32_t *src_offset,
        const int32_t *query_offset, int32_t B, int32_t *ret_idx, float *ret_dist, bool squared, float cell_size,
        void *workspace, size_t workspace_bytes, void *stream)
{
    if (K < 1 || K > S3D_KNN_KMAX)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_knn: K=%d outside 1..%d", K, S3D_KNN_KMAX);
    if (src_stride < 3 || query_stride < 3)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_knn: rows %lld and %lld floats apart", (long long)src_stride, (long long)query_stride);
    if (Ns < 0 || Nq < 0 || Ns > 0x7fffffffLL || Nq > 0x3fffffffLL || B < 1 || B > kMaxBatch)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_knn: Ns=%lld Nq=%lld B=%d out of range", (long long)Ns,
                    (long long)Nq, B);
    if (Nq == 0) return S3D_OK;
    if (!query_xyz || !src_offset || !query_offset || !ret_idx || !ret_dist || !workspace ||
        (Ns > 0 && !src_xyz))
        return fail(S3D_ERR_NULL_POINTER, "s3d_knn: null device pointer");
    const Layout L = make_layout(Ns);
    if (workspace_bytes < L.total)
        return fail(S3D_ERR_WORKSPACE, "s3d_knn: workspace %zu B < required %zu B", workspace_bytes,
                    L.total);
    hipStream_t s = static_cast<hipStream_t>(stream);
    char *base = static_cast<char *>(workspace);
    KnnPlan *plan = reinterpret_cast<KnnPlan *>(base + L.plan);
    int32_t *counts = reinterpret_cast<int32_t *>(base + L.counts);
    int32_t *starts = reinterpret_cast<int32_t *>(base + L.starts);
    int2 *src_place = reinterpret_cast<int2 *>(base + L.src_place);
    int32_t *partials = reinterpret_cast<int32_t *>(base + L.partials);
    float4 *sorted = reinterpret_cast<float4 *>(base + L.sorted);
    const int64_t cells = L.cells_cap;

    if (Ns > kSmallSources) {
        // bounding box + zeroed counters, places (grid derived in every workgroup), starts, scatter
        const dim3 sgrid(static_cast<unsigned>(ceil_div(Ns, kThreads)));
        hipLaunchKernelGGL(knn_bbox_kernel, dim3(kBboxBlocks), dim3(kThreads), 0, s, src_xyz, src_stride, Ns, partials, counts, cells);
        hipLaunchKernelGGL(knn_count_kernel, sgrid, dim3(kThreads), 0, s, src_xyz, src_stride, Ns, src_offset, B, partials,
                           kBboxBlocks, K, cell_size, L.cells_cap, plan, counts, src_place);
        // (workgroups: a share of whole rows is at least half of kStartCells, or a single row)
        hipLaunchKernelGGL(knn_starts_kernel, dim3(static_cast<unsigned>(2 * cells / kStartCells + 1)), dim3(kStartThreads), 0, s, plan, B,
                           counts, starts, partials + 6 * kBboxBlocks);
        hipLaunchKernelGGL(knn_scatter_kernel, sgrid, dim3(kThreads), 0, s, src_xyz, src_stride, Ns, src_place, starts, sorted);
        S3D_HIP_CHECK(hipGetLastError());
    } else if (Ns > 0) {
        const size_t lds = small_lds(cells);
        if (int rc = allow_dynamic_lds(reinterpret_cast<const void *>(knn_small_grid_kernel), small_lds(cells_cap_for(kSmallSources)))) return rc;
        hipLaunchKernelGGL(knn_small_grid_kernel, dim3(1), dim3(kSmallThreads), lds, s, src_xyz, src_stride, static_cast<int>(Ns), src_offset, B, K,
                           cell_size, static_cast<int>(cells), plan, starts, sorted);
        S3D_HIP_CHECK(hipGetLastError());
    } else {
        hipLaunchKernelGGL(knn_plan_kernel, dim3(1), dim3(64), 0, s, plan, src_offset, B, Ns, K,
                           cell_size, L.cells_cap);
        S3D_HIP_CHECK(hipGetLastError());
    }
    // lanes per query: the smallest group that holds the K entries, one per lane; sixteen where groups of four would not
    // fill the chip
    const bool few = Nq <= kFewQueries;
    const int G = K <= 4 && !few ? 4 : K <= 8 && !few ? 8 : K <= 16 ? 16 : 64;
    const dim3 qgrid(static_cast<unsigned>(ceil_div(Nq * G, kThreads)));
    auto query = G == 4 ? knn_query_kernel<4, 4> : G == 8 ? knn_query_kernel<8, 8> : G == 64 ? knn_query_kernel<64, 64>
                 : K <= 4 ? knn_query_kernel<16, 4> : K <= 8 ? knn_query_kernel<16, 8> : knn_query_kernel<16, 16>;
    hipLaunchKernelGGL(query, qgrid, dim3(kThreads), 0, s, K, query_xyz, query_stride, Nq, query_offset, B, plan, starts, sorted, ret_idx,
                       ret_dist, squared);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

}  // namespace
}  // namespace s3d

extern "C" __attribute__((visibility("default"))) int s3d_knn(
    int32_t K, const float *src_xyz, int64_t Ns, const float *query_xyz, int64_t Nq, const int32_t *src_offset,
    const int32_t *query_offset, int32_t B, int32_t *ret_idx, float *ret_dist2, float cell_size, void *workspace,
    size_t workspace_bytes, void *stream)
{
    return s3d::knn(K, src_xyz, 3, Ns, query_xyz, 3, Nq, src_offset, query_offset, B, ret_idx, ret_dist2, true, cell_size, workspace,
                    workspace_bytes, stream);
}

extern "C" __attribute__((visibility("default"))) int s3d_knn_strided(
    int32_t K, const float *src_xyz, int64_t src_stride, int64_t Ns, const float *query_xyz, int64_t query_stride, int64_t Nq,
    const int32_t *src_offset, const int32_t *query_offset, int32_t B, int32_t *ret_idx, float *ret_dist2, float cell_size,
    void *workspace, size_t workspace_bytes, void *stream)
{
    return s3d::knn(K, src_xyz, src_stride, Ns, query_xyz, query_stride, Nq, src_offset, query_offset, B, ret_idx, ret_dist2, true,
                    cell_size, workspace, workspace_bytes, stream);
}

extern "C" __attribute__((visibility("default"))) int s3d_knn_distances(
    int32_t K, const float *src_xyz, int64_t Ns, const float *query_xyz, int64_t Nq, const int32_t *src_offset,
    const int32_t *query_offset, int32_t B, int32_t *ret_idx, float *ret_dist, float cell_size, void *workspace,
    size_t workspace_bytes, void *stream)
{
    return s3d::knn(K, src_xyz, 3, Ns, query_xyz, 3, Nq, src_offset, query_offset, B, ret_idx, ret_dist, false, cell_size, workspace,
                    workspace_bytes, stream);
}

extern "C" __attribute__((visibility("default"))) int s3d_knn_interpolate(
    const int32_t *idx, const float *dist2, int32_t K, int64_t Nq, const void *src_feat, int64_t Ns, int32_t C,
    int32_t dtype, void *out, void *stream)
{
    using namespace s3d;
    if (K < 1 || K > S3D_KNN_KMAX) return fail(S3D_ERR_BAD_SHAPE, "s3d_knn_interpolate: K=%d outside 1..%d", K, S3D_KNN_KMAX);
    if (Nq < 0 || Ns < 0 || C < 1 || Nq * static_cast<int64_t>(C) > 0x3fffffffffLL)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_knn_interpolate: Nq=%lld Ns=%lld C=%d out of range", (long long)Nq,
                    (long long)Ns, C);
    if (dtype != S3D_DTYPE_F32 && dtype != S3D_DTYPE_F16)
        return fail(S3D_ERR_BAD_DTYPE, "s3d_knn_interpolate: dtype %d (0 = fp32, 1 = fp16)", dtype);
    if (Nq == 0) return S3D_OK;
    if (!idx || !dist2 || !out || (Ns > 0 && !src_feat))
        return fail(S3D_ERR_NULL_POINTER, "s3d_knn_interpolate: null device pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    return dtype == S3D_DTYPE_F16 ? launch_interpolate<_Float16>(idx, dist2, K, Nq, src_feat, C, out, s)
                                  : launch_interpolate<float>(idx, dist2, K, Nq, src_feat, C, out, s);
}

namespace s3d {
namespace {

int check_interpolation(const char *who, const void *idx, const void *dist2, int32_t K, int64_t Nq, int64_t Ns, int32_t C)
{
    if (K < 1 || K > S3D_KNN_KMAX) return fail(S3D_ERR_BAD_SHAPE, "%s: K=%d outside 1..%d", who, K, S3D_KNN_KMAX);
    if (Nq < 0 || Ns < 1 || C < 4 || C % 4 || Nq * static_cast<int64_t>(C) > 0x3fffffffffLL)
        return fail(S3D_ERR_BAD_SHAPE, "%s: Nq=%lld Ns=%lld C=%d (a multiple of 4) out of range", who, (long long)Nq, (long long)Ns, C);
    if (Nq > 0 && (!idx || !dist2)) return fail(S3D_ERR_NULL_POINTER, "%s: null device pointer", who);
    return S3D_OK;
}

}  // namespace
}  // namespace s3d

extern "C" __attribute__((visibility("default"))) int s3d_knn_interpolate_add(
    const int32_t *idx, const float *dist2, int32_t K, int64_t Nq, const void *src_feat, int64_t Ns, int32_t C,
    const void *skip, float *out, void *stream)
{
    using namespace s3d;
    if (int rc = check_interpolation("s3d_knn_interpolate_add", idx, dist2, K, Nq, Ns, C)) return rc;
    if (Nq == 0) return S3D_OK;
    if (!src_feat || !skip || !out) return fail(S3D_ERR_NULL_POINTER, "s3d_knn_interpolate_add: null device pointer");
    hipLaunchKernelGGL((knn_interpolate_kernel<_Float16, 4, true>), xcd_grid(Nq * (C / 4)), dim3(kThreads), 0, static_cast<hipStream_t>(stream),
                       idx, dist2, K, Nq, static_cast<const _Float16 *>(src_feat), C, static_cast<const _Float16 *>(skip), out);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

extern "C" __attribute__((visibility("default"))) int s3d_knn_interpolate_grad(
    const int32_t *idx, const float *dist2, int32_t K, int64_t Nq, const float *dout, int64_t Ns, int32_t C, float *dsrc_feat,
    void *dskip, void *stream)
{
    using namespace s3d;
    if (int rc = check_interpolation("s3d_knn_interpolate_grad", idx, dist2, K, Nq, Ns, C)) return rc;
    if (Nq == 0 || (!dsrc_feat && !dskip)) return S3D_OK;
    if (!dout) return fail(S3D_ERR_NULL_POINTER, "s3d_knn_interpolate_grad: null device pointer");
    const int own = C <= 128 ? 1 : C < 256 ? 2 : 4;
    auto kernel = own == 1 ? knn_interpolate_grad_kernel<1> : own == 2 ? knn_interpolate_grad_kernel<2> : knn_interpolate_grad_kernel<4>;
    hipLaunchKernelGGL(kernel, xcd_grid(Nq * (C / own)), dim3(kThreads), 0, static_cast<hipStream_t>(stream), idx, dist2, K, Nq, dout, C,
                       dsrc_feat, static_cast<_Float16 *>(dskip));
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}
