// Window sort + segment offsets for sparse-voxel window attention (gfx950).
//
// Replaces the MinkowskiEngine pooling / kernel_map / torch.sort pipeline of
// Swin3D/modules/swin3d_layers.py:713-787 and the w2n / w_sizes scans of
// :96-103.  Every voxel gets one 64-bit key
//     [ batch:12 | wx+8192:14 | wy+8192:14 | wz+8192:14 | local id:10 ]
// with w = floor((coord + shift*stride) / (window*stride)) and
// local id = (lx*window + ly)*window + lz; a stable radix sort of (key, row)
// yields the window-sorted order, a flag + scan pass yields the segments.
// Integer work only; HBM traffic is a handful of passes over 12 B per voxel.
#include "s3d_common.h"

#include <cstring>

#include <type_traits>

#include <rocprim/rocprim.hpp>

namespace s3d {
namespace {

constexpr int kThreads = 256;
constexpr int kLocalBits = 10;
constexpr int kAxisBits = 14;
constexpr int kAxisBias = 1 << (kAxisBits - 1);  // 8192
constexpr int kBatchBits = 12;

struct Layout {
    size_t keys_in, keys_out, vals_in, flags, ranks, temp, temp_bytes, total;
};

size_t sort_temp_bytes(int64_t N)
{
    size_t bytes = 0;
    uint64_t *kn = nullptr;
    int32_t *vn = nullptr;
    (void)rocprim::radix_sort_pairs(nullptr, bytes, kn, kn, vn, vn, static_cast<size_t>(N), 0, 64,
                                    hipStream_t(0));
    return bytes;
}

size_t scan_temp_bytes(int64_t N)
{
    size_t bytes = 0;
    int32_t *p = nullptr;
    (void)rocprim::inclusive_scan(nullptr, bytes, p, p, static_cast<size_t>(N),
                                  rocprim::plus<int32_t>(), hipStream_t(0));
    return bytes;
}

Layout make_layout(int64_t N)
{
    Layout L{};
    const size_t n = static_cast<size_t>(N > 0 ? N : 1);
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t at = off;
        off = align_up(off + bytes, 256);
        return at;
    };
    L.keys_in = take(n * sizeof(uint64_t));
    L.keys_out = take(n * sizeof(uint64_t));
    L.vals_in = take(n * sizeof(int32_t));
    L.flags = take(n * sizeof(int32_t));
    L.ranks = take(n * sizeof(int32_t));
    const size_t a = sort_temp_bytes(static_cast<int64_t>(n));
    const size_t b = scan_temp_bytes(static_cast<int64_t>(n));
    L.temp_bytes = a > b ? a : b;
    L.temp = take(L.temp_bytes);
    L.total = off;
    return L;
}

__device__ __forceinline__ int floordiv(int a, int b)
{
    int q = a / b;
    if ((a % b != 0) && ((a < 0) != (b < 0))) --q;
    return q;
}

__global__ void init_counts_kernel(int64_t *counts)
{
    if (threadIdx.x < 4) counts[threadIdx.x] = 0;
}

__global__ __launch_bounds__(kThreads) void build_keys_kernel(
    const int32_t *__restrict__ coords, int64_t N, int stride, int window, int shift,
    uint64_t *__restrict__ keys, int32_t *__restrict__ vals, int64_t *__restrict__ counts)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= N) return;
    const int4 c = reinterpret_cast<const int4 *>(coords)[i];
    const int span = window * stride;
    const int cc[3] = {c.y + shift * stride, c.z + shift * stride, c.w + shift * stride};
    int wv[3], lv[3];
    bool bad = c.x < 0 || c.x >= (1 << kBatchBits);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        wv[a] = floordiv(cc[a], span);
        lv[a] = (cc[a] - wv[a] * span) / stride;  // numerator in [0, span)
        bad = bad || wv[a] < -kAxisBias || wv[a] >= kAxisBias;
        wv[a] = min(max(wv[a], -kAxisBias), kAxisBias - 1);
    }
    if (bad) atomicMax(reinterpret_cast<unsigned long long *>(counts + 3), 1ULL);
    const uint64_t b = static_cast<uint64_t>(min(max(c.x, 0), (1 << kBatchBits) - 1));
    const uint64_t local = static_cast<uint64_t>((lv[0] * window + lv[1]) * window + lv[2]);
    uint64_t key = b;
    key = (key << kAxisBits) | static_cast<uint64_t>(wv[0] + kAxisBias);
    key = (key << kAxisBits) | static_cast<uint64_t>(wv[1] + kAxisBias);
    key = (key << kAxisBits) | static_cast<uint64_t>(wv[2] + kAxisBias);
    key = (key << kLocalBits) | local;
    keys[i] = key;
    vals[i] = static_cast<int32_t>(i);
}

__global__ __launch_bounds__(kThreads) void flag_kernel(const uint64_t *__restrict__ keys, int64_t N,
                                                        int32_t *__restrict__ flags,
                                                        int32_t *__restrict__ w_w_id)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= N) return;
    const uint64_t key = keys[i];
    const bool first = (i == 0) || ((keys[i - 1] >> kLocalBits) != (key >> kLocalBits));
    flags[i] = first ? 1 : 0;
    w_w_id[i] = static_cast<int32_t>(key & ((1u << kLocalBits) - 1));
}

__global__ __launch_bounds__(kThreads) void segment_start_kernel(
    const int32_t *__restrict__ flags, const int32_t *__restrict__ ranks, int64_t N,
    int32_t *__restrict__ w2n, int64_t *__restrict__ counts)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= N) return;
    if (flags[i]) w2n[ranks[i] - 1] = static_cast<int32_t>(i);
    if (i == N - 1) counts[0] = ranks[i];
}

__global__ __launch_bounds__(kThreads) void segment_size_kernel(const int32_t *__restrict__ w2n,
                                                                int64_t N,
                                                                int32_t *__restrict__ w_sizes,
                                                                int64_t *__restrict__ counts)
{
    const int64_t w = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    const int64_t W = counts[0];  // written by the previous kernel on the same stream
    long long size = 0;
    if (w < W) {
        const int32_t begin = w2n[w];
        const int32_t end = (w + 1 < W) ? w2n[w + 1] : static_cast<int32_t>(N);
        size = end - begin;
        w_sizes[w] = static_cast<int32_t>(size);
    }
    long long sq = size * size, mx = size;
    for (int off = 32; off > 0; off >>= 1) {
        sq += __shfl_down(sq, off);
        mx = max(mx, __shfl_down(mx, off));
    }
    if ((threadIdx.x & 63) == 0 && mx > 0) {
        atomicAdd(reinterpret_cast<unsigned long long *>(counts + 1), static_cast<unsigned long long>(sq));
        atomicMax(reinterpret_cast<unsigned long long *>(counts + 2), static_cast<unsigned long long>(mx));
    }
}

// ---- grid path: the same index without a sort of all voxels ----------------------------------------------
// When the windows of a scene fit a dense lattice of at most cells_cap cells (they do for room-sized scenes: the
// lattice is the bounding box of the window coordinates), a window is a lattice cell and the index is a counting
// sort: every voxel draws a slot in its cell, a sum over the cells before it gives every non-empty cell its rank (= window
// number, ascending (batch, wx, wy, wz) because the cell number is) and its first position, the voxels are placed
// there, and each window's few voxels are put in (local id, row) order by one wavefront.  Six launches of a few
// microseconds instead of a block sort and eight merge passes.
//
// Up to kMaxSets window sets of the same voxels are built together (blockIdx.y = set): what bounds a set alone is the
// launches, each with too little work for the card (199,327 voxels, two sets: 46 us of kernels instead of 73).  The lattices
// come from one bounding box of the coordinates (a window coordinate does not decrease with its voxel's).
//
// The windows, their pairs and the largest are known when the cells have been added up, and a host that sizes by them what
// follows on the same stream waits for that and not for the placing behind it (two sets with their signals at 199,327 voxels: 81 us a
// pass, 96 where it waits for all, which another stream that reads the sets needs).  (The sums run over the cells that the lattice has, not
// over those it may have, in two launches; a library's scan over 2 N took two as well, 14 us against 6 at 199,327 voxels.)
constexpr int kGridBoxes = 128;          // workgroups of the bounding-box pass
constexpr int kGridZeros = 384;          // ... and those beside them that only clear cells (without them two sets 1 to 2 us longer)
constexpr int kSlotBits = 20;            // a voxel's slot in its cell, below its local id in one word
constexpr int kBadRange = 1, kNoGrid = 2;   // counts[3]: coordinates out of range / lattice too large for the grid path

constexpr int kMaxSets = 4;

struct GridSet {
    int window, shift;
    int32_t *n2n, *w_w_id, *w_sizes, *w2n;
    int64_t *counts;
};

struct GridSets {
    GridSet set[kMaxSets];
    int num;
};

struct GridPlan {
    int lo[4], dim[4];   // batch, wx, wy, wz: lowest value and extent of the lattice
    int ok;              // the lattice fits
};

struct GridLayout {
    size_t plan, partials, cells, sums, place, keys, total;
    int64_t cells_cap;
};

int64_t grid_cells_cap(int64_t N)
{
    // (Voxels lie on surfaces, so the windows' lattice grows faster than they do: for cells of two voxels a side 1.1 a voxel in a
    // room of 25,000, 2.0 at 100,000, 4.3 at 450,000.  A set that does not fit is built again by the sort of all voxels after one
    // more wait of the host: three sets, the third of such cells, at 2 N 178 us for 100,000 voxels, 197 for 199,327 and 335 for
    // 595,677; at 6 N 69, 77 and 123.  Two sets of windows of five take what they took, 62 us at 199,327: the cells are cleared beside the
    // box, and those behind the lattice's own are not read.)
    int64_t cap = 6 * N;
    if (cap < 4096) cap = 4096;
    if (cap > (1LL << 24)) cap = 1LL << 24;
    return cap;
}

// cells of a run, which a workgroup of the two launches that add them up takes at a time, and what is left of them there
constexpr int kSumThreads = 1024, kSumCells = 4 * kSumThreads;
struct CellSum {
    uint64_t before;       // (non-empty << 32 | voxels)
    int64_t squares;
    int32_t largest, unused;
};
__host__ __device__ __forceinline__ int64_t sum_groups(int64_t cells_cap) { return (cells_cap + kSumCells - 1) / kSumCells; }
__host__ __device__ __forceinline__ uint64_t cell_word(int32_t count) { return (count > 0 ? (1ULL << 32) : 0ULL) | static_cast<uint32_t>(count); }

// plans, cells, sums, place and keys: one of each per set, one behind the other
GridLayout make_grid_layout(int64_t N, int sets)
{
    GridLayout L{};
    L.cells_cap = grid_cells_cap(N);
    const size_t n = static_cast<size_t>(N > 0 ? N : 1) * sets, cells = static_cast<size_t>(L.cells_cap) * sets;
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t at = off;
        off = align_up(off + bytes, 256);
        return at;
    };
    L.plan = take(sizeof(GridPlan) * sets);
    L.partials = take(sizeof(int32_t) * 8 * kGridBoxes);
    L.cells = take(cells * sizeof(int32_t));
    L.sums = take(sizeof(CellSum) * sets * static_cast<size_t>(sum_groups(L.cells_cap)));
    L.place = take(n * sizeof(int2));
    L.keys = take(n * sizeof(uint64_t));
    L.total = off;
    return L;
}

// window coordinates and local id of a voxel; false when they are outside the supported range
__device__ __forceinline__ bool window_of(const int4 c, int stride, int window, int shift, int *w, int *local)
{
    const int span = window * stride;
    const int cc[3] = {c.y + shift * stride, c.z + shift * stride, c.w + shift * stride};
    int lv[3];
    bool bad = c.x < 0 || c.x >= (1 << kBatchBits);
    w[0] = min(max(c.x, 0), (1 << kBatchBits) - 1);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int wv = floordiv(cc[a], span);
        lv[a] = (cc[a] - wv * span) / stride;
        bad = bad || wv < -kAxisBias || wv >= kAxisBias;
        w[1 + a] = min(max(wv, -kAxisBias), kAxisBias - 1);
    }
    *local = (lv[0] * window + lv[1]) * window + lv[2];
    return !bad;
}

// partial bounding boxes of the coordinates (one per workgroup, no atomics), the cell counters and the sets' totals and
// status words at zero (the later launches only ever OR bits into a status word)
__global__ __launch_bounds__(kThreads) void grid_bbox_kernel(const int32_t *__restrict__ coords, int64_t N, GridSets sets,
                                                             int32_t *__restrict__ partials, int32_t *__restrict__ cells,
                                                             int64_t num_cells)
{
    if (blockIdx.x == 0 && threadIdx.x < 4)
        for (int s = 0; s < sets.num; ++s) sets.set[s].counts[threadIdx.x] = 0;
    // (four cells at once; the room for them ends on a multiple of that)
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; i < (num_cells + 3) / 4;
         i += static_cast<int64_t>(gridDim.x) * kThreads)
        reinterpret_cast<int4 *>(cells)[i] = make_int4(0, 0, 0, 0);
    if (blockIdx.x >= kGridBoxes) return;
    int lo[4], hi[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) { lo[a] = 0x7fffffff; hi[a] = static_cast<int>(0x80000000u); }
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; i < N;
         i += static_cast<int64_t>(kGridBoxes) * kThreads) {
        const int4 c = reinterpret_cast<const int4 *>(coords)[i];
        const int x[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
        for (int a = 0; a < 4; ++a) { lo[a] = min(lo[a], x[a]); hi[a] = max(hi[a], x[a]); }
    }
    for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            lo[a] = min(lo[a], __shfl_down(lo[a], off));
            hi[a] = max(hi[a], __shfl_down(hi[a], off));
        }
    }
    __shared__ int part[kThreads / 64][8];
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int a = 0; a < 4; ++a) { part[threadIdx.x >> 6][a] = lo[a]; part[threadIdx.x >> 6][4 + a] = hi[a]; }
    }
    __syncthreads();
    if (threadIdx.x < 8) {
        int v = part[0][threadIdx.x];
        for (int wv = 1; wv < kThreads / 64; ++wv)
            v = threadIdx.x < 4 ? min(v, part[wv][threadIdx.x]) : max(v, part[wv][threadIdx.x]);
        partials[threadIdx.x * kGridBoxes + blockIdx.x] = v;
    }
}

// Every workgroup reduces the partial boxes to its set's lattice (workgroup 0 of a set records it and its bits of the
// status word); then every voxel draws a slot in its cell - neighbouring lanes of one cell with one atomic.  A cell that
// runs out of slot numbers (more than 2^kSlotBits voxels in one window: only with masses of equal coordinates) sets the
// "no grid" bit as well: the status word was zeroed by the launch before this one and every writer ORs into it, so
// no bit is lost whichever workgroup comes first, and the later launches of the call write nothing once it is set.
__global__ __launch_bounds__(kThreads) void grid_count_kernel(
    const int32_t *__restrict__ coords, int64_t N, int stride, GridSets sets, const int32_t *__restrict__ partials,
    int64_t cells_cap, GridPlan *__restrict__ plan_out, int32_t *__restrict__ cells, int2 *__restrict__ place)
{
    __shared__ GridPlan plan;
    __shared__ int box[8];
    const int set = blockIdx.y, window = sets.set[set].window, shift = sets.set[set].shift;
    int64_t *counts = sets.set[set].counts;
    cells += set * cells_cap;
    place += set * N;
    {
        // eight numbers by 32 lanes each
        static_assert(kThreads == 8 * 32 && kGridBoxes % 32 == 0, "a thread per part of a number");
        const int a = threadIdx.x >> 5;
        int v = partials[a * kGridBoxes + (threadIdx.x & 31)];
#pragma unroll
        for (int t = 32; t < kGridBoxes; t += 32) {
            const int o = partials[a * kGridBoxes + t + (threadIdx.x & 31)];
            v = a < 4 ? min(v, o) : max(v, o);
        }
        for (int off = 16; off > 0; off >>= 1) {
            const int o = __shfl_down(v, off, 32);
            v = a < 4 ? min(v, o) : max(v, o);
        }
        if ((threadIdx.x & 31) == 0) box[a] = v;
        __syncthreads();
        if (threadIdx.x == 0) {
            int lo[4], hi[4], local;
            const bool good = window_of(make_int4(box[0], box[1], box[2], box[3]), stride, window, shift, lo, &local) &
                              window_of(make_int4(box[4], box[5], box[6], box[7]), stride, window, shift, hi, &local);
            double total = 1.0;
            for (int x = 0; x < 4; ++x) {
                plan.lo[x] = lo[x];
                plan.dim[x] = hi[x] - lo[x] + 1;
                total *= static_cast<double>(plan.dim[x]);
            }
            plan.ok = good && total <= static_cast<double>(cells_cap);
            if (blockIdx.x == 0) {
                plan_out[set] = plan;
                const unsigned long long bits = (good ? 0 : kBadRange) | (plan.ok ? 0 : kNoGrid);
                if (bits) atomicOr(reinterpret_cast<unsigned long long *>(counts + 3), bits);
            }
        }
        __syncthreads();
    }
    if (!plan.ok) return;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    const int lane = threadIdx.x & 63;
    int cell = -1, local = 0;
    if (i < N) {
        int w[4];
        window_of(reinterpret_cast<const int4 *>(coords)[i], stride, window, shift, w, &local);
        cell = (((w[0] - plan.lo[0]) * plan.dim[1] + (w[1] - plan.lo[1])) * plan.dim[2] + (w[2] - plan.lo[2])) * plan.dim[3] +
               (w[3] - plan.lo[3]);
    }
    const int before = __shfl_up(cell, 1);
    const bool head = lane == 0 || before != cell;
    const unsigned long long heads = __ballot(head);
    const unsigned long long upto = heads & (lane == 63 ? ~0ull : ((2ull << lane) - 1));
    const int my_head = 63 - __clzll(static_cast<long long>(upto));
    const unsigned long long above = lane == 63 ? 0ull : heads & ~((2ull << lane) - 1);
    const int next = above ? __ffsll(static_cast<long long>(above)) - 1 : 64;
    int base = 0;
    if (head && cell >= 0) base = atomicAdd(&cells[cell], next - lane);
    base = __shfl(base, my_head);
    if (i < N) {
        const int slot = base + (lane - my_head);
        if (slot >= (1 << kSlotBits)) atomicOr(reinterpret_cast<unsigned long long *>(counts + 3), static_cast<unsigned long long>(kNoGrid));
        place[i] = make_int2(cell, (slot & ((1 << kSlotBits) - 1)) | (local << kSlotBits));
    }
}

// sum over the lanes before this one, by DPP moves, and over all lanes in the last
__device__ __forceinline__ uint64_t wave_scan(uint64_t x)
{
    auto add = [](uint64_t v, auto ctrl, auto rows) {
        const int lo = static_cast<int>(v), hi = static_cast<int>(v >> 32);
        const uint32_t l = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, lo, decltype(ctrl)::value, decltype(rows)::value, 0xf, true));
        const uint32_t h = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, hi, decltype(ctrl)::value, decltype(rows)::value, 0xf, true));
        return v + ((static_cast<uint64_t>(h) << 32) | l);
    };
    x = add(x, std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xf>{});      // row_shr 1, 2, 4, 8
    x = add(x, std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xf>{});
    x = add(x, std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xf>{});
    x = add(x, std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xf>{});
    x = add(x, std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});      // row_bcast15 into rows 1, 3
    return add(x, std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});   // row_bcast31 into rows 2, 3
}

__device__ __forceinline__ int64_t cells_of(const GridPlan &plan)
{
    return static_cast<int64_t>(plan.dim[0]) * plan.dim[1] * plan.dim[2] * plan.dim[3];
}

// what a workgroup's cells add up to
__global__ __launch_bounds__(kSumThreads) void grid_sums_kernel(GridSets sets, const GridPlan *__restrict__ plan,
                                                                const int32_t *__restrict__ cells, int64_t cells_cap,
                                                                CellSum *__restrict__ sums)
{
    const int set = blockIdx.y;
    if (!plan[set].ok || (sets.set[set].counts[3] & kNoGrid)) return;
    const int64_t total = cells_of(plan[set]);
    cells += set * cells_cap;
    sums += set * sum_groups(cells_cap);
    __shared__ CellSum part[kSumThreads / 64];
    for (int64_t group = blockIdx.x; group * kSumCells < total; group += gridDim.x) {
        const int64_t first = group * kSumCells;
        uint64_t sum = 0;
        int64_t squares = 0;
        int largest = 0;
#pragma unroll
        for (int e = 0; e < kSumCells / kSumThreads; ++e) {
            const int64_t c = first + e * kSumThreads + threadIdx.x;
            const int n = c < total ? cells[c] : 0;
            sum += cell_word(n);
            squares += static_cast<int64_t>(n) * n;
            largest = max(largest, n);
        }
        sum = wave_scan(sum);
        squares = static_cast<int64_t>(wave_scan(static_cast<uint64_t>(squares)));
        for (int off = 32; off > 0; off >>= 1) largest = max(largest, __shfl_xor(largest, off));
        if ((threadIdx.x & 63) == 63) part[threadIdx.x >> 6] = CellSum{sum, squares, largest, 0};
        __syncthreads();
        if (threadIdx.x == 0) {
            CellSum all = part[0];
            for (int w = 1; w < kSumThreads / 64; ++w) {
                all.before += part[w].before;
                all.squares += part[w].squares;
                all.largest = max(all.largest, part[w].largest);
            }
            sums[group] = all;
        }
        __syncthreads();
    }
}

// Every cell's first position, in the place of its count, and the windows: what the workgroups before this one add up to and
// a scan of its own cells.  (With window number and position of every cell in an array of its own a set took 72 bytes a voxel
// for its cells, not 24, and the placing read two of its words for a window's first voxel.)  The first workgroup of a set leaves
// the totals and the status word, also where the host reads them (or null).
__global__ __launch_bounds__(kSumThreads) void grid_starts_kernel(GridSets sets, const GridPlan *__restrict__ plan,
                                                                  int32_t *__restrict__ cells, int64_t cells_cap,
                                                                  const CellSum *__restrict__ sums, int64_t *host_counts)
{
    const int set = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int64_t *counts = sets.set[set].counts;
    const int64_t status = counts[3];
    const bool good = plan[set].ok && !(status & kNoGrid);
    const int64_t total = good ? cells_of(plan[set]) : 0;
    sums += set * sum_groups(cells_cap);
    __shared__ CellSum part[kSumThreads / 64];
    __shared__ uint64_t wave_sum[kSumThreads / 64];
    if (blockIdx.x == 0) {
        const int groups = static_cast<int>((total + kSumCells - 1) / kSumCells);
        CellSum all{0, 0, 0, 0};
        for (int g = threadIdx.x; g < groups; g += kSumThreads) {
            all.before += sums[g].before;
            all.squares += sums[g].squares;
            all.largest = max(all.largest, sums[g].largest);
        }
        all.before = wave_scan(all.before);
        all.squares = static_cast<int64_t>(wave_scan(static_cast<uint64_t>(all.squares)));
        for (int off = 32; off > 0; off >>= 1) all.largest = max(all.largest, __shfl_xor(all.largest, off));
        if (lane == 63) part[wave] = all;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int w = 1; w < kSumThreads / 64; ++w) {
                part[0].before += part[w].before;
                part[0].squares += part[w].squares;
                part[0].largest = max(part[0].largest, part[w].largest);
            }
            const int64_t totals[4] = {static_cast<int64_t>(part[0].before >> 32), part[0].squares, part[0].largest, status};
            for (int k = 0; k < 3 && good; ++k) counts[k] = totals[k];
            if (host_counts)
                for (int k = 0; k < 4; ++k) host_counts[4 * set + k] = totals[k];
        }
        __syncthreads();
    }
    int32_t *w2n = sets.set[set].w2n, *w_sizes = sets.set[set].w_sizes;
    cells += set * cells_cap;
    for (int64_t group = blockIdx.x; group * kSumCells < total; group += gridDim.x) {
        const int64_t first = group * kSumCells;
        uint64_t before = 0;
        for (int g = threadIdx.x; g < static_cast<int>(group); g += kSumThreads) before += sums[g].before;
        before = wave_scan(before);
        if (lane == 63) part[wave].before = before;
        // four neighbouring cells a thread
        int n[4];
        uint64_t own = 0;
        const int64_t mine = first + 4 * static_cast<int>(threadIdx.x);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            n[e] = mine + e < total ? cells[mine + e] : 0;
            own += cell_word(n[e]);
        }
        const uint64_t upto = wave_scan(own);
        if (lane == 63) wave_sum[wave] = upto;
        __syncthreads();
        uint64_t run = upto - own;
#pragma unroll
        for (int w = 0; w < kSumThreads / 64; ++w) run += part[w].before + (w < wave ? wave_sum[w] : 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int start = static_cast<int>(run & 0xffffffffu), rank = static_cast<int>(run >> 32);
            if (mine + e < total) cells[mine + e] = start;
            if (n[e] > 0) {
                w2n[rank] = start;
                w_sizes[rank] = n[e];
            }
            run += cell_word(n[e]);
        }
        __syncthreads();
    }
}

// every voxel to its window's segment (slot order)
__global__ __launch_bounds__(kThreads) void grid_place_kernel(const int2 *__restrict__ place, int64_t N, GridSets sets,
                                                              const GridPlan *__restrict__ plan,
                                                              const int32_t *__restrict__ cells, int64_t cells_cap,
                                                              uint64_t *__restrict__ keys)
{
    const int set = blockIdx.y;
    if (!plan[set].ok || (sets.set[set].counts[3] & kNoGrid)) return;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= N) return;
    cells += set * cells_cap;
    place += set * N;
    keys += set * N;
    const int2 p = place[i];
    const int slot = p.y & ((1 << kSlotBits) - 1);
    keys[cells[p.x] + slot] = (static_cast<uint64_t>(p.y >> kSlotBits) << 32) | static_cast<uint32_t>(i);
}

// One wavefront per window at a time: the window's voxels in (local id, row) order.  The rank of an element is
// the number of smaller ones, counted against every element of the window (a few dozen to a few hundred voxels).
__global__ __launch_bounds__(kThreads) void grid_order_kernel(const GridPlan *__restrict__ plan,
                                                              const uint64_t *__restrict__ keys, int64_t N, GridSets sets)
{
    const int set = blockIdx.y;
    const int32_t *w2n = sets.set[set].w2n, *w_sizes = sets.set[set].w_sizes;
    int32_t *n2n = sets.set[set].n2n, *w_w_id = sets.set[set].w_w_id;
    int64_t *counts = sets.set[set].counts;
    if (!plan[set].ok || (counts[3] & kNoGrid)) return;
    keys += set * N;
    constexpr int kOrderStage = 512;                       // keys of a window staged in LDS at a time, per wavefront
    __shared__ uint64_t stage_all[kThreads / 64][kOrderStage];
    uint64_t *stage = stage_all[threadIdx.x >> 6];
    const int lane = threadIdx.x & 63;
    const int W = static_cast<int>(counts[0]);
    const int waves = static_cast<int>(gridDim.x) * (kThreads / 64);
    // Two windows at a time: a wavefront's time is a chain of trips to memory (where a window lies, its keys), which both share (two
    // sets of 199,327 voxels 12.5 -> 10.8 us; four at a time 11.0).
    constexpr int kTogether = 2;
    for (int w0 = static_cast<int>(blockIdx.x) * (kThreads / 64) + (threadIdx.x >> 6); w0 < W; w0 += kTogether * waves) {
        int starts[kTogether], sizes[kTogether];
        uint64_t own[kTogether];
#pragma unroll
        for (int k = 0; k < kTogether; ++k) {
            const int w = min(w0 + k * waves, W - 1);
            starts[k] = w2n[w];
            sizes[k] = w0 + k * waves < W ? w_sizes[w] : 0;
        }
#pragma unroll
        for (int k = 0; k < kTogether; ++k) own[k] = lane < sizes[k] ? keys[starts[k] + lane] : ~0ULL;
#pragma unroll
        for (int k = 0; k < kTogether; ++k) {
            const int start = __builtin_amdgcn_readfirstlane(starts[k]), n = __builtin_amdgcn_readfirstlane(sizes[k]);
            if (n <= 64) {
                // one element per lane, the others read lane by lane
                const uint64_t mine = own[k];
                int rank = 0;
                for (int j = 0; j < n; ++j) {
                    const uint64_t other = (static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(mine >> 32), j))) << 32) |
                                           static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(mine), j));
                    rank += other < mine;
                }
                if (lane < n) {
                    n2n[start + rank] = static_cast<int32_t>(mine & 0xffffffffu);
                    w_w_id[start + rank] = static_cast<int32_t>(mine >> 32);
                }
                continue;
            }
            // larger windows: the keys staged in LDS, every lane ranks its elements against all of them; a window
            // beyond the staging area (only with many voxels of equal coordinates) is staged piece by piece per chunk
            auto stage_keys = [&](int base, int m) {
                __builtin_amdgcn_wave_barrier();
                for (int t = lane; t < m; t += 64) stage[t] = keys[start + base + t];
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            };
            const bool whole = n <= kOrderStage;
            if (whole) stage_keys(0, n);
            for (int first = 0; first < n; first += 64) {
                const int e = first + lane;
                const uint64_t mine = e < n ? (whole ? stage[e] : keys[start + e]) : ~0ULL;
                int rank = 0;
                for (int base = 0; base < n; base += kOrderStage) {
                    const int m = min(kOrderStage, n - base);
                    if (!whole) stage_keys(base, m);
#pragma unroll 4
                    for (int j = 0; j < m; ++j) rank += stage[j] < mine;
                }
                if (e < n) {
                    n2n[start + rank] = static_cast<int32_t>(mine & 0xffffffffu);
                    w_w_id[start + rank] = static_cast<int32_t>(mine >> 32);
                }
            }
        }
    }
}

// A thread per sorted position reads its voxel's row; the matrix leaves through LDS, a workgroup's rows in one piece (a
// thread per element divides by the columns and reads n2n nine times: 10.7 us for 199,327 x 9).  The add and the multiply
// stay separate roundings, as in the reference's tensor statement (sum, then scale).
__global__ __launch_bounds__(kThreads) void window_signals_kernel(
    const int32_t *__restrict__ w_w_id, const int32_t *__restrict__ n2n, const float *__restrict__ frac,
    const float *__restrict__ signals, int64_t signals_stride, int columns, int window, float xyz_scale,
    float other_scale, float *__restrict__ out, int64_t N)
{
#pragma clang fp contract(off)
    extern __shared__ float tile[];
    const int64_t p0 = static_cast<int64_t>(blockIdx.x) * kThreads, p = p0 + threadIdx.x;
    if (p < N) {
        float *to = tile + threadIdx.x * columns;
        const int64_t row = n2n[p];
        const int id = w_w_id[p];
        const int x = id / (window * window), rest = id - x * (window * window), y = rest / window, z = rest - y * window;
        to[0] = (static_cast<float>(x) + frac[row * 3]) * xyz_scale;
        to[1] = (static_cast<float>(y) + frac[row * 3 + 1]) * xyz_scale;
        to[2] = (static_cast<float>(z) + frac[row * 3 + 2]) * xyz_scale;
        const float *from = signals + row * signals_stride;
#pragma unroll 6
        for (int c = 3; c < columns; ++c) to[c] = from[c - 3] * other_scale;
    }
    __syncthreads();
    const int here = static_cast<int>(min(static_cast<int64_t>(kThreads), N - p0)) * columns;
    for (int t = threadIdx.x; t < here; t += kThreads) out[p0 * columns + t] = tile[t];
}

// The same for rows too wide for a workgroup's LDS: a thread per element.
__global__ __launch_bounds__(kThreads) void window_signals_wide_kernel(
    const int32_t *__restrict__ w_w_id, const int32_t *__restrict__ n2n, const float *__restrict__ frac,
    const float *__restrict__ signals, int64_t signals_stride, int columns, int window, float xyz_scale,
    float other_scale, float *__restrict__ out, int64_t N)
{
#pragma clang fp contract(off)
    const int64_t step = static_cast<int64_t>(gridDim.x) * kThreads;
    for (int64_t t = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; t < N * columns; t += step) {
        const int64_t p = t / columns, row = n2n[p];
        const int c = static_cast<int>(t - p * columns);
        if (c < 3) {
            const int id = w_w_id[p];
            const int cell = c == 0 ? id / (window * window) : c == 1 ? (id / window) % window : id % window;
            out[t] = (static_cast<float>(cell) + frac[row * 3 + c]) * xyz_scale;
        } else {
            out[t] = signals[row * signals_stride + (c - 3)] * other_scale;
        }
    }
}

// one thread per (sorted voxel, offset): binary search of key + delta in the sorted keys
__global__ __launch_bounds__(kThreads) void key_neighbours_kernel(const int64_t *__restrict__ sorted_keys,
                                                                  const int64_t *__restrict__ order, int64_t N,
                                                                  const int64_t *__restrict__ deltas, int M,
                                                                  int64_t *__restrict__ out)
{
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (t >= N * M) return;
    const int64_t i = t / M;
    const int d = static_cast<int>(t - i * M);
    const int64_t key = sorted_keys[i] + deltas[d];
    int64_t lo = 0, hi = N;   // first position whose key is not below `key`
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (sorted_keys[mid] < key) lo = mid + 1;
        else hi = mid;
    }
    const bool found = lo < N && sorted_keys[lo] == key;
    out[order[i] * M + d] = found ? order[lo] : N;
}

// one thread per cell (= window of the sort): mean of the members' signal rows, then the member nearest to it
constexpr int kMaxCellSignals = 16;
__global__ __launch_bounds__(kThreads) void cell_representatives_kernel(
    const int32_t *__restrict__ n2n, const int32_t *__restrict__ w2n, const int32_t *__restrict__ w_sizes, int64_t W,
    const float *__restrict__ signals, int64_t signals_stride, int S, int64_t *__restrict__ out)
{
#pragma clang fp contract(off)
    const int64_t w = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (w >= W) return;
    const int begin = w2n[w], size = w_sizes[w];
    float mean[kMaxCellSignals];
#pragma unroll
    for (int c = 0; c < kMaxCellSignals; ++c) mean[c] = 0.0f;
    for (int p = begin; p < begin + size; ++p) {
        const float *row = signals + static_cast<int64_t>(n2n[p]) * signals_stride;
#pragma unroll
        for (int c = 0; c < kMaxCellSignals; ++c)
            if (c < S) mean[c] += row[c];
    }
#pragma unroll
    for (int c = 0; c < kMaxCellSignals; ++c) mean[c] /= static_cast<float>(size);
    float best = INFINITY;
    int best_row = 0x7fffffff;
    for (int p = begin; p < begin + size; ++p) {
        const int r = n2n[p];
        const float *row = signals + static_cast<int64_t>(r) * signals_stride;
        float sq = 0.0f;
#pragma unroll
        for (int c = 0; c < kMaxCellSignals; ++c) {
            if (c < S) {
                const float d = row[c] - mean[c];
                sq += d * d;
            }
        }
        const float dist = sqrtf(sq);
        if (dist < best || (dist == best && r < best_row)) {
            best = dist;
            best_row = r;
        }
    }
    out[w] = best_row;
}

}  // namespace
}  // namespace s3d

extern "C" __attribute__((visibility("default"))) int s3d_cell_representatives(
    const int32_t *n2n, const int32_t *w2n, const int32_t *w_sizes, int64_t W, const float *signals,
    int64_t signals_stride, int32_t num_signals, int64_t *out, void *stream)
{
    using namespace s3d;
    if (W < 0 || num_signals < 1 || num_signals > kMaxCellSignals || signals_stride < num_signals)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_cell_representatives: W=%lld num_signals=%d (1..%d) signals_stride=%lld",
                    (long long)W, num_signals, kMaxCellSignals, (long long)signals_stride);
    if (W == 0) return S3D_OK;
    if (!n2n || !w2n || !w_sizes || !signals || !out)
        return fail(S3D_ERR_NULL_POINTER, "s3d_cell_representatives: null device pointer");
    const dim3 grid(static_cast<unsigned>(ceil_div(W, kThreads)));
    hipLaunchKernelGGL(cell_representatives_kernel, grid, dim3(kThreads), 0, static_cast<hipStream_t>(stream), n2n, w2n,
                       w_sizes, W, signals, signals_stride, num_signals, out);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

extern "C" __attribute__((visibility("default"))) int s3d_key_neighbours(const int64_t *sorted_keys,
                                                                          const int64_t *order, int64_t N,
                                                                          const int64_t *deltas, int32_t M,
                                                                          int64_t *out, void *stream)
{
    using namespace s3d;
    if (N < 0 || M < 1 || M > 1024 || N * static_cast<int64_t>(M) > 0x3fffffffffLL)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_key_neighbours: N=%lld M=%d out of range", (long long)N, M);
    if (N == 0) return S3D_OK;
    if (!sorted_keys || !order || !deltas || !out)
        return fail(S3D_ERR_NULL_POINTER, "s3d_key_neighbours: null device pointer");
    const dim3 grid(static_cast<unsigned>(ceil_div(N * M, kThreads)));
    hipLaunchKernelGGL(key_neighbours_kernel, grid, dim3(kThreads), 0, static_cast<hipStream_t>(stream), sorted_keys,
                       order, N, deltas, M, out);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

extern "C" __attribute__((visibility("default"))) int s3d_window_signals(
    const int32_t *w_w_id, const int32_t *n2n, const float *frac, const float *signals, int64_t signals_stride,
    int32_t num_signals, int32_t window, float xyz_scale, float other_scale, float *out, int64_t N, void *stream)
{
    using namespace s3d;
    if (N < 0 || num_signals < 0 || window < 1 || window > 10 || (num_signals > 0 && signals_stride < num_signals))
        return fail(S3D_ERR_BAD_SHAPE, "s3d_window_signals: N=%lld num_signals=%d signals_stride=%lld window=%d",
                    (long long)N, num_signals, (long long)signals_stride, window);
    if (N == 0) return S3D_OK;
    if (!w_w_id || !n2n || !frac || !out || (num_signals > 0 && !signals))
        return fail(S3D_ERR_NULL_POINTER, "s3d_window_signals: null device pointer");
    const int columns = 3 + num_signals;
    // a row per thread while a workgroup's rows fit half of the LDS of a launch without special attributes
    if (columns > 8192 / kThreads) {
        const int64_t groups = ceil_div(N * columns, kThreads);
        hipLaunchKernelGGL(window_signals_wide_kernel, dim3(static_cast<unsigned>(groups < 65536 ? groups : 65536)), dim3(kThreads), 0,
                           static_cast<hipStream_t>(stream), w_w_id, n2n, frac, signals, signals_stride, columns, window, xyz_scale,
                           other_scale, out, N);
        S3D_HIP_CHECK(hipGetLastError());
        return S3D_OK;
    }
    const dim3 grid(static_cast<unsigned>(ceil_div(N, kThreads)));
    const uint32_t lds = kThreads * columns * sizeof(float);
    hipLaunchKernelGGL(window_signals_kernel, grid, dim3(kThreads), lds, static_cast<hipStream_t>(stream), w_w_id, n2n,
                       frac, signals, signals_stride, columns, window, xyz_scale, other_scale, out, N);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

extern "C" __attribute__((visibility("default"))) size_t s3d_window_index_workspace_bytes(int64_t N)
{
    return s3d::make_layout(N).total;
}

extern "C" __attribute__((visibility("default"))) int s3d_window_index(const int32_t *coords, int64_t N, int32_t stride, int32_t window,
                                int32_t shift, int32_t *n2n, int32_t *w_w_id, int32_t *w_sizes,
                                int32_t *w2n, int64_t *counts, void *workspace,
                                size_t workspace_bytes, void *stream)
{
    using namespace s3d;
    if (N < 0 || N > 0x7fffffffLL)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_window_index: N=%lld out of range", (long long)N);
    if (stride < 1 || window < 1 || window > 10 || shift < 0 || shift >= window)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_window_index: stride=%d window=%d shift=%d (need stride>=1, "
                    "1<=window<=10, 0<=shift<window)", stride, window, shift);
    if (!counts) return fail(S3D_ERR_NULL_POINTER, "s3d_window_index: counts is null");
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(init_counts_kernel, dim3(1), dim3(64), 0, s, counts);
    S3D_HIP_CHECK(hipGetLastError());
    if (N == 0) return S3D_OK;
    if (!coords || !n2n || !w_w_id || !w_sizes || !w2n || !workspace)
        return fail(S3D_ERR_NULL_POINTER, "s3d_window_index: null device pointer");
    if (reinterpret_cast<uintptr_t>(coords) % 16 != 0)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_window_index: coords must be 16-byte aligned");
    const Layout L = make_layout(N);
    if (workspace_bytes < L.total)
        return fail(S3D_ERR_WORKSPACE, "s3d_window_index: workspace %zu B < required %zu B",
                    workspace_bytes, L.total);
    char *base = static_cast<char *>(workspace);
    uint64_t *keys_in = reinterpret_cast<uint64_t *>(base + L.keys_in);
    uint64_t *keys_out = reinterpret_cast<uint64_t *>(base + L.keys_out);
    int32_t *vals_in = reinterpret_cast<int32_t *>(base + L.vals_in);
    int32_t *flags = reinterpret_cast<int32_t *>(base + L.flags);
    int32_t *ranks = reinterpret_cast<int32_t *>(base + L.ranks);
    void *temp = base + L.temp;
    size_t temp_bytes = L.temp_bytes;

    const dim3 grid(static_cast<unsigned>(ceil_div(N, kThreads)));
    hipLaunchKernelGGL(build_keys_kernel, grid, dim3(kThreads), 0, s, coords, N, stride, window,
                       shift, keys_in, vals_in, counts);
    S3D_HIP_CHECK(hipGetLastError());
    S3D_HIP_CHECK(rocprim::radix_sort_pairs(temp, temp_bytes, keys_in, keys_out, vals_in, n2n,
                                            static_cast<size_t>(N), 0, 64, s));
    hipLaunchKernelGGL(flag_kernel, grid, dim3(kThreads), 0, s, keys_out, N, flags, w_w_id);
    S3D_HIP_CHECK(hipGetLastError());
    temp_bytes = L.temp_bytes;
    S3D_HIP_CHECK(rocprim::inclusive_scan(temp, temp_bytes, flags, ranks, static_cast<size_t>(N),
                                          rocprim::plus<int32_t>(), s));
    hipLaunchKernelGGL(segment_start_kernel, grid, dim3(kThreads), 0, s, flags, ranks, N, w2n, counts);
    S3D_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(segment_size_kernel, grid, dim3(kThreads), 0, s, w2n, N, w_sizes, counts);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

extern "C" __attribute__((visibility("default"))) size_t s3d_window_indices_workspace_bytes(int64_t N, int32_t num_sets)
{
    return num_sets < 1 || num_sets > s3d::kMaxSets ? 0 : s3d::make_grid_layout(N, num_sets).total;
}

namespace s3d {
namespace {

// counted, finished: recorded behind the launch that leaves the counts in host_counts (or null, as that), and behind the last
int window_indices(const int32_t *coords, int64_t N, int32_t stride, const s3d_window_index_set *jobs, int32_t num_sets,
                   int64_t *host_counts, hipEvent_t counted, hipEvent_t finished, void *workspace, size_t workspace_bytes, void *stream)
{
    if (N < 0 || N > 0x7fffffffLL || num_sets < 1 || num_sets > kMaxSets || N * num_sets > 0xffffffffLL)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_window_indices: N=%lld voxels, %d sets (1..%d)", (long long)N, num_sets, kMaxSets);
    if (!jobs) return fail(S3D_ERR_NULL_POINTER, "s3d_window_indices: sets is null");
    GridSets sets{};
    sets.num = num_sets;
    for (int i = 0; i < num_sets; ++i) {
        const s3d_window_index_set &j = jobs[i];
        if (stride < 1 || j.window < 1 || j.window > 10 || j.shift < 0 || j.shift >= j.window)
            return fail(S3D_ERR_BAD_SHAPE, "s3d_window_indices: stride=%d window=%d shift=%d (need stride>=1, "
                        "1<=window<=10, 0<=shift<window)", stride, j.window, j.shift);
        if (!j.counts) return fail(S3D_ERR_NULL_POINTER, "s3d_window_indices: counts is null");
        if (N > 0 && (!j.n2n || !j.w_w_id || !j.w_sizes || !j.w2n))
            return fail(S3D_ERR_NULL_POINTER, "s3d_window_indices: null device pointer");
        sets.set[i] = GridSet{j.window, j.shift, j.n2n, j.w_w_id, j.w_sizes, j.w2n, j.counts};
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (N == 0) {
        for (int i = 0; i < num_sets; ++i) hipLaunchKernelGGL(init_counts_kernel, dim3(1), dim3(64), 0, s, sets.set[i].counts);
        S3D_HIP_CHECK(hipGetLastError());
        for (int i = 0; host_counts && i < 4 * num_sets; ++i) host_counts[i] = 0;
        for (hipEvent_t e : {counted, finished})
            if (e) S3D_HIP_CHECK(hipEventRecord(e, s));
        return S3D_OK;
    }
    if (!coords || !workspace) return fail(S3D_ERR_NULL_POINTER, "s3d_window_indices: null device pointer");
    if (reinterpret_cast<uintptr_t>(coords) % 16 != 0)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_window_indices: coords must be 16-byte aligned");
    const GridLayout L = make_grid_layout(N, num_sets);
    if (workspace_bytes < L.total)
        return fail(S3D_ERR_WORKSPACE, "s3d_window_indices: workspace %zu B < required %zu B", workspace_bytes, L.total);
    char *base = static_cast<char *>(workspace);
    GridPlan *plan = reinterpret_cast<GridPlan *>(base + L.plan);
    int32_t *partials = reinterpret_cast<int32_t *>(base + L.partials);
    int32_t *cells = reinterpret_cast<int32_t *>(base + L.cells);
    int2 *place = reinterpret_cast<int2 *>(base + L.place);
    uint64_t *keys = reinterpret_cast<uint64_t *>(base + L.keys);
    CellSum *sums = reinterpret_cast<CellSum *>(base + L.sums);
    const int64_t num_cells = L.cells_cap * num_sets;
    const unsigned per_set = static_cast<unsigned>(num_sets);
    const dim3 grid(static_cast<unsigned>(ceil_div(N, kThreads)), per_set);
    hipLaunchKernelGGL(grid_bbox_kernel, dim3(kGridBoxes + kGridZeros), dim3(kThreads), 0, s, coords, N, sets, partials, cells, num_cells);
    S3D_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(grid_count_kernel, grid, dim3(kThreads), 0, s, coords, N, stride, sets, partials, L.cells_cap, plan,
                       cells, place);
    S3D_HIP_CHECK(hipGetLastError());
    // (a third of the runs there may be: most lattices are smaller, and a workgroup takes another run where one is not)
    const dim3 sum_grid(static_cast<unsigned>(ceil_div(L.cells_cap, 3 * kSumCells)), per_set);
    hipLaunchKernelGGL(grid_sums_kernel, sum_grid, dim3(kSumThreads), 0, s, sets, plan, cells, L.cells_cap, sums);
    hipLaunchKernelGGL(grid_starts_kernel, sum_grid, dim3(kSumThreads), 0, s, sets, plan, cells, L.cells_cap, sums, host_counts);
    S3D_HIP_CHECK(hipGetLastError());
    if (counted) S3D_HIP_CHECK(hipEventRecord(counted, s));
    hipLaunchKernelGGL(grid_place_kernel, grid, dim3(kThreads), 0, s, place, N, sets, plan, cells, L.cells_cap, keys);
    S3D_HIP_CHECK(hipGetLastError());
    // about two windows per wavefront if the windows hold 16 voxels on average, more in turn otherwise
    int64_t order_blocks = ceil_div(N, 128);
    order_blocks = order_blocks < 32 ? 32 : (order_blocks > 4096 ? 4096 : order_blocks);
    hipLaunchKernelGGL(grid_order_kernel, dim3(static_cast<unsigned>(order_blocks), per_set), dim3(kThreads), 0, s, plan, keys,
                       N, sets);
    S3D_HIP_CHECK(hipGetLastError());
    if (finished) S3D_HIP_CHECK(hipEventRecord(finished, s));
    return S3D_OK;
}

}  // namespace
}  // namespace s3d

extern "C" __attribute__((visibility("default"))) int s3d_window_indices(
    const int32_t *coords, int64_t N, int32_t stride, const s3d_window_index_set *sets, int32_t num_sets, void *workspace,
    size_t workspace_bytes, void *stream)
{
    return s3d::window_indices(coords, N, stride, sets, num_sets, nullptr, nullptr, nullptr, workspace, workspace_bytes, stream);
}

namespace s3d {
namespace {

// the sets, and the calling thread waits: for the counts, or for all that the call launched
int waited_window_indices(const char *name, bool all, const int32_t *coords, int64_t N, int32_t stride, const s3d_window_index_set *sets,
                          int32_t num_sets, int64_t *host_counts, void *workspace, size_t workspace_bytes, void *stream)
{
    if (!host_counts) return fail(S3D_ERR_NULL_POINTER, "%s: host_counts is null", name);
    hipEvent_t there = nullptr;
    S3D_HIP_CHECK(hipEventCreateWithFlags(&there, hipEventDisableTiming));
    int rc = window_indices(coords, N, stride, sets, num_sets, host_counts, all ? nullptr : there, all ? there : nullptr, workspace,
                            workspace_bytes, stream);
    // (after an error between the launches the event may not have been recorded: host_counts is the caller's again all the same)
    const hipError_t waited = rc == S3D_OK ? hipEventSynchronize(there) : hipStreamSynchronize(static_cast<hipStream_t>(stream));
    if (rc == S3D_OK && waited != hipSuccess) rc = hip_fail(waited, "hipEventSynchronize");
    (void)hipEventDestroy(there);
    return rc;
}

}  // namespace
}  // namespace s3d

extern "C" __attribute__((visibility("default"))) int s3d_window_indices_counted(
    const int32_t *coords, int64_t N, int32_t stride, const s3d_window_index_set *sets, int32_t num_sets, int64_t *host_counts,
    void *workspace, size_t workspace_bytes, void *stream)
{
    return s3d::waited_window_indices("s3d_window_indices_counted", false, coords, N, stride, sets, num_sets, host_counts, workspace,
                                      workspace_bytes, stream);
}

extern "C" __attribute__((visibility("default"))) int s3d_window_indices_finished(
    const int32_t *coords, int64_t N, int32_t stride, const s3d_window_index_set *sets, int32_t num_sets, int64_t *host_counts,
    void *workspace, size_t workspace_bytes, void *stream)
{
    return s3d::waited_window_indices("s3d_window_indices_finished", true, coords, N, stride, sets, num_sets, host_counts, workspace,
                                      workspace_bytes, stream);
}

extern "C" __attribute__((visibility("default"))) size_t s3d_window_index_grid_workspace_bytes(int64_t N)
{
    return s3d_window_indices_workspace_bytes(N, 1);
}

extern "C" __attribute__((visibility("default"))) int s3d_window_index_grid(
    const int32_t *coords, int64_t N, int32_t stride, int32_t window, int32_t shift, int32_t *n2n, int32_t *w_w_id,
    int32_t *w_sizes, int32_t *w2n, int64_t *counts, void *workspace, size_t workspace_bytes, void *stream)
{
    const s3d_window_index_set set{n2n, w_w_id, w_sizes, w2n, counts, window, shift};
    return s3d_window_indices(coords, N, stride, &set, 1, workspace, workspace_bytes, stream);
}
