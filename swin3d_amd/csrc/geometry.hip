// The small steps of a level's geometry, a launch each where the tensor statements take three to nine (gfx950): what bounds
// them on a small scan is the host, some six to ten microseconds a launch.
#include "s3d_common.h"

namespace s3d {
namespace {

constexpr int kThreads = 256;

// Ends of the batch elements in one or two columns of ascending batch ids.
struct SegmentColumns {
    const int32_t *batch[2];
    int64_t stride[2], N[2];
};

// A wavefront looks for one end, 64 places at a time (a thread's search by halves was a chain of fifteen loads); both columns of a
// query in one launch.  A network on 25,013 voxels: sixteen launches of 3.3 us before, eight of 1.8 now.
__global__ __launch_bounds__(kThreads) void segment_ends_kernel(SegmentColumns columns, int count, int B, int32_t *__restrict__ out)
{
    const int lane = threadIdx.x & 63, step = static_cast<int>(gridDim.x) * (kThreads / 64);
    for (int64_t at = static_cast<int>(blockIdx.x) * (kThreads / 64) + static_cast<int>(threadIdx.x) / 64; at < static_cast<int64_t>(count) * B; at += step) {
        const bool second = at >= B;
        const int b = static_cast<int>(second ? at - B : at);
        const int32_t *batch = second ? columns.batch[1] : columns.batch[0];
        const int64_t stride = second ? columns.stride[1] : columns.stride[0];
        int64_t lo = 0, hi = second ? columns.N[1] : columns.N[0];
        while (lo < hi) {      // the end is from lo to hi
            const int64_t piece = (hi - lo + 63) / 64, probe = min(lo + (lane + 1) * piece, hi) - 1;
            const int below = __popcll(__ballot(batch[probe * stride] <= b));
            const int64_t first = lo + below * piece;
            hi = below == 64 ? hi : min(first + piece, hi) - 1;
            lo = min(first, hi);
        }
        if (lane == 0) out[at] = static_cast<int32_t>(lo);
    }
}

// The voxels by their packed coordinates: an open table of at least twice as many slots, four neighbours in z side by side.
// Of voxels with the same coordinates the first row counts.  Bound by the places of the table that a neighbour's look-up reads;
// a group of four is 64 bytes, so that a voxel's nine columns read nine to eighteen groups.  Measured with the list's
// allocation: 626,507 voxels of a surface in ascending order 229 us, by windows 252, in no order 380; 156,509 69 to 83; 1,568 15
// (sorting the keys and a search for each neighbour: 438, 443, 468; 140 to 148; 42).
struct VoxelSlot {
    int64_t key;
    int32_t row, unused;
};
constexpr int64_t kNoKey = INT64_MIN;

// (linear in the coordinates: a neighbour's key is the voxel's and a constant)
__device__ __forceinline__ int64_t packed_key(int4 c, int field)
{
    const int64_t bias = int64_t(1) << (field - 1);
    return (((static_cast<int64_t>(c.x) * (bias << 1) + (c.y + bias)) * (bias << 1)) + (c.z + bias)) * (bias << 1) + (c.w + bias);
}
__device__ __forceinline__ uint32_t first_slot(int64_t key, int bits)
{
    const uint64_t group = (static_cast<uint64_t>(key) >> 2) * 0x9E3779B97F4A7C15ull >> (64 - (bits - 2));
    return static_cast<uint32_t>(group) << 2 | (static_cast<uint32_t>(key) & 3u);
}

__global__ __launch_bounds__(kThreads) void voxel_table_clear_kernel(VoxelSlot *__restrict__ table, int64_t slots)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i < slots) table[i] = VoxelSlot{kNoKey, 0x7fffffff, 0};
}

__global__ __launch_bounds__(kThreads) void voxel_table_fill_kernel(const int4 *__restrict__ coords, int64_t N, int field,
                                                                    VoxelSlot *__restrict__ table, int bits)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= N) return;
    const int64_t key = packed_key(coords[i], field);
    const uint32_t mask = (1u << bits) - 1;
    // (at most half of the slots are taken: the walk ends)
    for (uint32_t at = first_slot(key, bits);; at = (at + 1) & mask) {
        const int64_t there = static_cast<int64_t>(atomicCAS(reinterpret_cast<unsigned long long *>(&table[at].key),
                                                             static_cast<unsigned long long>(kNoKey), static_cast<unsigned long long>(key)));
        if (there != kNoKey && there != key) continue;
        atomicMin(&table[at].row, static_cast<int32_t>(i));
        return;
    }
}

// A thread looks up three neighbours of a voxel, one above the other in z.
constexpr int kStemVoxels = 64, kStemThreads = 9 * kStemVoxels;

__global__ __launch_bounds__(kStemThreads) void voxel_neighbours_kernel(const int4 *__restrict__ coords, int64_t N, int field, int64_t stride,
                                                                    const VoxelSlot *__restrict__ table, int bits, int64_t *__restrict__ out)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kStemVoxels + threadIdx.x / 9;
    const int xy = static_cast<int>(threadIdx.x % 9);
    if (i >= N) return;
    const uint32_t mask = (1u << bits) - 1;
    const int64_t key = packed_key(coords[i], field) + (((static_cast<int64_t>(xy / 3 - 1) << field) + (xy % 3 - 1)) << field) * stride;
    uint32_t at[3];
    VoxelSlot slot[3];
#pragma unroll
    for (int z = 0; z < 3; ++z) {   // (three loads on their way before the first is waited for)
        at[z] = first_slot(key + (z - 1) * stride, bits);
        slot[z] = table[at[z]];
    }
#pragma unroll
    for (int z = 0; z < 3; ++z) {
        const int64_t wanted = key + (z - 1) * stride;
        while (slot[z].key != kNoKey && slot[z].key != wanted) {
            at[z] = (at[z] + 1) & mask;
            slot[z] = table[at[z]];
        }
        out[i * 27 + xy * 3 + z] = slot[z].key == kNoKey ? N : slot[z].row;
    }
}

// Rows of `width` words side by side, zeros for row n.  Bound by the work a word: a word a lane, so that a wavefront writes
// one run and reads a few rows, and a lane's row and place in it move on by additions.  27 rows of 9 for 626,507 voxels:
// fp16 0.20 ms, fp32 0.25 (an index into a copy with the row of zeros: 0.39, 0.44); of 6: 0.14, 0.18 (0.27, 0.31).
constexpr int kGatherRows = 512;
constexpr int32_t kZeroRow = -1, kNoRow = -2;

template <typename Word>
__global__ __launch_bounds__(kThreads) void gather_rows_kernel(const Word *__restrict__ from, int64_t n, const int64_t *__restrict__ rows,
                                                               int64_t M, int width, Word nan, Word *__restrict__ out)
{
    __shared__ int32_t word_of[kGatherRows];
    const int64_t first = static_cast<int64_t>(blockIdx.x) * kGatherRows;
    const int here = static_cast<int>(min(int64_t(kGatherRows), M - first));
    for (int r = threadIdx.x; r < here; r += kThreads) {
        int64_t row = rows[first + r];
        if (row < 0) row += n + 1;   // (counted from behind the row of zeros, as an index is)
        word_of[r] = row < 0 || row > n ? kNoRow : row == n ? kZeroRow : static_cast<int32_t>(row * width);
    }
    __syncthreads();
    const int words = here * width, rows_on = kThreads / width, words_on = kThreads % width;
    int r = threadIdx.x / width, c = threadIdx.x % width;
    Word *to = out + first * width;
#pragma unroll 4
    for (int e = threadIdx.x; e < words; e += kThreads) {
        const int32_t word = word_of[r];
        Word value = word == kNoRow ? nan : Word(0);
        if (word >= 0) value = from[static_cast<uint32_t>(word + c)];
        to[e] = value;
        r += rows_on, c += words_on;
        if (c >= width) c -= width, ++r;
    }
}

int voxel_table_bits(int64_t N)
{
    int bits = 4;
    while ((int64_t(1) << bits) < 2 * N) ++bits;
    return bits;
}

// Sixteen lanes a cell (= window of the sort).  The mean of the members' signal rows, a column per lane, members in sorted
// order; then the member nearest to it, a member per lane, columns in order; then what the level above is made of: the
// cell's coordinates and the chosen member's signals.
constexpr int kLanes = 16;
__global__ __launch_bounds__(kThreads) void pool_cells_kernel(
    const int32_t *__restrict__ n2n, const int32_t *__restrict__ w2n, const int32_t *__restrict__ w_sizes, int64_t W,
    const int4 *__restrict__ coords, int step, const float *__restrict__ signals, int64_t stride, int S,
    int64_t *__restrict__ pick, int4 *__restrict__ out_coords, float *__restrict__ out_signals)
{
#pragma clang fp contract(off)
    const int t = threadIdx.x % kLanes;
    const int64_t w_raw = (static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x) / kLanes, w = min(w_raw, W - 1);
    const int begin = w2n[w], size = w_sizes[w];
    float mean = 0.0f;
    for (int p0 = 0; p0 < size; p0 += kLanes) {
        const int row = n2n[begin + min(p0 + t, size - 1)];
        for (int m = 0; m < min(kLanes, size - p0); ++m) {
            const int64_t from = __shfl(row, m, kLanes);
            if (t < S) mean += signals[from * stride + t];
        }
    }
    mean /= static_cast<float>(size);
    float best = INFINITY;
    int best_row = 0x7fffffff;
    for (int p0 = 0; p0 < size; p0 += kLanes) {
        const int row = n2n[begin + min(p0 + t, size - 1)];
        float sq = 0.0f;
        for (int c = 0; c < S; ++c) {
            const float d = signals[static_cast<int64_t>(row) * stride + c] - __shfl(mean, c, kLanes);
            sq += d * d;
        }
        const float dist = sqrtf(sq);
        if (p0 + t < size && (dist < best || (dist == best && row < best_row))) {
            best = dist;
            best_row = row;
        }
    }
#pragma unroll
    for (int other = 1; other < kLanes; other <<= 1) {
        const float d = __shfl_xor(best, other, kLanes);
        const int r = __shfl_xor(best_row, other, kLanes);
        if (d < best || (d == best && r < best_row)) {
            best = d;
            best_row = r;
        }
    }
    if (w_raw >= W) return;
    if (t == 0) {
        pick[w] = best_row;
        const int4 c = coords[n2n[begin]];
        auto down = [&](int x) { return (x >= 0 ? x / step : -((-x + step - 1) / step)) * step; };
        // (no member is nearest where a signal is NaN: a batch that no window index takes says so at the level above, at the
        // wait which that level has anyway)
        out_coords[w] = make_int4(best_row == 0x7fffffff ? -1 : c.x, down(c.y), down(c.z), down(c.w));
    }
    if (t < S) out_signals[w * S + t] = best_row == 0x7fffffff ? __int_as_float(0x7fc00000) : signals[static_cast<int64_t>(best_row) * stride + t];
}

// As window_signals_kernel, from what a level holds: voxels and the points' signals (batch, x, y, z in voxels, others).
// The position inside the voxel is a difference times the stride's reciprocal, as the framework divides by a number.
__global__ __launch_bounds__(kThreads) void level_signals_kernel(
    const int32_t *__restrict__ w_w_id, const int32_t *__restrict__ n2n, const int4 *__restrict__ coords, float inv_stride,
    const float *__restrict__ signals, int64_t signals_stride, int columns, int window, float xyz_scale, float other_scale,
    float *__restrict__ out, int64_t N)
{
#pragma clang fp contract(off)
    extern __shared__ float tile[];
    const int64_t p0 = static_cast<int64_t>(blockIdx.x) * kThreads, p = p0 + threadIdx.x;
    if (p < N) {
        float *to = tile + threadIdx.x * columns;
        const int64_t row = n2n[p];
        const int id = w_w_id[p];
        const int x = id / (window * window), rest = id - x * (window * window), y = rest / window, z = rest - y * window;
        const int4 c = coords[row];
        const float *from = signals + row * signals_stride;
        to[0] = (static_cast<float>(x) + (from[1] - static_cast<float>(c.y)) * inv_stride) * xyz_scale;
        to[1] = (static_cast<float>(y) + (from[2] - static_cast<float>(c.z)) * inv_stride) * xyz_scale;
        to[2] = (static_cast<float>(z) + (from[3] - static_cast<float>(c.w)) * inv_stride) * xyz_scale;
#pragma unroll 6
        for (int k = 3; k < columns; ++k) to[k] = from[k + 1] * other_scale;
    }
    __syncthreads();
    const int here = static_cast<int>(min(static_cast<int64_t>(kThreads), N - p0)) * columns;
    for (int t = threadIdx.x; t < here; t += kThreads) out[p0 * columns + t] = tile[t];
}

int launch_segment_ends(const SegmentColumns &columns, int count, int B, int32_t *out, hipStream_t stream)
{
    // (a launch has at most 2^32 threads, and an end has 64)
    const int64_t blocks = ceil_div(static_cast<int64_t>(count) * B, kThreads / 64);
    hipLaunchKernelGGL(segment_ends_kernel, dim3(static_cast<unsigned>(blocks < (1 << 16) ? blocks : 1 << 16)), dim3(kThreads), 0, stream, columns, count, B, out);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

}  // namespace
}  // namespace s3d

extern "C" __attribute__((visibility("default"))) int s3d_segment_ends_of_two(const int32_t *first, int64_t first_stride, int64_t first_N,
                                                                              const int32_t *second, int64_t second_stride, int64_t second_N,
                                                                              int32_t B, int32_t *out, void *stream)
{
    using namespace s3d;
    if (first_N < 0 || first_N > 0x7fffffffLL || second_N < 0 || second_N > 0x7fffffffLL || B < 0 || B > 0x3fffffff || first_stride < 1 || second_stride < 1)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_segment_ends_of_two: N=%lld, %lld B=%d strides=%lld, %lld", (long long)first_N, (long long)second_N, B,
                    (long long)first_stride, (long long)second_stride);
    if (B == 0) return S3D_OK;
    if (!out || (first_N > 0 && !first) || (second_N > 0 && !second)) return fail(S3D_ERR_NULL_POINTER, "s3d_segment_ends_of_two: null device pointer");
    return launch_segment_ends({{first, second}, {first_stride, second_stride}, {first_N, second_N}}, 2, B, out, static_cast<hipStream_t>(stream));
}

extern "C" __attribute__((visibility("default"))) int s3d_segment_ends(const int32_t *batch, int64_t stride, int64_t N, int32_t B,
                                                                       int32_t *out, void *stream)
{
    using namespace s3d;
    if (N < 0 || N > 0x7fffffffLL || B < 0 || stride < 1) return fail(S3D_ERR_BAD_SHAPE, "s3d_segment_ends: N=%lld B=%d stride=%lld", (long long)N, B, (long long)stride);
    if (B == 0) return S3D_OK;
    if (!out || (N > 0 && !batch)) return fail(S3D_ERR_NULL_POINTER, "s3d_segment_ends: null device pointer");
    return launch_segment_ends({{batch, nullptr}, {stride, 1}, {N, 0}}, 1, B, out, static_cast<hipStream_t>(stream));
}

extern "C" __attribute__((visibility("default"))) size_t s3d_voxel_neighbours_workspace_bytes(int64_t N)
{
    using namespace s3d;
    return N < 0 || N > 0x3fffffff ? 0 : (sizeof(VoxelSlot) << voxel_table_bits(N));
}

extern "C" __attribute__((visibility("default"))) int s3d_voxel_neighbours(const int32_t *coords, int64_t N, int32_t field, int32_t stride,
                                                                           int64_t *out, void *workspace, size_t workspace_bytes, void *stream)
{
    using namespace s3d;
    if (N < 0 || N > 0x3fffffff || field < 2 || field > 20 || stride < 1)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_voxel_neighbours: N=%lld field=%d (2..20 bits) stride=%d", (long long)N, field, stride);
    if (N == 0) return S3D_OK;
    if (!coords || !out) return fail(S3D_ERR_NULL_POINTER, "s3d_voxel_neighbours: null device pointer");
    if (reinterpret_cast<uintptr_t>(coords) % 16 != 0 || reinterpret_cast<uintptr_t>(workspace) % 16 != 0)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_voxel_neighbours: coords and workspace must be 16-byte aligned");
    const size_t need = s3d_voxel_neighbours_workspace_bytes(N);
    if (!workspace || workspace_bytes < need)
        return fail(S3D_ERR_WORKSPACE, "s3d_voxel_neighbours: workspace %zu B < required %zu B", workspace ? workspace_bytes : size_t(0), need);
    const int bits = voxel_table_bits(N);
    const int64_t slots = int64_t(1) << bits;
    VoxelSlot *table = static_cast<VoxelSlot *>(workspace);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int4 *voxels = reinterpret_cast<const int4 *>(coords);
    hipLaunchKernelGGL(voxel_table_clear_kernel, dim3(static_cast<unsigned>(ceil_div(slots, kThreads))), dim3(kThreads), 0, s, table, slots);
    hipLaunchKernelGGL(voxel_table_fill_kernel, dim3(static_cast<unsigned>(ceil_div(N, kThreads))), dim3(kThreads), 0, s, voxels, N, field, table, bits);
    hipLaunchKernelGGL(voxel_neighbours_kernel, dim3(static_cast<unsigned>(ceil_div(N, kStemVoxels))), dim3(kStemThreads), 0, s, voxels, N,
                       field, static_cast<int64_t>(stride), table, bits, out);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

extern "C" __attribute__((visibility("default"))) int s3d_pool_cells(
    const int32_t *n2n, const int32_t *w2n, const int32_t *w_sizes, int64_t W, const int32_t *coords, int32_t step,
    const float *signals, int64_t signals_stride, int32_t num_signals, int64_t *pick, int32_t *out_coords, float *out_signals,
    void *stream)
{
    using namespace s3d;
    if (W < 0 || step < 1 || num_signals < 1 || num_signals > kLanes || signals_stride < num_signals)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_pool_cells: W=%lld step=%d num_signals=%d (1..%d) signals_stride=%lld", (long long)W, step,
                    num_signals, kLanes, (long long)signals_stride);
    if (W == 0) return S3D_OK;
    if (!n2n || !w2n || !w_sizes || !coords || !signals || !pick || !out_coords || !out_signals)
        return fail(S3D_ERR_NULL_POINTER, "s3d_pool_cells: null device pointer");
    if (reinterpret_cast<uintptr_t>(coords) % 16 != 0 || reinterpret_cast<uintptr_t>(out_coords) % 16 != 0)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_pool_cells: coordinates must be 16-byte aligned");
    hipLaunchKernelGGL(pool_cells_kernel, dim3(static_cast<unsigned>(ceil_div(W * kLanes, kThreads))), dim3(kThreads), 0,
                       static_cast<hipStream_t>(stream), n2n, w2n, w_sizes, W, reinterpret_cast<const int4 *>(coords), step, signals,
                       signals_stride, num_signals, pick, reinterpret_cast<int4 *>(out_coords), out_signals);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

extern "C" __attribute__((visibility("default"))) int s3d_level_signals(
    const int32_t *w_w_id, const int32_t *n2n, const int32_t *coords, int32_t stride, const float *signals, int64_t signals_stride,
    int32_t num_signals, int32_t window, float xyz_scale, float other_scale, float *out, int64_t N, void *stream)
{
    using namespace s3d;
    if (N < 0 || stride < 1 || num_signals < 0 || num_signals > 29 || window < 1 || window > 10 || signals_stride < 4 + num_signals)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_level_signals: N=%lld stride=%d num_signals=%d (0..29) signals_stride=%lld window=%d", (long long)N,
                    stride, num_signals, (long long)signals_stride, window);
    if (N == 0) return S3D_OK;
    if (!w_w_id || !n2n || !coords || !signals || !out) return fail(S3D_ERR_NULL_POINTER, "s3d_level_signals: null device pointer");
    if (reinterpret_cast<uintptr_t>(coords) % 16 != 0) return fail(S3D_ERR_BAD_SHAPE, "s3d_level_signals: coords must be 16-byte aligned");
    const int columns = 3 + num_signals;
    hipLaunchKernelGGL(level_signals_kernel, dim3(static_cast<unsigned>(ceil_div(N, kThreads))), dim3(kThreads),
                       kThreads * columns * sizeof(float), static_cast<hipStream_t>(stream), w_w_id, n2n,
                       reinterpret_cast<const int4 *>(coords), 1.0f / static_cast<float>(stride), signals, signals_stride, columns, window,
                       xyz_scale, other_scale, out, N);
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}

extern "C" __attribute__((visibility("default"))) int s3d_gather_rows(const void *from, int64_t n, const int64_t *rows, int64_t M, int32_t width,
                                                                      int32_t word_bytes, void *out, void *stream)
{
    using namespace s3d;
    if (n < 0 || width < 1 || width > 1024 || n > 0x7fffffff / width || M < 0 || M > 0xffffffffffLL || (word_bytes != 2 && word_bytes != 4))
        return fail(S3D_ERR_BAD_SHAPE, "s3d_gather_rows: n=%lld M=%lld width=%d (1..1024, below 2^31 words) word_bytes=%d (2 or 4)", (long long)n, (long long)M,
                    width, word_bytes);
    if (M == 0) return S3D_OK;
    if ((n > 0 && !from) || !rows || !out) return fail(S3D_ERR_NULL_POINTER, "s3d_gather_rows: null device pointer");
    const dim3 grid(static_cast<unsigned>(ceil_div(M, kGatherRows)));
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (word_bytes == 2)
        hipLaunchKernelGGL((gather_rows_kernel<uint16_t>), grid, dim3(kThreads), 0, s, static_cast<const uint16_t *>(from), n, rows, M, width,
                           static_cast<uint16_t>(0x7e00), static_cast<uint16_t *>(out));
    else
        hipLaunchKernelGGL((gather_rows_kernel<uint32_t>), grid, dim3(kThreads), 0, s, static_cast<const uint32_t *>(from), n, rows, M, width,
                           0x7fc00000u, static_cast<uint32_t *>(out));
    S3D_HIP_CHECK(hipGetLastError());
    return S3D_OK;
}
