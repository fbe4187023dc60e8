/*
 * swin3d_amd -- C ABI of the MI355X (gfx950) sparse window-attention forward,
 * window index builder and KNN helper.
 *
 * Plain pointers and sizes only: every pointer named "device" is a HIP device
 * address, `stream` is a hipStream_t passed as void* (NULL = the null stream).
 * All entry points enqueue work on `stream` and return without synchronising
 * unless stated otherwise.  Every output and every workspace is allocated by the
 * caller; the only device memory the library itself holds is the fixed scratch
 * array of s3d_attn_fwd_noalloc (8 MiB per GPU, part of the code object).
 *
 * Return value: 0 on success, a negative S3D_ERR_* code for a rejected argument,
 * a positive value = the hipError_t of a failed runtime call.  A human readable
 * description of the last failure on the calling thread is returned by
 * s3d_last_error_string().
 *
 * Each declaration cites the reference interface it replaces (paths relative to
 * the microsoft/Swin3D tree).
 */
#ifndef SWIN3D_AMD_H
#define SWIN3D_AMD_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define S3D_OK 0
#define S3D_ERR_NULL_POINTER (-1)
#define S3D_ERR_BAD_SHAPE (-2)
#define S3D_ERR_BAD_DTYPE (-3)
#define S3D_ERR_UNSUPPORTED (-4)
#define S3D_ERR_WORKSPACE (-5)

/* element type of q/k/v, the tables and the attention output */
#define S3D_DTYPE_F32 0
#define S3D_DTYPE_F16 1
/* s3d_attn_bwd only: fp32 tables beside fp16 rows (q, k, v, out, dout, dq, dk, dv): the backward of an fp16 forward
 * computed in fp32, as PrecisionMode.HALF_FORWARD asks (Swin3D/sparse_dl/attn/attn_coff.py:206-215 casts the rows
 * up and the gradients down; here they are widened as they are loaded and rounded as they are stored) */
#define S3D_DTYPE_F32_F16_ROWS 2

/* largest K of s3d_knn (K_MAX of Swin3D/src/knn/knn_cuda_kernel.cu:4) */
#define S3D_KNN_KMAX 64
/* squared distance stored in unfilled KNN slots: float(0x7fffffff)
 * (MAX_DIST of Swin3D/src/knn/knn_cuda_kernel.cu:5); their index is -1 */
#define S3D_KNN_PAD_DIST2 2147483648.0f

/* Library version, major*10000 + minor*100 + patch. */
int s3d_version(void);

/* Description of the last error raised on the calling thread ("" if none). */
const char *s3d_last_error_string(void);

/*
 * Windowed self-attention forward with contextual relative signal encoding.
 *
 * Replaces the pair of pybind entry points
 *   cal_max_coffs           Swin3D/src/attn/self_attn_aio_fwd.cu:255-455
 *   self_attn_cuda_forward  Swin3D/src/attn/self_attn_aio_fwd.cu:457-688
 * (declared in Swin3D/src/attn/self_attn_aio_fwd.h:11-26, exported at
 * Swin3D/src/attn/attn_api.cpp:20,23) and the division
 * Swin3D/sparse_dl/attn/attn_coff.py:184, for pos_mode SEPARATE (3) and
 * indice_mode INDIRECT (2), in ONE pass and without the O(M) pair arrays
 * m2w_indices / w2m_offsets.
 *
 *   q, k, v        device [N,H,D] of `dtype`, original voxel order (q pre-scaled); see qkv_row_stride
 *   table_q/k/v    device [table_len] of `dtype`, layout [axis][row][h][c]
 *   table_sizes    HOST int32 [nd], table_sizes[n] = rows_n * H * D (the values of the
 *                  reference's `table_offsets` tensor, fwd.cu:258,285; read on the host so
 *                  that the row counts travel as kernel arguments)
 *                  With the flag S3D_ATTN_SIZES_ON_DEVICE the pointer is a DEVICE int32 [nd] array instead - the
 *                  tensor the reference's caller builds on every call (Swin3D/modules/swin3d_layers.py:511) - and
 *                  the host never reads it: the sweep kernel takes the row counts from it (clipped so that no
 *                  access leaves the head's table; sizes that do not add up to table_len give a wrong result, not
 *                  a fault).  s3d_attn_plan accepts NULL for table_sizes for such callers.
 *   table_len      elements per table = sum_n table_sizes[n]
 *   w_sizes, w2n   device int32 [W]: voxels per window, exclusive prefix sum
 *   n2n            device int32 [N]: window-sorted position -> original row, or NULL when the rows of q, k,
 *                  v and out are in window-sorted order already (position = row): the kernels then read and
 *                  write the rows in place, without the gather of Swin3D/src/attn/attn_utils.cuh:391-409
 *   n_coords       device fp32 [N,nd], window-sorted order, scaled by the quant sizes
 *   out            device [N,H,D] of `dtype`: softmax-normalised attention output
 *   out_max        device fp32 [N,H] or NULL: max logit per (voxel, head)
 *                  (the tensor cal_max_coffs returns)
 *   out_sum        device fp32 [N,H] or NULL: sum_j exp(logit - max)
 *                  (second tensor of self_attn_cuda_forward; raw = out * sum)
 *   qkv_row_stride elements between consecutive voxel rows of q, k and v (0 = H*D, dense).  A multiple
 *                  of 8 that is >= H*D: with 3*H*D and q, k, v pointing H*D apart the kernels read the
 *                  [N, 3*H*D] output of the qkv projection (Swin3D/modules/swin3d_layers.py:502-509) in
 *                  place, without the reference's reshape / permute / contiguous copy.
 *   flags          0, or S3D_ATTN_PLANNED (`workspace` holds a work list built by s3d_attn_plan, see below)
 *                  and / or S3D_ATTN_SIZES_ON_DEVICE (see table_sizes)
 *   workspace      device scratch of at least s3d_attn_fwd_workspace_bytes(H, N, W) bytes: the work list of the
 *                  launch (work-queue counters, one record per unit of 8 to 64 queries and one per window, the
 *                  list builder's notes, which give way to the strip list), about 2 N + 24 W bytes + 0.3 MB whatever
 *                  the window sizes, and where a call of this shape may run on tiles their unit list, about N / 2 + 8 W bytes
 *   w2n must be ascending (the exclusive prefix sum of w_sizes, as the reference builds it:
 *   Swin3D/modules/swin3d_layers.py:100-103).
 *   D in {8,16,32}, nd in {3,6,9}, H >= 1 (the reference takes head_dim up to 32: self_attn_aio_fwd.cu:486).
 *
 * Row index of axis n for the pair (query i, key j), all in fp32:
 *   rel = (n_coords[i][n] - n_coords[j][n]) + float(rows_n / 2)
 *   row = min(int(min(max(rel, 0), rows_n)), rows_n - 1)
 * (Swin3D/src/attn/attn_utils.cuh:444-450; the reference indexes one row past
 * the axis table when the clamped value equals rows_n, this library folds that
 * case onto the last row).
 *
 * fp16: inputs, tables and output are fp16; products accumulate in fp32, exp in fp32.  Every call gives the same bits
 * for the same inputs (no atomics on data but integer ones, work list in window order).
 *
 * Three kernels.  The sweep serves every shape: persistent workgroups that keep their heads' table slices in LDS, a lane
 * per query streaming its window's keys (VALU; packed fp16 dot products for fp16 I/O; there the value-table rows of a
 * pair are added three at a time in fp16 before they enter the fp32 sums - the reference's half path adds all of them
 * and the value in half2, Swin3D/src/attn/self_attn_aio_fwd.cu:147).  At head_dim 16 in launches that do not fill the
 * chip, without out_max and out_sum, it is a kernel with the tables on the matrix pipe and no sum in fp16: in fp16 on strips
 * of 16 queries, in fp32, with a mean window of at least 40 voxels, on tiles of 64 queries by 64 keys.  A NaN or an infinity in q, k, v or a table reaches the queries of
 * its own window, or of the pairs that use the table row, and no others.
 */
#define S3D_ATTN_PLANNED 4   /* `workspace` holds a plan written by s3d_attn_plan: see there */
#define S3D_ATTN_SIZES_ON_DEVICE 8   /* `table_sizes` is a DEVICE int32 [nd] array (see s3d_attn_fwd) */
size_t s3d_attn_fwd_workspace_bytes(int32_t H, int64_t N, int64_t W);
int s3d_attn_fwd(const void *q, const void *k, const void *v, const void *table_q,
                 const void *table_k, const void *table_v, const int32_t *table_sizes, int32_t nd,
                 int64_t table_len, const int32_t *w_sizes, const int32_t *w2n, const int32_t *n2n,
                 const float *n_coords, void *out, float *out_max, float *out_sum, int64_t N,
                 int32_t H, int32_t D, int64_t W, int64_t qkv_row_stride, int32_t dtype, int32_t flags,
                 void *workspace, size_t workspace_bytes, void *stream);

/*
 * Work list of the kernel that runs, built once per window set ("plan").
 *
 * The reference builds its O(pairs) index arrays once per window set and hands them to every attention call
 * of the blocks that share the set (Swin3D/modules/swin3d_layers.py:857-871: one `get_index01` per window
 * set, `indices` reused by the blocks).  The counterpart here is O(N + W): the windows sorted by size and cut into
 * units of 64 lanes.  s3d_attn_fwd builds it on every call (two small kernels); a caller that keeps a window set
 * for several calls builds it once with s3d_attn_plan and passes the plan buffer as `workspace` together with
 * the flag S3D_ATTN_PLANNED, for calls with the same w_sizes, w2n, N, W, H, D, dtype and table_sizes.  Such a call
 * runs the sweep, strip or tile kernel and nothing else (with table sizes on the device the sweep and the other, and one
 * of them returns); the plan has both lists where the shape may use either.  It holds the sweep's work counters, which a
 * launch leaves at zero again: a plan serves one call at a time (calls in stream order; not two streams at once).
 *   plan           device buffer of at least s3d_attn_plan_bytes(H, N, W) bytes (= s3d_attn_fwd_workspace_bytes)
 */
size_t s3d_attn_plan_bytes(int32_t H, int64_t N, int64_t W);
int s3d_attn_plan(const int32_t *table_sizes, int32_t nd, int64_t table_len, const int32_t *w_sizes,
                  const int32_t *w2n, int64_t N, int32_t H, int32_t D, int64_t W, int32_t dtype, void *plan,
                  size_t plan_bytes, void *stream);

/*
 * The same forward without a workspace argument and without any allocation.
 *
 * It has no counterpart in the reference.  It is for callers that cannot allocate device memory around the
 * call: code under HIP graph capture, tight serving loops, harnesses that forbid hipMalloc.  The work list lives
 * in a device array of 8 MiB that is part of the library's code object, one copy per GPU, held until the process
 * ends.  The call fails with S3D_ERR_WORKSPACE when s3d_attn_fwd_workspace_bytes(H, N, W) exceeds 8 MiB (about
 * 2 N + 24 W bytes + 0.3 MB, and N / 2 + 8 W where a call may run on tiles: e.g. one million voxels in up to 200 000
 * windows fit).  No call allocates or frees.
 * The first call on a device looks up the array's address there (hipGetSymbolAddress) and the first call of a
 * shape (dtype, head_dim, axes, heads per wavefront) raises that kernel's dynamic-LDS limit (hipFuncSetAttribute):
 * neither belongs into a stream capture, so make ONE eager call per device and shape before capturing; the calls
 * after it enqueue kernels only.
 * Every call on a GPU uses that GPU's one array: calls that overlap on one GPU (two streams, two host
 * threads) race on it and must be serialised by the caller; calls in stream order on one stream are safe,
 * and nothing is carried over from one call to the next.
 * Arguments, results and status codes as for s3d_attn_fwd.
 */
int s3d_attn_fwd_noalloc(const void *q, const void *k, const void *v, const void *table_q,
                         const void *table_k, const void *table_v, const int32_t *table_sizes, int32_t nd,
                         int64_t table_len, const int32_t *w_sizes, const int32_t *w2n, const int32_t *n2n,
                         const float *n_coords, void *out, float *out_max, float *out_sum, int64_t N,
                         int32_t H, int32_t D, int64_t W, int64_t qkv_row_stride, int32_t dtype, void *stream);

/*
 * Windowed self-attention backward.
 *
 * Replaces cal_exp_sum_grads and self_attn_indir_backward
 * (Swin3D/src/attn/self_attn_aio_bwd.cu:14-47 and :49-113, 197-509, exported at
 * Swin3D/src/attn/attn_api.cpp:21,24; called from
 * Swin3D/sparse_dl/attn/attn_coff.py:219-224) for pos_mode SEPARATE and indice_mode INDIRECT,
 * without the O(M) pair arrays.  Arithmetic is fp32 for both dtypes.
 *
 *   q .. n_coords  as for s3d_attn_fwd (the forward's inputs; with n2n NULL - rows in window order - the call
 *                  writes the identity map into its workspace and reads that)
 *   out, out_max, out_sum   the forward's outputs for the same inputs (out of `dtype`, statistics fp32):
 *                  the tensors the reference saves for backward (attn_coff.py:186-187)
 *   dout           device [N,H,D] of `dtype`: gradient of the loss w.r.t. `out`
 *   dq, dk, dv     device [N,H,D] of `dtype`, overwritten (every row belongs to exactly one window)
 *   dtable_q/k/v   device FP32 [table_len], overwritten; layout of the tables
 *   pairs          M = sum of w_sizes^2, the pairs of the window set (counts[1] of s3d_window_index; the length
 *                  of the reference's index arrays), or 0.  With M the call runs two pair sweeps on the forward's
 *                  kind of work list (dq, which leaves dL and P of every (pair, head) in the workspace, 8 * H * pairs
 *                  bytes; dk and dv, which reads them), and two table-gradient sweeps that read them too; with tables of at
 *                  most 64 rows on a position axis and 32 on a signal axis strips of 16 voxels with all their pairs give
 *                  all six gradients by matrix products instead: at head_dim 16, where strips leave dL and P too (tiles of
 *                  64 queries by 64 keys in fp32 and where the mean window has fewer than 14 voxels), and at head_dim 8,
 *                  where the first pair sweep does, but for the largest launches in fp32 and with three axes.  With 0 it runs two fused
 *                  sweeps that recompute the logits for the table gradients and need no such store (about a third
 *                  more time).  A value below M cannot hold the records of every window: the rows of dq, dk, dv
 *                  that belong to the windows beyond it and all three table gradients then come out as NaN.
 *   workspace      device scratch of at least s3d_attn_bwd_workspace_least_bytes(H, D, nd, table_len, N, W, pairs) bytes;
 *                  s3d_attn_bwd_workspace_bytes is never less, and has the 12 bytes a (pair, head) of an earlier store
 *   dtype          S3D_DTYPE_F32, S3D_DTYPE_F16, or S3D_DTYPE_F32_F16_ROWS: the tables fp32, every [N,H,D] tensor
 *                  fp16, the results those of dtype S3D_DTYPE_F32 on fp32 copies of the rows with dq, dk, dv
 *                  rounded to fp16 (the same arithmetic; the two launches may pack the windows differently, which
 *                  reorders the fp32 sums); needs pairs > 0
 *   D in {8,16,32}, nd in {3,6,9}.  head_dim 32 and tables of more than 64 * nd rows per head in total (quant 8
 *                  with wide windows) run in a general form in the manner of the reference - one thread per
 *                  (query, head), atomic adds for dk, dv (fp32 accumulators in the workspace) and for the table
 *                  gradients (per workgroup in LDS, then global), so only dq is then the same bits on every
 *                  call; `pairs` is ignored.  It is some fifty times slower per pair than the forms described
 *                  here (0.2 s for 200 000 voxels at head_dim 32) and exists so that every shape of the forward
 *                  has a backward; its workspace is 8 * N * H * D bytes plus the statistics.
 *
 * No global atomics (the general form apart).  dq, dk, dv have one owning lane per row and are sums in a fixed order: the same bits on
 * every call.  The table gradients are accumulated per wavefront over the units it draws from the work queues,
 * left in a slot of the workspace and summed per head, slots in order, by a reduction kernel: which units a
 * wavefront draws varies from call to call, so these sums are regrouped and agree between calls to fp32 rounding
 * (about 1e-6 of the largest element), not bit for bit.
 *
 * On tiles and strips, what is not finite in q, k, v, dout or a table makes NaN of the gradients that it belongs to as a sum over
 * pairs - those of its window, and of the table rows of its pairs - and of no others, but for the other channels of a
 * voxel or table row with such a dout; so does a statistic that is not the forward's, where it makes a weight above 8.
 */
size_t s3d_attn_bwd_workspace_bytes(int32_t H, int32_t D, int32_t nd, int64_t table_len, int64_t N, int64_t W,
                                    int64_t pairs);
size_t s3d_attn_bwd_workspace_least_bytes(int32_t H, int32_t D, int32_t nd, int64_t table_len, int64_t N, int64_t W,
                                          int64_t pairs);
int s3d_attn_bwd(const void *q, const void *k, const void *v, const void *table_q, const void *table_k,
                 const void *table_v, const int32_t *table_sizes, int32_t nd, int64_t table_len,
                 const int32_t *w_sizes, const int32_t *w2n, const int32_t *n2n, const float *n_coords,
                 const void *out, const float *out_max, const float *out_sum, const void *dout, void *dq,
                 void *dk, void *dv, float *dtable_q, float *dtable_k, float *dtable_v, int64_t N,
                 int32_t H, int32_t D, int64_t W, int64_t pairs, int32_t dtype, void *workspace,
                 size_t workspace_bytes, void *stream);
/*
 * The same with rows of q, k, v `qkv_row_stride` and of dq, dk, dv `grad_row_stride` elements apart (multiples of 8, at
 * least H*D, base addresses 16-byte aligned): slices of a projection's [N, 3 H D] output and of its gradient, in place.
 * Other than H*D they need pairs > 0 and a shape that the forms with a pair store take (head_dim 8 or 16).
 */
int s3d_attn_bwd_strided(const void *q, const void *k, const void *v, const void *table_q, const void *table_k,
                         const void *table_v, const int32_t *table_sizes, int32_t nd, int64_t table_len,
                         const int32_t *w_sizes, const int32_t *w2n, const int32_t *n2n, const float *n_coords,
                         const void *out, const float *out_max, const float *out_sum, const void *dout, void *dq,
                         void *dk, void *dv, float *dtable_q, float *dtable_k, float *dtable_v, int64_t N,
                         int32_t H, int32_t D, int64_t W, int64_t pairs, int64_t qkv_row_stride, int64_t grad_row_stride,
                         int32_t dtype, void *workspace, size_t workspace_bytes, void *stream);

/*
 * Up to 16 arrays from fp32 to fp16 (round to nearest even, as a cast of the framework's), in one launch.
 * from, to, counts: HOST arrays of device addresses and element counts.
 */
int s3d_cast_half(const float *const *from, void *const *to, const int64_t *counts, int32_t num, void *stream);

/*
 * Up to 24 fp32 arrays [rows, cols] to fp16, as they are and / or transposed, the first scaled_rows rows times `scale` (in
 * fp32, then rounded), and / or as they are to fp32; in one launch.
 *   from    HOST array of device addresses
 *   copies  HOST array
 *   half    device, fp16, 16-byte aligned: what `to` and `transposed` are offsets into, in elements (-1: not wanted)
 *   same    device, fp32, 16-byte aligned: what `same` is an offset into (-1: not wanted)
 * A transposed array has rows and cols that are multiples of 8, and it and its offsets are 16-byte aligned.
 */
typedef struct {
    int64_t rows, cols, scaled_rows, to, transposed, same;
    float scale;
} s3d_half_copy;

int s3d_half_copies(const float *const *from, const s3d_half_copy *copies, int32_t num, void *half, float *same, void *stream);

/* out = x + residual (fp16, widened first); count a multiple of 4, all 16-byte aligned; out may be x. */
int s3d_add_half(const float *x, const void *residual, float *out, int64_t count, void *stream);

/*
 * Window sort + segment offsets.
 *
 * Replaces BasicLayer.get_map_pair / get_window_mapping
 * (Swin3D/modules/swin3d_layers.py:713-787, MinkowskiEngine pooling + kernel_map +
 * torch.sort) and the w2n / w_sizes part of sparse_self_attention (:96-103).
 *
 *   coords     device int32 [N,4] rows (batch, x, y, z); x,y,z multiples of `stride`
 *   stride     tensor stride of the voxel grid (>= 1)
 *   window     window size in voxels per side (1..10)
 *   shift      window shift in voxels (0 or window/2; get_shifted_sp, :824-838)
 *   n2n        device int32 [N]  out: window-sorted position -> original row
 *   w_w_id     device int32 [N]  out: local id lx*window^2 + ly*window + lz per sorted position
 *   w_sizes    device int32 [N]  out: first W entries = voxels per window
 *   w2n        device int32 [N]  out: first W entries = exclusive prefix sum of w_sizes
 *   counts     device int64 [4]  out: {W, M = sum w_sizes^2, max w_size, error flag}
 *                                 error flag != 0: a coordinate was outside the supported
 *                                 range (batch 0..4095, window coordinates -8192..8191)
 *   workspace  device scratch of at least s3d_window_index_workspace_bytes(N) bytes
 *
 * Window order: ascending (batch, wx, wy, wz) with floor division of the shifted
 * coordinate by window*stride; inside a window ascending local id; equal keys by
 * ascending original row.
 */
size_t s3d_window_index_workspace_bytes(int64_t N);
int s3d_window_index(const int32_t *coords, int64_t N, int32_t stride, int32_t window,
                     int32_t shift, int32_t *n2n, int32_t *w_w_id, int32_t *w_sizes, int32_t *w2n,
                     int64_t *counts, void *workspace, size_t workspace_bytes, void *stream);

/*
 * The same index by a counting sort over the lattice of windows, for scenes whose windows fit a dense lattice of
 * at most max(4096, 6 N) cells (capped at 2^24): the bounding box of (batch, wx, wy, wz) over the voxels.  Room-sized
 * scenes do; the call is then six launches of a few microseconds instead of a sort of all voxels.  Same arguments
 * and outputs as s3d_window_index (the results are identical, rows of equal coordinates in row order); own
 * workspace size.  When the lattice is too large, counts[3] has bit 1 (value 2) set and NO output is written: call
 * s3d_window_index instead.  counts[3] bit 0 (value 1): coordinates out of range, as for s3d_window_index.
 */
size_t s3d_window_index_grid_workspace_bytes(int64_t N);
int s3d_window_index_grid(const int32_t *coords, int64_t N, int32_t stride, int32_t window,
                          int32_t shift, int32_t *n2n, int32_t *w_w_id, int32_t *w_sizes, int32_t *w2n,
                          int64_t *counts, void *workspace, size_t workspace_bytes, void *stream);

/*
 * s3d_window_index_grid for up to four window sets of the same voxels in one run of launches.  sets: HOST array.
 */
typedef struct {
    int32_t *n2n, *w_w_id, *w_sizes, *w2n;   /* device int32 [N] out, as for s3d_window_index_grid */
    int64_t *counts;                         /* device int64 [4] out */
    int32_t window, shift;
} s3d_window_index_set;

size_t s3d_window_indices_workspace_bytes(int64_t N, int32_t num_sets);
int s3d_window_indices(const int32_t *coords, int64_t N, int32_t stride, const s3d_window_index_set *sets, int32_t num_sets,
                       void *workspace, size_t workspace_bytes, void *stream);
/*
 * The same, and the calling thread waits for the counts, which also go to host_counts: pinned HOST int64 [num_sets][4]
 * (hipHostMalloc).  It waits for the launches that lead to them and not for those behind them, which put the voxels in
 * order.  Not for graph capture.
 */
int s3d_window_indices_counted(const int32_t *coords, int64_t N, int32_t stride, const s3d_window_index_set *sets,
                               int32_t num_sets, int64_t *host_counts, void *workspace, size_t workspace_bytes, void *stream);
/*
 * The same, but the calling thread waits for all of the stream's work: the sets are finished when this returns.
 */
int s3d_window_indices_finished(const int32_t *coords, int64_t N, int32_t stride, const s3d_window_index_set *sets,
                                int32_t num_sets, int64_t *host_counts, void *workspace, size_t workspace_bytes, void *stream);

/*
 * Representative voxel of every cell of a window sort: the member whose signal row is nearest (Euclidean, fp32) to
 * the mean of the cell's signal rows; ties go to the lower row.  With a sort at window = 2 a cell is a coarse voxel
 * of the stride-2 downsample (GridCoordsDown, Swin3D/modules/swin3d_layers.py:179-231, a chain of scatter
 * reductions there).  Members are summed in sorted order, so the result is deterministic.
 *
 *   n2n, w2n, w_sizes  device int32: outputs of s3d_window_index (W = counts[0] cells)
 *   signals            device fp32 rows of `signals_stride` floats, original row order; the first `num_signals`
 *                      columns (1..16) enter the distance
 *   out                device int64 [W]: the chosen row of every cell (2^31 - 1 where NaN leaves no member nearest)
 */
int s3d_cell_representatives(const int32_t *n2n, const int32_t *w2n, const int32_t *w_sizes, int64_t W,
                             const float *signals, int64_t signals_stride, int32_t num_signals, int64_t *out,
                             void *stream);

/*
 * Rows of the lattice neighbours of every voxel, from the voxels' sorted packed keys.
 *
 * A packed coordinate key is linear in (batch, x, y, z), so a neighbour's key is the voxel's key plus a constant
 * per offset.  Used for the 27 offsets of the stem's 3x3x3 sparse convolution (the reference takes the kernel map
 * from MinkowskiEngine, Swin3D/models/Swin3D.py:75-86); no counterpart kernel in the reference.
 *
 *   sorted_keys  device int64 [N] ascending, distinct      order  device int64 [N]: order[i] = row of sorted_keys[i]
 *   deltas       device int64 [M] key offsets (1 <= M <= 1024)
 *   out          device int64 [N,M]: out[order[i]][d] = order[p] with sorted_keys[p] = sorted_keys[i] + deltas[d],
 *                or N when no voxel has that key
 */
int s3d_key_neighbours(const int64_t *sorted_keys, const int64_t *order, int64_t N, const int64_t *deltas, int32_t M,
                       int64_t *out, void *stream);
/*
 * The 27 neighbours (x first, then y, z; the voxel itself among them) of every voxel on a lattice of `stride`: out int64 [N][27],
 * the first row with these coordinates, N where there is none.  coords device int32 [N,4] (batch, x, y, z), 16-byte
 * aligned, x, y, z of less than 2^(field - 1) either side.  N below 2^30.
 */
size_t s3d_voxel_neighbours_workspace_bytes(int64_t N);
int s3d_voxel_neighbours(const int32_t *coords, int64_t N, int32_t field, int32_t stride, int64_t *out, void *workspace,
                         size_t workspace_bytes, void *stream);
/*
 * out [M][width]: rows[m] (device int64) of from [n][width], words of 2 (fp16) or 4 (fp32) bytes; row n is a row of zeros,
 * below zero counts back from behind it, any other index gives a row of NaN.
 */
int s3d_gather_rows(const void *from, int64_t n, const int64_t *rows, int64_t M, int32_t width, int32_t word_bytes, void *out,
                    void *stream);
/* out int32 [B]: how many of the N ascending batch ids (`stride` apart) are at most b */
int s3d_segment_ends(const int32_t *batch, int64_t stride, int64_t N, int32_t B, int32_t *out, void *stream);
/* the same for two columns, out int32 [2][B]: sources and queries of s3d_knn */
int s3d_segment_ends_of_two(const int32_t *first, int64_t first_stride, int64_t first_N, const int32_t *second, int64_t second_stride,
                            int64_t second_N, int32_t B, int32_t *out, void *stream);
/*
 * The next coarser level from a sort of the voxels into its cells: what s3d_cell_representatives gives (pick), the cells'
 * coordinates (int32 [W][4], rounded down to multiples of `step`) and the picked rows' signals (fp32 [W][num_signals]).
 * Where NaN among its members' signals leaves a cell without a nearest one, pick is 2^31 - 1 (as there), the batch -1, which
 * s3d_window_index and its kin report as out of range, and the signals NaN.
 */
int s3d_pool_cells(const int32_t *n2n, const int32_t *w2n, const int32_t *w_sizes, int64_t W, const int32_t *coords,
                   int32_t step, const float *signals, int64_t signals_stride, int32_t num_signals, int64_t *pick,
                   int32_t *out_coords, float *out_signals, void *stream);
/*
 * s3d_window_signals from a level's voxels and signals (batch, x, y, z in voxel units, num_signals others): the position
 * inside a voxel is (signal - coordinate) times the reciprocal of the stride.
 */
int s3d_level_signals(const int32_t *w_w_id, const int32_t *n2n, const int32_t *coords, int32_t stride, const float *signals,
                      int64_t signals_stride, int32_t num_signals, int32_t window, float xyz_scale, float other_scale,
                      float *out, int64_t N, void *stream);

/*
 * Signal matrix of the attention op in window-sorted order (the `n_coords` argument of s3d_attn_fwd), one pass.
 *
 * Replaces the tensor statements of BasicLayer.get_index01 (Swin3D/modules/swin3d_layers.py:800-804: window-local
 * voxel position + fractional position, other signals appended, both gathered into sorted order) and, with the
 * two scales, of WindowAttention.forward (:513-536: xyz columns times quant_size, the others times 2 * quant_size).
 *
 *   w_w_id, n2n   device int32 [N]   outputs of s3d_window_index
 *   frac          device fp32 [N,3]  position of the point inside its voxel, in voxels, original row order
 *   signals       device fp32 rows of `signals_stride` floats, original row order; the first `num_signals`
 *                 columns are used (0, 3 or 6: colour, normal); may be null when num_signals = 0
 *   out           device fp32 [N, 3 + num_signals]:
 *                 out[p] = ((lx, ly, lz) + frac[n2n[p]]) * xyz_scale, signals[n2n[p]] * other_scale
 *                 (sum and product rounded separately, as the tensor statements do)
 *   scales 1, 1 give the reference's unscaled n_coords.
 */
int s3d_window_signals(const int32_t *w_w_id, const int32_t *n2n, const float *frac, const float *signals,
                       int64_t signals_stride, int32_t num_signals, int32_t window, float xyz_scale,
                       float other_scale, float *out, int64_t N, void *stream);

/*
 * K nearest sources of every query inside the same batch segment.
 *
 * Replaces knn_cuda (Swin3D/src/knn/knn_cuda_kernel.cu:207-244, declared in
 * Swin3D/src/knn/knn_cuda_kernel.h:5-12, exported at Swin3D/src/knn/knn_api.cpp:5).
 *
 *   src_xyz      device fp32 [Ns,3]      query_xyz  device fp32 [Nq,3]
 *   src_offset   device int32 [B] cumulative END offsets of the batch segments of src
 *   query_offset device int32 [B] same for the queries
 *   ret_idx      device int32 [Nq,K] out: global source rows
 *   ret_dist2    device fp32 [Nq,K] out: SQUARED distances ((dx*dx + dy*dy) + dz*dz with
 *                every operation rounded to fp32, d = src - query)
 *   cell_size    edge of the bucketing grid in the units of xyz; <= 0 picks it from the data
 *   workspace    device scratch of at least s3d_knn_workspace_bytes(Ns, Nq, B) bytes
 *
 * Result per query: the K smallest sources under the order (distance, source row),
 * emitted in that order (ties go to the lower row).  Segments with fewer than K
 * sources are padded with row -1 and S3D_KNN_PAD_DIST2.  1 <= K <= S3D_KNN_KMAX.
 */
size_t s3d_knn_workspace_bytes(int64_t Ns, int64_t Nq, int32_t B);
int s3d_knn(int32_t K, const float *src_xyz, int64_t Ns, const float *query_xyz, int64_t Nq,
            const int32_t *src_offset, const int32_t *query_offset, int32_t B, int32_t *ret_idx,
            float *ret_dist2, float cell_size, void *workspace, size_t workspace_bytes,
            void *stream);
/* The same with Euclidean distances (the square roots, sqrt(S3D_KNN_PAD_DIST2) for padded slots) in ret_dist. */
/* ... with rows of three coordinates src_stride and query_stride floats apart (columns of a wider matrix), in place. */
int s3d_knn_strided(int32_t K, const float *src_xyz, int64_t src_stride, int64_t Ns, const float *query_xyz,
                    int64_t query_stride, int64_t Nq, const int32_t *src_offset, const int32_t *query_offset, int32_t B,
                    int32_t *ret_idx, float *ret_dist2, float cell_size, void *workspace, size_t workspace_bytes, void *stream);
int s3d_knn_distances(int32_t K, const float *src_xyz, int64_t Ns, const float *query_xyz, int64_t Nq,
                      const int32_t *src_offset, const int32_t *query_offset, int32_t B, int32_t *ret_idx,
                      float *ret_dist, float cell_size, void *workspace, size_t workspace_bytes, void *stream);

/*
 * Inverse-distance interpolation of source features at the queries, from the result of s3d_knn.
 *
 * Replaces the torch statement knn_linear_interpolation
 * (Swin3D/modules/swin3d_layers.py:53-73: K indexing passes over src_feat and the weight
 * arithmetic, about 3*K + 4 kernels) with one gather kernel:
 *   weight_i = 1 / (sqrt(dist2_i) + 1e-8), normalised over the K neighbours of the query
 *   out[q]   = sum_i weight_i * src_feat[idx[q][i]]
 *
 *   idx, dist2   device [Nq,K] as written by s3d_knn (squared distances)
 *   src_feat     device [Ns,C] of `dtype`        out   device [Nq,C] of `dtype`
 * Neighbour slots padded with row -1 carry no weight (the reference's torch indexing would read the
 * LAST source row there, with a weight of about 2e-5); a query with no neighbour at all gets zeros.
 * Accumulation is fp32, one rounding to `dtype`.
 */
/*
 * Channel-wise maximum of the source features over the K nearest sources of every query, from the result of s3d_knn.
 *
 * Replaces the gather + max of the KNN downsample (Swin3D/modules/swin3d_layers.py:292-312: query_knn_feature
 * builds [Nq,K,C], then max over K) with one kernel that never writes the gathered copies:
 *   out[q][c] = max_i src_feat[max(idx[q][i], 0)][c]
 * A slot padded with row -1 reads row 0, exactly as the clamped index of the tensor statement does;
 * NaN in one of the rows gives NaN, as under torch's amax.
 *   idx        device int32 [Nq,K] as written by s3d_knn
 *   src_feat   device [Ns,C] of `dtype` (Ns >= 1)        out   device [Nq,C] of `dtype`
 */
int s3d_knn_max_pool(const int32_t *idx, int32_t K, int64_t Nq, const void *src_feat, int64_t Ns, int32_t C,
                     int32_t dtype, void *out, void *stream);
/* The same of fp16 rows, the maxima in fp32. */
int s3d_knn_max_pool_widened(const int32_t *idx, int32_t K, int64_t Nq, const void *src_feat, int64_t Ns, int32_t C, float *out,
                             void *stream);

/*
 * The gradient of that call for src_feat: every query's dout goes in equal shares to the rows of its list that hold the
 * maximum `out`; a maximum that is not a number gives NaN to all of them.  dsrc_feat device [Ns,C] of `dtype`, written
 * whole; Nq and Ns at least 1.
 */
size_t s3d_knn_max_pool_grad_workspace_bytes(int64_t Nq, int32_t K, int64_t Ns, int32_t C, int32_t dtype);
int s3d_knn_max_pool_grad(const int32_t *idx, int32_t K, int64_t Nq, const void *src_feat, int64_t Ns, int32_t C,
                          int32_t dtype, const void *out, const void *dout, void *dsrc_feat, void *workspace,
                          size_t workspace_bytes, void *stream);

int s3d_knn_interpolate(const int32_t *idx, const float *dist2, int32_t K, int64_t Nq, const void *src_feat,
                        int64_t Ns, int32_t C, int32_t dtype, void *out, void *stream);

/*
 * The same for fp16 features, in fp32 and added to a row of features beside it: out = skip + interpolation, src_feat device
 * [Ns,C] and skip device [Nq,C] fp16, out device [Nq,C] fp32, dense and 16-byte aligned, C a multiple of 4 (an upsample's sum:
 * Swin3D/modules/swin3d_layers.py:358-366).  Its gradients: dout fp32, to dsrc_feat fp32 [Ns,C], which holds zeros before (by
 * atomic additions, in any order), and dskip fp16 [Nq,C]; either may be null.
 */
int s3d_knn_interpolate_add(const int32_t *idx, const float *dist2, int32_t K, int64_t Nq, const void *src_feat,
                            int64_t Ns, int32_t C, const void *skip, float *out, void *stream);
int s3d_knn_interpolate_grad(const int32_t *idx, const float *dist2, int32_t K, int64_t Nq, const float *dout, int64_t Ns,
                             int32_t C, float *dsrc_feat, void *dskip, void *stream);

/*
 * Residual add fused with LayerNorm, for the Swin block on either side of the attention operator.
 *
 * The reference block (Swin3D/modules/swin3d_layers.py:617-623) computes
 *   feats = short_cut + attn(norm1(feats));  feats = feats + mlp(norm2(feats))
 * with torch kernels (add, LayerNorm in fp32, and under autocast a cast in front of the next GEMM).  This call
 * does, per row of C channels,
 *   s = x + residual            (residual null: s = x)
 *   x_out = s                   (skipped when residual or x_out is null; x_out may be x)
 *   y = (s - mean(s)) / sqrt(var(s) + eps) * gamma + beta      (biased variance, as torch.nn.LayerNorm)
 *
 *   x              device [N,C] fp32 (the residual stream)
 *   residual       device [N,C] of residual_dtype (S3D_DTYPE_F32 / S3D_DTYPE_F16), or null
 *   gamma, beta    device [C] fp32
 *   y              device [N,C] of y_dtype
 * C a multiple of 4 and at most 1024; arithmetic in fp32.
 */
int s3d_add_layernorm(const float *x, const void *residual, int32_t residual_dtype, const float *gamma,
                      const float *beta, float eps, float *x_out, void *y, int32_t y_dtype, int64_t N, int32_t C,
                      void *stream);

/*
 * The same for training: sum = x + residual (fp16, widened first) and y = LayerNorm of it in fp16, with the bits that
 * torch.nn.functional.layer_norm gives in fp32, rounded to the nearest.  residual and sum may be null (then the rows are x
 * themselves).  All dense and 16-byte aligned, sum apart from x, y the residual's place or apart; C a multiple of 4 and at most 1024.
 */
int s3d_train_add_layernorm(const float *x, const void *residual, const float *gamma, const float *beta, float eps, float *sum,
                            void *y, int64_t N, int32_t C, void *stream);

/*
 * The gradients of either call with y in fp16: dx = dsum + the gradient of LayerNorm in fp32, dresidual the same in fp16,
 * dgamma and dbeta [C] in fp32.  sum device [N,C] is the call's x_out (x without a residual), dsum fp32 [N,C] or null,
 * dy fp16 [N,C]; dx and dresidual may be null; all dense and 16-byte aligned.  The same bits on every call.
 */
size_t s3d_layernorm_grad_workspace_bytes(int64_t N, int32_t C);
int s3d_layernorm_grad(const float *sum, const float *dsum, const void *dy, const float *gamma, float eps, float *dx,
                       void *dresidual, float *dgamma, float *dbeta, int64_t N, int32_t C, void *workspace,
                       size_t workspace_bytes, void *stream);

/*
 * y = x w^T + bias, then GELU (the exact form) where gelu is not zero; fp16 operands and result, fp32 accumulation, bias
 * and GELU, one rounding at the end.  x device [M,K], w device [N,K] (torch.nn.Linear's weight), bias device [N] or null,
 * y device [M,N], all dense and 16-byte aligned; N a multiple of 8, K of 16.
 */
int s3d_linear(const void *x, const void *w, const void *bias, void *y, int64_t M, int32_t N, int32_t K, int32_t gelu,
               void *stream);
/*
 * The same without GELU, the K products of a number added up one after the other: the bits of a product that is not split.
 * gelu, [M,N] or null: GELU (by erf, in fp32) of the rounded rows y, with the bits that torch's vectorized kernel gives.
 */
int s3d_linear_in_order(const void *x, const void *w, const void *bias, void *y, void *gelu, int64_t M, int32_t N, int32_t K,
                        void *stream);

/*
 * Both layers of an MLP in one kernel, y = fc2(GELU(fc1(x))), with the bits of two calls of s3d_linear on many rows: x, y device
 * [M,C], apart; w1 [hidden,C], b1 [hidden] or null, w2 [C,hidden], b2 [C] or null; fp16, dense and 16-byte aligned.  hidden a
 * multiple of 32 up to 1024, C one of 48, 64, 80, 96, 128, 160 and 192.
 */
int s3d_mlp(const void *x, const void *w1, const void *b1, const void *w2, const void *b2, void *y, int64_t M, int32_t C, int32_t hidden,
            void *stream);

/*
 * The gradients of that layer's weight and bias: dw = dy^T x [N,K] and db = column sums of dy [N], either may be null.
 * dy device [M,N], x device [M,K], fp16, dense and 16-byte aligned; dw, db of grad_dtype (fp32 sums, rounded once for
 * fp16); N and K multiples of 8, M at least 1.  The same bits on every call.
 */
size_t s3d_linear_grad_workspace_bytes(int64_t M, int32_t N, int32_t K);
int s3d_linear_grad(const void *dy, const void *x, void *dw, void *db, int32_t grad_dtype, int64_t M, int32_t N, int32_t K,
                    void *workspace, size_t workspace_bytes, void *stream);

/*
 * The stem at inference (Swin3D/modules/mink_layers.py:50-80): the 3x3x3 convolution over a voxel's neighbours, rounded to fp16,
 * BatchNorm with its running statistics and ReLU in fp32.
 *   feats        device [N,cin] of `dtype` (fp32 is rounded to fp16), cin at most 16
 *   neighbours   device int64 [N,27]: rows of feats, N where there is none (zeros)
 *   weight       device fp32 [27,cin,cout] (rounded to fp16), cout a multiple of 16 up to 96
 *   mean, var    device fp32 [cout];  gamma, beta likewise, or null;  out device fp32 [N,cout], 16-byte aligned
 */
size_t s3d_stem_workspace_bytes(int64_t N, int32_t cout);
int s3d_stem(const void *feats, int32_t dtype, int64_t N, int32_t cin, const int64_t *neighbours, const float *weight, int32_t cout,
             const float *mean, const float *var, const float *gamma, const float *beta, float eps, float *out, void *workspace,
             size_t workspace_bytes, void *stream);

/*
 * The Swin blocks of a stage at inference (Swin3D/modules/swin3d_layers.py:563-625): per block
 *   x = x + proj(attention(qkv(LayerNorm(x))));  x = x + fc2(GELU(fc1(LayerNorm(x))))
 * with the residual stream in fp32 and the branches in fp16, in one host call.  Block i works on window set i % num_sets.
 *
 *   x              device [N,C] fp32, C = H*D; left as it is
 *   x_out          device [N,C] fp32, and
 *   pending        device [N,C] fp16: the result is x_out + pending (the sum is the next LayerNorm's, which can make it
 *                  on its way)
 *   table_sizes    HOST [nd], as for s3d_attn_fwd
 *   sets, blocks   HOST arrays of the structs below, which hold device pointers
 * C and hidden multiples of 16, C at most 1024; head_dim, axes and tables as for s3d_attn_fwd in fp16.
 */
typedef struct {
    const int32_t *w_sizes, *w2n, *n2n;      /* as for s3d_attn_fwd (n2n may be null) */
    const float *n_coords;
    int64_t num_windows;
    void *plan;                              /* of s3d_attn_plan for these windows, H, D and fp16; where planned is 0, as */
    size_t plan_bytes;                       /* much memory, and every block makes its own list there */
    int32_t planned;
} s3d_window_set;

typedef struct {
    const float *norm1_weight, *norm1_bias, *norm2_weight, *norm2_bias;   /* fp32 [C] */
    const void *qkv_weight, *qkv_bias;       /* fp16 [3C,C] (the q rows scaled by D^-0.5), [3C] or null */
    const void *table_q, *table_k, *table_v; /* fp16 [table_len] */
    const void *proj_weight, *proj_bias;     /* fp16 [C,C], [C] or null */
    const void *fc1_weight, *fc1_bias;       /* fp16 [hidden,C], [hidden] or null */
    const void *fc2_weight, *fc2_bias;       /* fp16 [C,hidden], [C] or null */
    float norm1_eps, norm2_eps;
} s3d_swin_block;

size_t s3d_swin_blocks_workspace_bytes(int64_t N, int32_t C, int32_t hidden);
int s3d_swin_blocks(const float *x, float *x_out, void *pending, int64_t N, int32_t H, int32_t D, int32_t hidden,
                    const int32_t *table_sizes, int32_t nd, int64_t table_len, const s3d_window_set *sets, int32_t num_sets,
                    const s3d_swin_block *blocks, int32_t num_blocks, void *workspace, size_t workspace_bytes, void *stream);

/*
 * A Swin block behind its first LayerNorm in training, in fp16 with parameters in fp32:
 *   qkv = normed1 Wqkv^T + b;  attended = attention(qkv);  sum = x + (attended Wproj^T + b);  normed2 = LayerNorm(sum);
 *   hidden_in = normed2 Wfc1^T + b;  hidden_out = GELU(hidden_in);  pending = hidden_out Wfc2^T + b
 * in one host call: s3d_half_copies of the parameters, then products, attention and norm as s3d_linear_in_order, s3d_attn_fwd
 * and s3d_train_add_layernorm give them.
 *   params, copies   HOST, as for s3d_half_copies, which fills half and same
 *   qkv_weight ..    where in half, in elements, the copies of a layer and the tables begin; -1: there is no such bias
 *   pending          null: the last product is left to the caller
 *   windows          HOST, as for s3d_swin_blocks
 * N at least 1, C = H*D and hidden multiples of 16, C at most 1024; all device pointers 16-byte aligned.
 */
typedef struct {
    const float *const *params;
    const s3d_half_copy *copies;
    int64_t num_copies;
    void *half;
    float *same;                                             /* or null */
    int64_t qkv_weight, qkv_bias, proj_weight, proj_bias, fc1_weight, fc1_bias, fc2_weight, fc2_bias, table_q, table_k, table_v;
    const float *norm2_weight, *norm2_bias, *x;              /* fp32 [C], [C], [N,C] */
    const void *normed1;                                     /* fp16 [N,C] */
    void *qkv, *attended;                                    /* fp16 [N,3C], [N,C] */
    float *out_max, *out_sum, *sum;                          /* [N,H], [N,H], [N,C] */
    void *normed2, *hidden_in, *hidden_out, *pending;        /* fp16 [N,C], [N,hidden], [N,hidden], [N,C] */
    const s3d_window_set *windows;
    float norm2_eps;
} s3d_block_pass;

int s3d_swin_block_train(const s3d_block_pass *pass, int64_t N, int32_t H, int32_t D, int32_t hidden, const int32_t *table_sizes, int32_t nd,
                         int64_t table_len, void *stream);

/*
 * The gradients of a Swin block behind its first LayerNorm, in training in fp16 with parameters in fp32:
 *   sum = x + proj(attention(qkv(normed1)));  normed2 = LayerNorm(sum);
 *   hidden_in = fc1(normed2);  hidden_out = GELU(hidden_in);  pending = fc2(hidden_out)
 * with dsum [N,C] fp32 and dpending [N,C] fp16 the gradients of sum and pending, C = H*D.
 *   saved     HOST: what the forward left.  Weights transposed, in fp16 ([in,out]; the q columns of qkv times q_scale)
 *   grads     HOST: where the gradients go; null for those that are not wanted, but for norm2 and normed1
 *   dtype     S3D_DTYPE_F16, or S3D_DTYPE_F32_F16_ROWS with tables in fp32, as for s3d_attn_bwd
 *   pairs     at least 1; head_dim, tables and windows as the forms of s3d_attn_bwd with a pair store take them
 * N at least 1, C and hidden multiples of 16, C at most 1024; all device pointers 16-byte aligned.
 */
typedef struct {
    const void *normed1, *qkv, *attended;                    /* fp16 [N,C], [N,3C], [N,C] */
    const float *out_max, *out_sum, *sum;                    /* [N,H], [N,H], [N,C] */
    const void *normed2, *hidden_in, *hidden_out;            /* fp16 [N,C], [N,hidden], [N,hidden] */
    const void *qkv_weight_t, *proj_weight_t, *fc1_weight_t, *fc2_weight_t;
    const void *table_q, *table_k, *table_v;
    const float *norm2_weight;
    const int32_t *w_sizes, *w2n, *n2n;                      /* n2n may be null */
    const float *n_coords;
    float norm2_eps;
} s3d_block_saved;

typedef struct {
    float *x;                                                /* [N,C] */
    void *normed1;                                           /* fp16 [N,C] */
    float *norm2_weight, *norm2_bias;
    float *qkv_weight, *qkv_bias, *proj_weight, *proj_bias, *fc1_weight, *fc1_bias, *fc2_weight, *fc2_bias;
    float *table_q, *table_k, *table_v;
} s3d_block_gradients;

size_t s3d_swin_block_grad_workspace_bytes(int64_t N, int32_t H, int32_t D, int32_t hidden, int32_t nd, int64_t table_len, int64_t W,
                                           int64_t pairs);
int s3d_swin_block_grad(const s3d_block_saved *saved, const s3d_block_gradients *grads, const float *dsum, const void *dpending, int64_t N,
                        int32_t H, int32_t D, int32_t hidden, const int32_t *table_sizes, int32_t nd, int64_t table_len, int64_t W,
                        int64_t pairs, float q_scale, int32_t dtype, void *workspace, size_t workspace_bytes, void *stream);

#ifdef __cplusplus
}
#endif
#endif /* SWIN3D_AMD_H */
