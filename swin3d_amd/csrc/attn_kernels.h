// Internal interface between the attention entry point and its kernel families.
#pragma once

#include "s3d_common.h"
#include "attn_strip_list.h"

namespace s3d {

constexpr int kMaxAxes = 9;

// Everything a window-attention kernel needs, by value (lives in kernel-argument SGPRs).
struct AttnArgs {
    const void *q, *k, *v;                 // [N,H,D], voxel rows `row_stride` elements apart
    int64_t row_stride;
    const void *table_q, *table_k, *table_v;  // flat [sum rows][H][D]
    const int32_t *w_sizes, *w2n, *n2n;    // n2n may be null: rows already in window-sorted order
    const int32_t *sizes_dev;              // per-axis table sizes on the device (rows[] / base[] unset), or null
    const float *n_coords;                 // [N,nd], window-sorted
    void *out;                             // [N,H,D]
    float *out_max, *out_sum;              // [N,H] or null
    void *workspace;                       // the work list: queue counters, unit and window records
    int32_t block_shift;                   // the step target, a lane streams about 2^block_shift keys
    int32_t target_items;                  // wavefronts a head group's list is cut for (sizes the finer units at its end)
    int32_t leave_to_tiles;                // sizes_dev: the tile or strip kernel was launched too and serves sizes that fit it
    int32_t set_groups;                    // workgroups that come in runs of eight to a head group (the others in turn)
    int32_t H, D, nd, total_rows;
    int64_t N, W;
    int32_t rows[kMaxAxes];                // rows of each axis table
    int32_t base[kMaxAxes];                // first row of each axis table in the flat table
};
// With 264 bytes in place of 248 the sweep took, statistics asked for, 10,000 voxels x 6 heads of 8, 6 axes, 75.1 us for 72.3, 6,000 x 6
// of 16, 9 axes, 98.3 for 95.1, 1,500 x 12 88.4 for 87.2; launches from 12,421 x 12 on the same.
static_assert(sizeof(AttnArgs) <= 256, "four lines of kernel arguments");

// Table rows of an axis that the tile and strip kernels take: of a position axis, of a colour or normal axis.
constexpr int kTileRows = 64, kTileSignalRows = 32;
template <typename Rows> __host__ __device__ inline bool rows_fit_tiles(const Rows &rows, int nd)
{
    for (int n = 0; n < nd; ++n)
        if (rows[n] < 1 || rows[n] > (n < 3 ? kTileRows : kTileSignalRows)) return false;
    return true;
}
#ifdef __HIPCC__
// Rows of axis n by the caller's device tensor of table sizes, clipped so that every axis keeps a row inside the head's
// table; `run`: rows of the axes before it.
__device__ __forceinline__ int device_rows(const AttnArgs &a, int n, int nd, int run)
{
    const int rows = __builtin_amdgcn_readfirstlane(a.sizes_dev[n]) / (a.H * a.D);
    return max(1, min(rows, a.total_rows - run - (nd - 1 - n)));
}
#endif

// Persistent workgroups, one to three heads each with their table slices in LDS; lane = one query of some window,
// which streams that window's keys; VALU math (packed fp16 dot products for fp16 I/O), any dtype, windows of any
// size.  Needs a.workspace (work queues, sorted window list, unit list).
size_t attn_sweep_workspace_bytes(int H, int64_t W, int64_t N);
// The part of it that holds notes of the list builder, its size, and how much of it a builder of one workgroup has at its front.
constexpr size_t kSweepNotesBytes = size_t(320) << 10, kSweepNotesKept = size_t(16) << 10;
void *attn_sweep_notes(const AttnArgs &a);
// what: kAttnBuildList (the list kernels: needs w_sizes, w2n and the shape only), kAttnSweep (the sweep on a
// work list that is already in a.workspace; the launch leaves it ready for the next one), or both; with kAttnStripList the
// strip kernel's list along with the sweep's, in the launch that makes it of a few windows.
constexpr int kAttnBuildList = 1, kAttnSweep = 2, kAttnStripList = 4;
int launch_attn_sweep(const AttnArgs &a, int dtype, hipStream_t stream, int what = kAttnBuildList | kAttnSweep);
// Up to this many windows one launch makes the sweep's list, and with kAttnStripList the strip kernel's.
constexpr int64_t kFewWindows = 256;

// The tile kernel (attn_tile.hip), fp32: a workgroup works off tiles of up to 64 queries by 64 keys of a head, the table
// products on the matrix pipe.  `list` is its unit list, attn_tile_list_bytes of device memory.
// With sizes_dev the host cannot tell whether every axis fits: it launches the tile kernel and the sweep kernel, and each
// works or returns by what it reads.
bool attn_tile_shape(int64_t N, int64_t W, int H, int nd);
bool attn_tile_applies(const AttnArgs &a, int dtype);
size_t attn_tile_list_bytes(int H, int64_t N, int64_t W);
int launch_attn_tile(const AttnArgs &a, void *list, hipStream_t stream, int what = kAttnBuildList | kAttnSweep);

// The strip kernel (attn_strip_fwd.hip), fp16: a workgroup works off strips of up to 16 queries of a window and a head, the
// table products on the matrix pipe.  Its strip list lies where the sweep's list builder has its notes, which nothing reads once
// that list is there: a plan with both builds the sweep's first, or both in one launch (kAttnStripList).  With sizes_dev as above.
bool attn_strip_shape(int64_t N, int64_t W, int H, int nd);
tile::StripList attn_strip_list(const AttnArgs &a);
bool attn_strip_applies(const AttnArgs &a, int dtype);
int launch_attn_strip(const AttnArgs &a, hipStream_t stream, int what = kAttnBuildList | kAttnSweep);

// host side: a kernel's dynamic-LDS limit (see there), compute units of the current device
int allow_dynamic_lds(const void *kernel, size_t bytes);
int device_cus();

// The pair sweeps of the backward on the sweep kernel's work list (built here, in b.f.workspace, which needs
// attn_sweep_workspace_bytes): dq, dk, dv, and dL, P of every (pair, head) for the table-gradient kernels.
constexpr int kPairSpare = 4;     // records that a lane of the key-owned sweep reads at a time
struct BwdPairArgs {
    AttnArgs f;                  // shape, q, k, v, tables, index arrays (n2n required), rows[] / base[], workspace
    const void *dout, *out;      // [N,H,D]
    const float *stat_max, *stat_sum, *delta;   // [N,H]: the forward's statistics, dout_i . o_i
    void *dq, *dk, *dv;          // [N,H,D], rows `grad_stride` elements apart (q, k, v: f.row_stride)
    int64_t grad_stride;
    const int64_t *pos_base;     // [N]: at a window's first sorted position, the pairs of the windows before it
    float2 *pd;                  // [H][pairs], and kPairSpare more: (dL, P) at base + j n + i  (i, j: query, key position inside the window)
    int64_t pairs;               // capacity of pd per head; windows beyond it are skipped
};
int launch_attn_bwd_pairs(const BwdPairArgs &b, int dtype, hipStream_t stream);
// dL and P alone (head_dim 8), with dout_i . o_i made from b.out in place of b.delta, and the lists of the strips that read them
namespace tile { struct StripSetup; }
int launch_attn_bwd_records(const BwdPairArgs &b, const tile::StripSetup &strips, int dtype, hipStream_t stream);

// The backward on tiles or strips (attn_tile_bwd.hip, attn_strip_records.hip): head_dim 16, tables that fit a stage, the pair count known.  Of the
// arguments it takes the shape, inputs and dq, dk, dv; its own workspace holds records, slots, unit and strip list.
bool attn_tile_bwd_applies(const int32_t *rows, int nd, int D, int64_t pairs);
size_t attn_tile_bwd_bytes(int H, int nd, int64_t N, int64_t W, int64_t pairs);
int launch_attn_tile_bwd(const BwdPairArgs &p, const void *out, float *dtq, float *dtk, float *dtv, void *workspace, int dtype,
                         hipStream_t stream);

// The backward at head_dim 8 on strips (attn_strip_bwd.hip): records by launch_attn_bwd_records, everything that is a sum over
// pairs from those.  `room`: attn_strip8_bytes of device memory beside what the pair sweeps have.
bool attn_strip8_applies(const int32_t *rows, int nd, int D, int dtype, int64_t N, int64_t W, int H, int64_t pairs, size_t room);
size_t attn_strip8_bytes(int H, int nd, int64_t N, int64_t W);
int launch_attn_strip8(const BwdPairArgs &p, float *dtq, float *dtk, float *dtv, void *room, int dtype, hipStream_t stream);

}  // namespace s3d
