// Interface between the backward's records kernel (attn_tile_bwd.hip) and the kernels that sum over pairs
// (attn_strip_bwd.hip).
#pragma once

#include "attn_tile.h"

namespace s3d {
namespace tile {

// rows and first row of axis n: a choice among the kernel's arguments (an index would put them into scratch memory)
template <int ND> __device__ __forceinline__ int axis_rows(const AttnArgs &a, int axis)
{
    int r = a.rows[0];
#pragma unroll
    for (int n = 1; n < ND; ++n) r = axis == n ? a.rows[n] : r;
    return r;
}
template <int ND> __device__ __forceinline__ int axis_base(const AttnArgs &a, int axis)
{
    int r = a.base[0];
#pragma unroll
    for (int n = 1; n < ND; ++n) r = axis == n ? a.base[n] : r;
    return r;
}

struct StripArgs {
    AttnArgs f;                 // shape, q, k, tables, index arrays, rows[] / base[]
    UnitList list;              // entries and strips
    const void *dout;
    const float2 *records;      // [H][pairs]: (dL, P) at pairs before the window + j n + i  (i, j: query, key inside the window)
    int64_t pairs;              // capacity of records per head; windows beyond it are not there
    const int4 *columns;        // [strip][column]: sorted position, row, window's first position, pairs before it (-1: beyond
                                // the records)
    const int32_t *column_rows; // [strip][column], and 64 more that nothing is made of
    const float *scales;        // [head][Tq, Tk, Tv]: what a product with the table's operand is multiplied by
    float *slots;               // [workgroup][kind][tile][lane][4]: table gradients as the products leave them
    void *dq, *dk, *dv;
    uint32_t grad_stride;       // elements between rows of dq, dk, dv (of q, k, v: f.row_stride)
    float *dtq, *dtk, *dtv;
    float half_rows[kMaxAxes], upper[kMaxAxes];    // what crse_row takes (made here, they would take two vector registers an axis)
};
size_t strip_slots_bytes(int H, int nd);
int launch_strip_gradients(const StripArgs &b, int dtype, hipStream_t stream);

}  // namespace tile
}  // namespace s3d
