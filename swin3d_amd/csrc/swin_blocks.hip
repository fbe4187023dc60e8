// The Swin blocks of a stage at inference (Swin3D/modules/swin3d_layers.py:563-625, 760-871) in one call.
//
// What bounds them on small scans is the host: through torch a block is some fifteen dispatches (300 us), while its seven
// kernels take a third of that.  Here the launches follow each other with nothing in between: per block
//   LayerNorm, qkv, attention, proj, add + LayerNorm, fc1 + GELU, fc2 (the last two as one on many rows)
// with the residual stream in fp32 and everything else in fp16, as under autocast.
#include "linear.h"

namespace s3d {
namespace {

// q, k, v and the attention's result side by side, then the hidden layer
size_t wide_bytes(int64_t N, int32_t C, int32_t hidden) { return align_up(static_cast<size_t>(N) * (hidden > 4 * C ? hidden : 4 * C) * 2, 256); }

}  // namespace
}  // namespace s3d

extern "C" __attribute__((visibility("default"))) size_t s3d_swin_blocks_workspace_bytes(int64_t N, int32_t C, int32_t hidden)
{
    using namespace s3d;
    if (N < 0 || C < 1 || hidden < 1) return 0;
    return align_up(static_cast<size_t>(N) * C * 2, 256) + wide_bytes(N, C, hidden);
}

extern "C" __attribute__((visibility("default"))) int s3d_swin_blocks(
    const float *x, float *x_out, void *pending, int64_t N, int32_t H, int32_t D, int32_t hidden, const int32_t *table_sizes,
    int32_t nd, int64_t table_len, const s3d_window_set *sets, int32_t num_sets, const s3d_swin_block *blocks,
    int32_t num_blocks, void *workspace, size_t workspace_bytes, void *stream)
{
    using namespace s3d;
    const int32_t C = H * D;
    if (N < 0 || H < 1 || D < 1 || C % 16 || C > 1024 || hidden < 16 || hidden % 16 || num_sets < 1 || num_blocks < 1)
        return fail(S3D_ERR_BAD_SHAPE, "s3d_swin_blocks: N=%lld H=%d D=%d hidden=%d (H D and hidden multiples of 16, H D at most "
                    "1024), %d sets, %d blocks", (long long)N, H, D, hidden, num_sets, num_blocks);
    if (N == 0) return S3D_OK;
    if (!x || !x_out || !pending || !table_sizes || !sets || !blocks)
        return fail(S3D_ERR_NULL_POINTER, "s3d_swin_blocks: null pointer");
    const size_t need = s3d_swin_blocks_workspace_bytes(N, C, hidden);
    if (!workspace || workspace_bytes < need)
        return fail(S3D_ERR_WORKSPACE, "s3d_swin_blocks: workspace %zu B < required %zu B", workspace ? workspace_bytes : size_t(0), need);
    hipStream_t s = static_cast<hipStream_t>(stream);
    char *normed = static_cast<char *>(workspace), *wide = normed + align_up(static_cast<size_t>(N) * C * 2, 256);
    const size_t row = static_cast<size_t>(C) * 2;                  // bytes of C fp16 channels
    char *attended = wide + static_cast<size_t>(N) * 3 * row;       // behind q, k, v
    for (int i = 0; i < num_blocks; ++i) {
        const s3d_swin_block &b = blocks[i];
        const s3d_window_set &w = sets[i % num_sets];
        // (x itself stays as it is: from the first block's second sum on the stream is in x_out)
        const float *from = i == 0 ? x : x_out;
        if (int rc = s3d_add_layernorm(from, i == 0 ? nullptr : pending, S3D_DTYPE_F16, b.norm1_weight, b.norm1_bias, b.norm1_eps,
                                       i == 0 ? nullptr : x_out, normed, S3D_DTYPE_F16, N, C, stream))
            return rc;
        if (int rc = launch_linear({normed, b.qkv_weight, b.qkv_bias, wide, N, 3 * C, C, false}, s)) return rc;
        if (int rc = s3d_attn_fwd(wide, wide + row, wide + 2 * row, b.table_q, b.table_k, b.table_v, table_sizes, nd, table_len,
                                  w.w_sizes, w.w2n, w.n2n, w.n_coords, attended, nullptr, nullptr, N, H, D, w.num_windows, 3 * C,
                                  S3D_DTYPE_F16, w.planned ? S3D_ATTN_PLANNED : 0, w.plan, w.plan_bytes, stream))
            return rc;
        if (int rc = launch_linear({attended, b.proj_weight, b.proj_bias, pending, N, C, C, false}, s)) return rc;
        if (int rc = s3d_add_layernorm(from, pending, S3D_DTYPE_F16, b.norm2_weight, b.norm2_bias, b.norm2_eps, x_out, normed,
                                       S3D_DTYPE_F16, N, C, stream))
            return rc;
        if (mlp_pays(N, C, hidden)) {
            if (int rc = launch_mlp({normed, b.fc1_weight, b.fc1_bias, b.fc2_weight, b.fc2_bias, pending, N, C, hidden}, s)) return rc;
            continue;
        }
        if (int rc = launch_linear({normed, b.fc1_weight, b.fc1_bias, wide, N, hidden, C, true}, s)) return rc;
        if (int rc = launch_linear({wide, b.fc2_weight, b.fc2_bias, pending, N, C, hidden, false}, s)) return rc;
    }
    return S3D_OK;
}
