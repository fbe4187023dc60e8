// A Swin block behind its first LayerNorm (Swin3D/modules/swin3d_layers.py:563-625) in training, and its gradients, a call each:
//   sum = x + proj(attention(qkv(normed)));  pending = fc2(GELU(fc1(LayerNorm(sum))))
//
// What bounds a training pass on scans of 10,000 to 100,000 voxels is the host: through autograd a block's backward is
// some twenty nodes and fifty dispatches (0.57 ms a block, 15 ms of Swin3D-S's pass), while its kernels take a third of that
// at 10,000 voxels.  Here the launches follow each other with nothing in between.  And there are fewer of them: the
// derivative of GELU is taken where fc2's gradient leaves its tile (a launch and two passes over the hidden layer less),
// dq, dk, dv are written where the projection's gradient reads them (no stacking copy), the parts of two
// layers' weight gradients come from one launch where their tiles are the same, and those of all four and of the norm are
// summed by one.
#include "linear.h"

namespace s3d {
namespace {

struct Places {
    size_t wide, normed, residual, parts, norm, rest, total;
};

// the layers in the order of the calls: fc2, fc1, proj, qkv
struct Layers {
    LinearGrad of[kMostLinearGrads];
};

Layers layers_of(int64_t N, int32_t C, int32_t hidden)
{
    return {{{nullptr, nullptr, nullptr, nullptr, N, C, hidden, 0, 1.0f},
             {nullptr, nullptr, nullptr, nullptr, N, hidden, C, 0, 1.0f},
             {nullptr, nullptr, nullptr, nullptr, N, C, C, 0, 1.0f},
             {nullptr, nullptr, nullptr, nullptr, N, 3 * C, C, 0, 1.0f}}};
}

// wide: the hidden layer's gradient, then that of q, k, v;  normed: that of LayerNorm's rows, then of the attention's
// result;  residual: that of proj's result;  parts, norm: of the weights' and of
// the norm's gradients;  rest: the scratch of one call at a time
Places places_of(int64_t N, int32_t C, int32_t hidden, int32_t H, int32_t D, int32_t nd, int64_t table_len, int64_t W, int64_t pairs)
{
    Places p;
    const size_t row = static_cast<size_t>(N) * 2;
    p.wide = 0;
    p.normed = p.wide + align_up(row * (hidden > 3 * C ? hidden : 3 * C), 256);
    p.residual = p.normed + align_up(row * C, 256);
    p.parts = p.residual + align_up(row * C, 256);
    const Layers layers = layers_of(N, C, hidden);
    p.norm = p.parts + align_up(linear_grads_bytes(layers.of, kMostLinearGrads), 256);
    p.rest = p.norm + align_up(layernorm_grad_bytes(N, C), 256);
    p.total = p.rest + s3d_attn_bwd_workspace_least_bytes(H, D, nd, table_len, N, W, pairs);
    return p;
}

bool fits(int64_t N, int32_t H, int32_t D, int32_t hidden)
{
    return N > 0 && N <= 0x7fffffff && H >= 1 && D >= 1 && H <= 1024 && D <= 1024 && H * D % 16 == 0 && H * D <= 1024 && hidden >= 16 &&
           hidden % 16 == 0 && hidden <= 16384;
}

}  // namespace
}  // namespace s3d

extern "C" __attribute__((visibility("default"))) int s3d_swin_block_train(const s3d_block_pass *pass, int64_t N, int32_t H, int32_t D, int32_t hidden,
                                                                           const int32_t *table_sizes, int32_t nd, int64_t table_len, void *stream)
{
    using namespace s3d;
    if (!fits(N, H, D, hidden))
        return fail(S3D_ERR_BAD_SHAPE, "s3d_swin_block_train: N=%lld H=%d D=%d hidden=%d (H D and hidden multiples of 16, H D at most 1024)",
                    (long long)N, H, D, hidden);
    if (!pass || !pass->windows || !table_sizes) return fail(S3D_ERR_NULL_POINTER, "s3d_swin_block_train: null pointer");
    const s3d_block_pass &p = *pass;
    const s3d_window_set &w = *p.windows;
    if (!p.half || !p.norm2_weight || !p.norm2_bias || !p.x || !p.normed1 || !p.qkv || !p.attended || !p.out_max || !p.out_sum || !p.sum || !p.normed2 ||
        !p.hidden_in || !p.hidden_out || p.qkv_weight < 0 || p.proj_weight < 0 || p.fc1_weight < 0 || p.fc2_weight < 0 || p.table_q < 0 ||
        p.table_k < 0 || p.table_v < 0)
        return fail(S3D_ERR_NULL_POINTER, "s3d_swin_block_train: null device pointer");
    if (p.num_copies < 0 || p.num_copies > 0x7fffffff) return fail(S3D_ERR_BAD_SHAPE, "s3d_swin_block_train: %lld copies", (long long)p.num_copies);
    if (int rc = s3d_half_copies(p.params, p.copies, static_cast<int32_t>(p.num_copies), p.half, p.same, stream)) return rc;
    const int32_t C = H * D;
    const size_t row = static_cast<size_t>(C) * 2;
    auto at = [&](int64_t element) { return element < 0 ? nullptr : static_cast<const char *>(p.half) + 2 * element; };
    auto dense = [&](const void *x, int64_t weight, int64_t bias, void *y, void *gelu, int32_t n, int32_t k) {
        return s3d_linear_in_order(x, at(weight), at(bias), y, gelu, N, n, k, stream);
    };
    if (int rc = dense(p.normed1, p.qkv_weight, p.qkv_bias, p.qkv, nullptr, 3 * C, C)) return rc;
    const char *qkv = static_cast<const char *>(p.qkv);
    if (int rc = s3d_attn_fwd(qkv, qkv + row, qkv + 2 * row, at(p.table_q), at(p.table_k), at(p.table_v), table_sizes, nd, table_len, w.w_sizes,
                              w.w2n, w.n2n, w.n_coords, p.attended, p.out_max, p.out_sum, N, H, D, w.num_windows, 3 * C, S3D_DTYPE_F16,
                              w.planned ? S3D_ATTN_PLANNED : 0, w.plan, w.plan_bytes, stream))
        return rc;
    // (proj's rows are needed until the norm has added them: in the place of the norm's rows that come after)
    if (int rc = dense(p.attended, p.proj_weight, p.proj_bias, p.normed2, nullptr, C, C)) return rc;
    if (int rc = s3d_train_add_layernorm(p.x, p.normed2, p.norm2_weight, p.norm2_bias, p.norm2_eps, p.sum, p.normed2, N, C, stream)) return rc;
    if (int rc = dense(p.normed2, p.fc1_weight, p.fc1_bias, p.hidden_in, p.hidden_out, hidden, C)) return rc;
    return p.pending ? dense(p.hidden_out, p.fc2_weight, p.fc2_bias, p.pending, nullptr, C, hidden) : S3D_OK;
}

extern "C" __attribute__((visibility("default"))) size_t s3d_swin_block_grad_workspace_bytes(
    int64_t N, int32_t H, int32_t D, int32_t hidden, int32_t nd, int64_t table_len, int64_t W, int64_t pairs)
{
    using namespace s3d;
    return fits(N, H, D, hidden) ? places_of(N, H * D, hidden, H, D, nd, table_len, W, pairs).total : 0;
}

extern "C" __attribute__((visibility("default"))) int s3d_swin_block_grad(
    const s3d_block_saved *saved, const s3d_block_gradients *grads, const float *dsum, const void *dpending, int64_t N, int32_t H, int32_t D,
    int32_t hidden, const int32_t *table_sizes, int32_t nd, int64_t table_len, int64_t W, int64_t pairs, float q_scale, int32_t dtype,
    void *workspace, size_t workspace_bytes, void *stream)
{
    using namespace s3d;
    if (!fits(N, H, D, hidden))
        return fail(S3D_ERR_BAD_SHAPE, "s3d_swin_block_grad: N=%lld H=%d D=%d hidden=%d (H D and hidden multiples of 16, H D at most 1024)",
                    (long long)N, H, D, hidden);
    if (pairs < 1) return fail(S3D_ERR_BAD_SHAPE, "s3d_swin_block_grad: pairs = %lld", (long long)pairs);
    if (dtype != S3D_DTYPE_F16 && dtype != S3D_DTYPE_F32_F16_ROWS)
        return fail(S3D_ERR_BAD_DTYPE, "s3d_swin_block_grad: dtype %d (1 = fp16, 2 = fp32 on fp16 rows)", dtype);
    if (!saved || !grads || !dsum || !dpending) return fail(S3D_ERR_NULL_POINTER, "s3d_swin_block_grad: null pointer");
    const s3d_block_saved &b = *saved;
    const s3d_block_gradients &g = *grads;
    if (!b.normed1 || !b.qkv || !b.attended || !b.sum || !b.normed2 || !b.hidden_in || !b.hidden_out || !b.qkv_weight_t || !b.proj_weight_t ||
        !b.fc1_weight_t || !b.fc2_weight_t || !b.norm2_weight || !g.norm2_weight || !g.norm2_bias || !g.normed1)
        return fail(S3D_ERR_NULL_POINTER, "s3d_swin_block_grad: null device pointer");
    const int32_t C = H * D;
    const Places p = places_of(N, C, hidden, H, D, nd, table_len, W, pairs);
    if (!workspace || workspace_bytes < p.total)
        return fail(S3D_ERR_WORKSPACE, "s3d_swin_block_grad: workspace %zu B < required %zu B", workspace ? workspace_bytes : size_t(0), p.total);
    hipStream_t s = static_cast<hipStream_t>(stream);
    char *base = static_cast<char *>(workspace);
    char *wide = base + p.wide, *normed = base + p.normed, *residual = base + p.residual, *rest = base + p.rest;
    float *parts = reinterpret_cast<float *>(base + p.parts);
    const size_t rest_bytes = p.total - p.rest, row = static_cast<size_t>(C) * 2;
    LinearGrad wanted[kMostLinearGrads];
    int num = 0, launched = 0;
    // the parts of a layer's weight and bias gradients, where they are wanted: with those of the layer behind it, in one launch
    auto layer = [&](const void *dy, const void *x, float *dw, float *db, int32_t n, int32_t k, int32_t scaled, float scale) {
        if (dw || db) wanted[num++] = LinearGrad{dy, x, dw, db, N, n, k, scaled, scale};
    };
    auto launch_parts = [&]() {
        const int rc = launch_linear_grad_parts(wanted + launched, num - launched, &parts, s);
        launched = num;
        return rc;
    };
    layer(dpending, b.hidden_out, g.fc2_weight, g.fc2_bias, C, hidden, 0, 1.0f);
    if (int rc = launch_linear({dpending, b.fc2_weight_t, nullptr, wide, N, hidden, C, false, b.hidden_in}, s)) return rc;
    layer(wide, b.normed2, g.fc1_weight, g.fc1_bias, hidden, C, 0, 1.0f);
    if (int rc = launch_parts()) return rc;
    if (int rc = launch_linear({wide, b.fc1_weight_t, nullptr, normed, N, C, hidden, false}, s)) return rc;
    NormGrad norm{nullptr, g.norm2_weight, g.norm2_bias};
    if (int rc = launch_layernorm_grad(b.sum, dsum, normed, b.norm2_weight, b.norm2_eps, g.x, residual, &norm, N, C,
                                       reinterpret_cast<float *>(base + p.norm), s))
        return rc;
    layer(residual, b.attended, g.proj_weight, g.proj_bias, C, C, 0, 1.0f);
    if (int rc = launch_linear({residual, b.proj_weight_t, nullptr, normed, N, C, C, false}, s)) return rc;
    const char *qkv = static_cast<const char *>(b.qkv);
    if (int rc = s3d_attn_bwd_strided(qkv, qkv + row, qkv + 2 * row, b.table_q, b.table_k, b.table_v, table_sizes, nd, table_len, b.w_sizes,
                                      b.w2n, b.n2n, b.n_coords, b.attended, b.out_max, b.out_sum, normed, wide, wide + row, wide + 2 * row,
                                      g.table_q, g.table_k, g.table_v, N, H, D, W, pairs, 3 * C, 3 * C, dtype, rest, rest_bytes, stream))
        return rc;
    layer(wide, b.normed1, g.qkv_weight, g.qkv_bias, 3 * C, C, C, q_scale);
    if (int rc = launch_parts()) return rc;
    if (int rc = launch_linear({wide, b.qkv_weight_t, nullptr, g.normed1, N, C, 3 * C, false}, s)) return rc;
    return launch_linear_grad_sums(wanted, num, &norm, S3D_DTYPE_F32, s);
}
