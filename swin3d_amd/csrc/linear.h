// Dense layers of fp16 rows (linear.hip).
#pragma once

#include "s3d_common.h"

namespace s3d {

struct LinearArgs {
    const void *x, *w, *bias;   // [M,K], [N,K], [N] or null; fp16
    void *y;                    // [M,N] fp16
    int64_t M;
    int32_t N, K;
    bool gelu;
    const void *gelu_at = nullptr;   // [M,N] fp16: the rows, rounded, are gradients behind a GELU of these, and y those before it
    bool in_order = false;           // a number's K products are added up one after the other, whatever the tile
    void *gelu_out = nullptr;        // [M,N] fp16: GELU of y's rounded rows, beside them (in_order; without gelu and gelu_at)
};

int launch_linear(const LinearArgs &a, hipStream_t stream);

// Both layers of an MLP in one kernel (mlp.hip): y = fc2(GELU(fc1(x)))
struct MlpArgs {
    const void *x, *w1, *b1, *w2, *b2;   // [M,C], [hidden,C], [hidden] or null, [C,hidden], [C] or null; fp16
    void *y;                             // [M,C] fp16, apart from x
    int64_t M;
    int32_t C, hidden;
};
bool mlp_takes(int64_t M, int32_t C, int32_t hidden);
bool mlp_pays(int64_t M, int32_t C, int32_t hidden);      // ... and is faster than the layers apart
int launch_mlp(const MlpArgs &a, hipStream_t stream);

// A layer's weight and bias gradients (linear_grad.hip): dw = dy^T x, db = the column sums of dy; the first `scaled` rows of
// the weight (and numbers of the bias) are parameters times `scale`
struct LinearGrad {
    const void *dy, *x;   // [M,N], [M,K] fp16
    void *dw, *db;        // [N,K], [N]; one of them may be null
    int64_t M;
    int32_t N, K, scaled;
    float scale;
    const float *parts = nullptr;   // where launch_linear_grad_parts has put them, and how many
    int32_t splits = 0;
};

constexpr int kMostLinearGrads = 4;
// room for the parts of `num` layers, however they are grouped
size_t linear_grads_bytes(const LinearGrad *grads, int num);
// the parts of `num` layers of as many rows, to *parts and on, which is moved behind them
int launch_linear_grad_parts(LinearGrad *grads, int num, float **parts, hipStream_t stream);

// The gradients of (sum, y) = (x + residual, LayerNorm(x + residual)) (layernorm.hip), those of the norm's parameters in parts
struct NormGrad {
    const float *parts;      // [count][2 C]: of the weight, of the bias
    float *dgamma, *dbeta;
    int32_t count, C;
};
size_t layernorm_grad_bytes(int64_t N, int32_t C);
int launch_layernorm_grad(const float *sum, const float *dsum, const void *dy, const float *gamma, float eps, float *dx, void *dresidual, NormGrad *norm,
                          int64_t N, int32_t C, float *parts, hipStream_t stream);

// the sums of the parts of `num` layers and, unless null, of a norm in one launch
int launch_linear_grad_sums(const LinearGrad *grads, int num, const NormGrad *norm, int32_t grad_dtype, hipStream_t stream);

}  // namespace s3d
