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
};

int launch_linear(const LinearArgs &a, hipStream_t stream);

}  // namespace s3d
