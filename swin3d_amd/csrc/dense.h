// Pieces shared by the kernels of the dense layers (linear.hip, mlp.hip).
#pragma once

#include "s3d_common.h"

namespace s3d {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2 __attribute__((ext_vector_type(2)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// x Phi(x) = (x + |x|) / 2 - |x| Phi(-|x|), with 2 Phi(-u) = 2^p(u): the logarithm of the normal distribution's tail is
// close to a parabola, and the polynomial of degree 7 with p(0) = 0 that fits it best for |x| Phi(-|x|) over [0, 5.8] (least
// squares at Chebyshev nodes) is 2.5e-7 off, the rounding of fp32; from 5.8 on the tail is below fp16's smallest number.
// Fifteen instruction slots where a rational form with an exponential took 22, and small results keep fp16's relative
// precision.  Infinities and NaN as x Phi(x) has them: the first sum is NaN for -infinity.
__device__ __forceinline__ float gelu(float x)
{
    const float u = fabsf(x), c = fminf(u, 5.8f);
    float p = fmaf(-7.429386528e-7f, c, 4.341329259e-5f);
    p = fmaf(p, c, -8.166006301e-4f);
    p = fmaf(p, c, 8.171264082e-3f);
    p = fmaf(p, c, -5.347365886e-2f);
    p = fmaf(p, c, -4.587851465e-1f);
    p = fmaf(p, c, -1.151172519f);
    return 0.5f * fmaf(-c, __builtin_amdgcn_exp2f(p * c), x + u);
}

// between what a wavefront's lanes write to its LDS and what other lanes of it read (it serves a wavefront in order)
__device__ __forceinline__ void wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

}  // namespace s3d
