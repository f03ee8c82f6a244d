// LayerNormalization of rows: what the operator's kernels (vit_glue.hip) and the products that normalise their own rows
// (igemm_f3_kernel.hpp) share.
#pragma once
#include "onhip_internal.hpp"

namespace onhip {

// layer_normalization.c:62-97: per row, psum and psum of squares added up element by element in float, then
// mean = psum / n (as a product with 1/n), var = (1/n) * psq - mean * mean, + 1e-20 (a double constant),
// 1 / sqrtf(var), and out = (x - mean) * inv_std * weight + bias with every operation rounded.
__device__ __forceinline__ void ln_stats(float psum, float psq, float inv_n, float *mean, float *inv_std) {
    const float m = __fmul_rn(psum, inv_n);
    float var = __fsub_rn(__fmul_rn(inv_n, psq), __fmul_rn(m, m));
    var = (float) ((double) var + 1e-20);
    *mean = m;
    // sqrtf, then 1 / std, each correctly rounded as on the CPU.  The single-precision square root of this
    // toolchain is the bare v_sqrt_f32 (a last bit off on some inputs); the double-precision one rounded to float
    // is exact (53 >= 2 * 24 + 2 bits).  The two steps are kept apart so that they cannot merge into v_rsq_f32.
    float sd = (float) sqrt((double) var);
    asm volatile("" : "+v"(sd));
    *inv_std = __fdiv_rn(1.0f, sd);
}

// One sum of a row in LDS, element by element: of the elements, or of their squares.  The additions of a row are one chain, which sets the
// pace; elements are read ahead of them.
template <bool SQ>
__device__ __forceinline__ float ln_chain(const float *t, int reduce) {
    constexpr int AHEAD = 16;
    float sum = 0.0f, next[AHEAD];
    auto add = [&](float v) { sum = __fadd_rn(sum, SQ ? __fmul_rn(v, v) : v); };
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) next[j] = t[j];
    int i = AHEAD;
    for (; i + AHEAD <= reduce; i += AHEAD) {
        float now[AHEAD];
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) now[j] = next[j];
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) next[j] = t[i + j];
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) add(now[j]);
    }
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) add(next[j]);
    for (; i < reduce; ++i) add(t[i]);
    return sum;
}

// (x - mean) * inv_std * weight + bias, every operation rounded
__device__ __forceinline__ float ln_one(float x, float mean, float inv_std, float w, float b) {
    return __fadd_rn(__fmul_rn(__fmul_rn(__fsub_rn(x, mean), inv_std), w), b);
}

}  // namespace onhip
