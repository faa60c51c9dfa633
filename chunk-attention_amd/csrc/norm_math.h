// The two halves of an RMS norm over one 16-byte piece of a row, as every kernel that normalises computes them.
// Rounding points are the reference's (cpp/chunk_attn/layernorm_kernels.cu:23-117): the normalised value is rounded to
// fp16, then multiplied by the weight in fp16.
#pragma once

#include <hip/hip_runtime.h>

namespace ca {
namespace norm {

typedef _Float16 half_t;
typedef half_t h8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ float sum_of_squares8(const h8 x) {
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; e++) ss += float(x[e]) * float(x[e]);
    return ss;
}

// what the sum of the squares of a row of `hidden` elements makes of its elements
__device__ __forceinline__ float inverse_rms(float sum, int hidden, float epsilon) {
    return __builtin_amdgcn_rsqf(sum / float(hidden) + epsilon);
}

__device__ __forceinline__ h8 scaled8(const h8 x, const h8 w, float inv) {
    h8 y;
#pragma unroll
    for (int e = 0; e < 8; e++) y[e] = half_t(float(x[e]) * inv) * w[e];
    return y;
}

}  // namespace norm
}  // namespace ca
