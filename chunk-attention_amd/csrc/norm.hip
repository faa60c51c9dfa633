// RMS normalisation for gfx950 (MI355X), fp16 rows, fp32 statistics: the two operators the
// reference exports beside rotary_embedding (cpp/chunk_attn/layernorm_kernels.cu:23-117,
// python_exports_ops.cpp:16-18).  One workgroup per token row; 16-byte accesses when the row
// length allows; the second pass re-reads the row from cache.
//
//   rms_norm            out = fp16(x * rsqrt(mean(x^2) + eps)) * weight
//   fused_add_rms_norm  residual = fp16(input + residual);  input = fp16(residual * rsqrt(...)) * weight
//                       with the mean taken over the unrounded fp32 sums, as the reference does
//   add_rms_norm        the same with the mean over the rounded sums: bit for bit what an fp16 addition
//                       and rms_norm give in two launches
// Rounding points are the reference's: the normalised value is rounded to fp16, then multiplied
// by the weight in fp16.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.h"
#include "norm_math.h"

namespace ca {
namespace {

using norm::h8;
using norm::half_t;
using norm::scaled8;

constexpr int WG = 256;
enum { kNoAdd = 0, kAdd = 1, kAddRounded = 2 };   // what a row is added to first, and which sums the mean is of

__device__ __forceinline__ float block_sum(float v, float* sm) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) sm[w] = v;
    __syncthreads();
    return sm[0] + sm[1] + sm[2] + sm[3];
}

// VEC = 8: rows are multiples of 8 elements and 16-byte aligned; VEC = 1: any row length.
// With VEC = 8 a thread keeps the first KEEP pieces it reads (rows of up to KEEP * 2048 elements
// entirely) in registers between the two passes, so the row is read from memory once; longer rows
// re-read the rest.
constexpr int KEEP = 4;

// One 8-element piece of the first pass: returns its contribution to the sum of squares and
// leaves in x what the second pass normalises (with ADD: the rounded sum, also written to residual).
template <int ADD>
__device__ __forceinline__ float first_pass8(h8& x, half_t* __restrict__ residual_piece) {
    float ss = 0.f;
    if constexpr (ADD != kNoAdd) {
        const h8 r = *reinterpret_cast<const h8*>(residual_piece);
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float s = float(x[e]) + float(r[e]);
            if constexpr (ADD == kAdd) ss += s * s;
            x[e] = half_t(s);
            if constexpr (ADD == kAddRounded) ss += float(x[e]) * float(x[e]);
        }
        *reinterpret_cast<h8*>(residual_piece) = x;
    } else {
        ss = norm::sum_of_squares8(x);
    }
    return ss;
}

template <int VEC, int ADD>
__global__ __launch_bounds__(WG) void rms_norm_kernel(half_t* __restrict__ out, half_t* __restrict__ input,
                                                      half_t* __restrict__ residual,
                                                      const half_t* __restrict__ weight, float epsilon,
                                                      int hidden) {
    __shared__ float sm[4];
    const size_t row = size_t(blockIdx.x) * hidden;
    const half_t* src = ADD ? residual : input;
    half_t* dst = ADD ? input : out;
    float ss = 0.f;
    if constexpr (VEC == 8) {
        h8 kept[KEEP];
#pragma unroll
        for (int it = 0; it < KEEP; it++) {  // the loads of all kept pieces go out together
            const int idx = (threadIdx.x + it * WG) * 8;
            if (idx < hidden) kept[it] = *reinterpret_cast<const h8*>(input + row + idx);
        }
#pragma unroll
        for (int it = 0; it < KEEP; it++) {
            const int idx = (threadIdx.x + it * WG) * 8;
            if (idx < hidden) ss += first_pass8<ADD>(kept[it], ADD ? residual + row + idx : nullptr);
        }
        for (int idx = (threadIdx.x + KEEP * WG) * 8; idx < hidden; idx += WG * 8) {
            h8 x = *reinterpret_cast<const h8*>(input + row + idx);
            ss += first_pass8<ADD>(x, ADD ? residual + row + idx : nullptr);
        }
        const float inv = norm::inverse_rms(block_sum(ss, sm), hidden, epsilon);
#pragma unroll
        for (int it = 0; it < KEEP; it++) {
            const int idx = (threadIdx.x + it * WG) * 8;
            if (idx < hidden) {
                *reinterpret_cast<h8*>(dst + row + idx) =
                  scaled8(kept[it], *reinterpret_cast<const h8*>(weight + idx), inv);
            }
        }
        // (with ADD, a thread re-reads here only what it wrote above itself)
        for (int idx = (threadIdx.x + KEEP * WG) * 8; idx < hidden; idx += WG * 8) {
            *reinterpret_cast<h8*>(dst + row + idx) =
              scaled8(*reinterpret_cast<const h8*>(src + row + idx), *reinterpret_cast<const h8*>(weight + idx), inv);
        }
    } else {
        for (int idx = threadIdx.x; idx < hidden; idx += WG) {
            float s = float(input[row + idx]);
            if constexpr (ADD) {
                s += float(residual[row + idx]);
                residual[row + idx] = half_t(s);
                if (ADD == kAddRounded) s = float(half_t(s));
            }
            ss += s * s;
        }
        const float inv = norm::inverse_rms(block_sum(ss, sm), hidden, epsilon);
        for (int idx = threadIdx.x; idx < hidden; idx += WG) {
            dst[row + idx] = half_t(float(src[row + idx]) * inv) * weight[idx];
        }
    }
}

// A model's first launch: row r of the embedding of tokens.id[r], into `residual` and normalised into `out` (bit for
// bit what a gather and rms_norm give; not at all without an `out`), and tokens.position[r] where the layers read it.  The ids travel as a kernel
// argument: no pinned upload, no gather and no norm of their own in front of the first layer (8 rows of 1024: 3.3 us
// for four launches of 2.5 to 6).  One workgroup a row; rows of whole 16-byte pieces.
struct EmbedTokens {
    int32_t id[kEmbedRows];
    int32_t position[kEmbedRows];
};
__global__ __launch_bounds__(WG) void embed_norm_kernel(const half_t* __restrict__ embedding, half_t* __restrict__ residual,
                                                        half_t* __restrict__ out, int64_t* __restrict__ positions,
                                                        const half_t* __restrict__ weight, float epsilon, int hidden,
                                                        const EmbedTokens tokens) {
    __shared__ float sm[4];
    const half_t* src = embedding + size_t(tokens.id[blockIdx.x]) * hidden;
    const size_t row = size_t(blockIdx.x) * hidden;
    if (threadIdx.x == 0) positions[blockIdx.x] = tokens.position[blockIdx.x];
    float ss = 0.f;
    h8 kept[KEEP];
#pragma unroll
    for (int it = 0; it < KEEP; it++) {
        const int idx = (threadIdx.x + it * WG) * 8;
        if (idx < hidden) kept[it] = *reinterpret_cast<const h8*>(src + idx);
    }
#pragma unroll
    for (int it = 0; it < KEEP; it++) {
        const int idx = (threadIdx.x + it * WG) * 8;
        if (idx < hidden) {
            *reinterpret_cast<h8*>(residual + row + idx) = kept[it];
            ss += first_pass8<kNoAdd>(kept[it], nullptr);
        }
    }
    for (int idx = (threadIdx.x + KEEP * WG) * 8; idx < hidden; idx += WG * 8) {
        h8 x = *reinterpret_cast<const h8*>(src + idx);
        *reinterpret_cast<h8*>(residual + row + idx) = x;
        ss += first_pass8<kNoAdd>(x, nullptr);
    }
    if (!out) return;
    const float inv = norm::inverse_rms(block_sum(ss, sm), hidden, epsilon);
#pragma unroll
    for (int it = 0; it < KEEP; it++) {
        const int idx = (threadIdx.x + it * WG) * 8;
        if (idx < hidden) {
            *reinterpret_cast<h8*>(out + row + idx) = scaled8(kept[it], *reinterpret_cast<const h8*>(weight + idx), inv);
        }
    }
    for (int idx = (threadIdx.x + KEEP * WG) * 8; idx < hidden; idx += WG * 8) {
        *reinterpret_cast<h8*>(out + row + idx) =
          scaled8(*reinterpret_cast<const h8*>(src + idx), *reinterpret_cast<const h8*>(weight + idx), inv);
    }
}

}  // namespace

int launch_embed_norm(const void* embedding, const int32_t* ids, const int32_t* positions, int n_rows, void* residual,
                      void* out, int64_t* positions_out, const void* weight, float epsilon, int hidden, hipStream_t st) {
    if (hidden <= 0 || hidden % 8 != 0) return -1;
    for (int r0 = 0; r0 < n_rows; r0 += kEmbedRows) {
        const int n = n_rows - r0 < kEmbedRows ? n_rows - r0 : kEmbedRows;
        EmbedTokens tokens;
        for (int r = 0; r < n; r++) {
            tokens.id[r] = ids[r0 + r];
            tokens.position[r] = positions[r0 + r];
        }
        const size_t at = size_t(r0) * hidden;
        hipLaunchKernelGGL(embed_norm_kernel, dim3(n), dim3(WG), 0, st, static_cast<const half_t*>(embedding),
                           static_cast<half_t*>(residual) + at, out ? static_cast<half_t*>(out) + at : nullptr, positions_out + r0,
                           static_cast<const half_t*>(weight), epsilon, hidden, tokens);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return static_cast<int>(e);
    }
    return 0;
}

int launch_rms_norm(void* out, void* input, void* residual, const void* weight, float epsilon,
                    int64_t n_tokens, int hidden, bool vec8, bool mean_of_rounded, hipStream_t st) {
    if (n_tokens <= 0 || hidden <= 0) return 0;
    if (n_tokens > 0x7fffffff) return -1;
    const dim3 grid(static_cast<unsigned>(n_tokens)), block(WG);
    half_t* o = static_cast<half_t*>(out);
    half_t* in = static_cast<half_t*>(input);
    half_t* res = static_cast<half_t*>(residual);
    const half_t* w = static_cast<const half_t*>(weight);
    if (residual && mean_of_rounded) {
        if (vec8) hipLaunchKernelGGL((rms_norm_kernel<8, kAddRounded>), grid, block, 0, st, o, in, res, w, epsilon, hidden);
        else hipLaunchKernelGGL((rms_norm_kernel<1, kAddRounded>), grid, block, 0, st, o, in, res, w, epsilon, hidden);
    } else if (residual) {
        if (vec8) hipLaunchKernelGGL((rms_norm_kernel<8, kAdd>), grid, block, 0, st, o, in, res, w, epsilon, hidden);
        else hipLaunchKernelGGL((rms_norm_kernel<1, kAdd>), grid, block, 0, st, o, in, res, w, epsilon, hidden);
    } else {
        if (vec8) hipLaunchKernelGGL((rms_norm_kernel<8, kNoAdd>), grid, block, 0, st, o, in, res, w, epsilon, hidden);
        else hipLaunchKernelGGL((rms_norm_kernel<1, kNoAdd>), grid, block, 0, st, o, in, res, w, epsilon, hidden);
    }
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : static_cast<int>(e);
}

}  // namespace ca
