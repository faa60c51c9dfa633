// Projections of a batch of token rows for gfx950 (MI355X): y = x . W^T with one to three weights in one
// launch, fp16 data, fp32 sums rounded once.  What the attention layer does around its attention call
// (the reference calls a library for each, src/chunk_attn/models/llama_hf/modeling_llama.py:52-62,111):
//
//   plain     any row-major weights [N, K]: output projection, language-model head
//   rotary    q, k and v of a layer, q and k turned by their positions' angles before they are rounded
//   append    the same for a decode step: k and v go straight to the free row of each sequence's last chunk
#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.h"
#include "rotary_math.h"

namespace ca {
namespace {

using rotary::half_t;
using rotary::h8;
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int D = 128;
constexpr int NW = 8;              // waves of a workgroup: each sums its share of k for the whole tile
constexpr int WG = 64 * NW;
constexpr int UNIT = 64;           // k elements a wave takes at a time: one 128-byte line of every row

enum { kPlain = 0, kRotary = 1, kAppend = 2 };

// A workgroup owns 16 * MB rows and 16 * NB columns.  Few rows (a decode batch, one prompt) make this a
// read of the weights: what counts is that all of their bytes are on request at once, so the tile is
// small (every compute unit has one) and k is split over the eight waves instead of being walked by one.
// Waves share nothing until the end: R units of a wave are on their way in registers in turn, the one that
// has come goes through the wave's own LDS into the operands' layout (no barrier), W as the A operand, so
// that a lane ends up with four neighbouring columns of one row; the eight partial tiles are added in LDS.
//
// What bounds it: with few rows the weights' bytes ([32000, 4096] from memory on 1 row 46.5 us, 5.6 TB/s, on 8 rows
// 49.9, on 16 59.6; the library 55.6 to 56.4; the same weight again and again 41 to 42, the library likewise),
// below that the launch and two round trips to memory (1024 x 1024: 3.3 us, the library 4.4; q, k
// and v together 4.3, as three library calls 13.3, the rotary launch not counted); with hundreds of rows
// LDS, which every wave fills and reads for itself, and from some n_rows * n_in on a library product that
// shares its tiles between waves is faster (projection_pays in capi.py has the line).
//
// Columns of a rotary tile: half of them from the first half of a head, half their partners 64 further on.
template <int MB, int NB, int R, int MODE>
__global__ __launch_bounds__(WG) void project_kernel(const ProjectArgs a) {
    constexpr int MT = 16 * MB, NT = 16 * NB, PITCH = NT + 4;
    constexpr int ROWS = MT + NT;                    // rows of a unit: the tile's columns (rows of W), then its rows
    __shared__ __attribute__((aligned(16))) union {
        half_t stage[NW][ROWS * UNIT];
        float red[NW][MT][PITCH];
    } sm;
    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l = tid & 63, g = l >> 4, i = l & 15;
    const int per_w = (a.N + NT - 1) / NT;           // column blocks of one weight
    const int n_cb = per_w * a.n_w;
    const int cb = blockIdx.x % n_cb, rb = blockIdx.x / n_cb;
    const int which = cb / per_w, blk = cb - which * per_w;
    const half_t* __restrict__ wt = static_cast<const half_t*>(which == 0 ? a.w[0] : which == 1 ? a.w[1] : a.w[2]);
    const half_t* __restrict__ x = static_cast<const half_t*>(a.x);
    // column c of the tile in the weight
    constexpr int HALF = NT / 2;
    constexpr int PER_HEAD = D / NT;                 // rotary tiles of a head
    const int col0 = (MODE == kPlain) ? blk * NT : (blk / PER_HEAD) * D + (blk % PER_HEAD) * HALF;
    const int row0 = rb * MT;

    // Load r of a unit brings rows 8r .. 8r+7, eight lanes to the 128 bytes of a row (requested in the
    // matrix cores' layout, neighbouring lanes would lie in different rows, and every lane would cost a
    // look-up of its own).
    constexpr int NL = ROWS / 8;
    const half_t* src[NL];
#pragma unroll
    for (int r = 0; r < NL; r++) {
        if (8 * r < NT) {
            const int c = 8 * r + (l >> 3);
            int n = (MODE == kPlain || c < HALF) ? col0 + c : col0 + c + D / 2 - HALF;
            if (n >= a.N) n = a.N - 1;               // computed, not stored
            src[r] = wt + size_t(n) * a.K + 8 * (l & 7);
        } else {
            int m = row0 + 8 * r - NT + (l >> 3);
            if (m >= a.M) m = a.M - 1;
            src[r] = x + size_t(m) * a.K + 8 * (l & 7);
        }
    }
    f4 acc[MB][NB];
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
#pragma unroll
        for (int nb = 0; nb < NB; nb++) acc[mb][nb] = f4{ 0.f, 0.f, 0.f, 0.f };
    }

    const int units = a.K / UNIT;
    const int mine = (units - w + NW - 1) / NW;      // of them this wave's: w, w + NW, ...
    h8 st[R][NL];
    auto load = [&](int u, h8 (&d)[NL]) {
        // past the wave's last unit that one again (cached, not used): every step issues the same loads
        const int k0 = (w + NW * (u < mine ? u : mine - 1)) * UNIT;
#pragma unroll
        for (int r = 0; r < NL; r++) d[r] = *reinterpret_cast<const h8*>(src[r] + k0);
    };
    // Through the wave's own piece of LDS into the matrix cores' layout: piece p of row r stands at place
    // p ^ (r & 7), which spreads the eight rows that a read touches at one column over the banks.
    half_t* stage = sm.stage[w];
    auto multiply = [&](const h8 (&d)[NL]) {
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < NL; r++) {
            *reinterpret_cast<h8*>(&stage[(8 * r + (l >> 3)) * UNIT + 8 * ((l & 7) ^ (l >> 3))]) = d[r];
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            const half_t* p = &stage[i * UNIT + 8 * ((4 * ks + g) ^ (i & 7))];
            h8 wr[NB], xr[MB];
#pragma unroll
            for (int nb = 0; nb < NB; nb++) wr[nb] = *reinterpret_cast<const h8*>(p + 16 * nb * UNIT);
#pragma unroll
            for (int mb = 0; mb < MB; mb++) xr[mb] = *reinterpret_cast<const h8*>(p + (NT + 16 * mb) * UNIT);
#pragma unroll
            for (int nb = 0; nb < NB; nb++) {
#pragma unroll
                for (int mb = 0; mb < MB; mb++) {
                    acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wr[nb], xr[mb], acc[mb][nb], 0, 0, 0);
                }
            }
        }
    };
    if (mine > 0) {
#pragma unroll
        for (int r = 0; r + 1 < R; r++) load(r, st[r]);
        for (int u = 0; u < mine; u += R) {
#pragma unroll
            for (int r = 0; r < R; r++) {
                load(u + r + R - 1, st[(r + R - 1) % R]);
                if (r == 0 || u + r < mine) multiply(st[r]);
            }
        }
    }
    // the loop's last matrix ops are read behind a branch, where the compiler's own wait states do not reach
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 15\n\ts_nop 15");
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    auto& red = sm.red;
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
#pragma unroll
        for (int nb = 0; nb < NB; nb++) *reinterpret_cast<f4*>(&red[w][16 * mb + i][16 * nb + 4 * g]) = acc[mb][nb];
    }
    __syncthreads();
    for (int u = tid; u < MT * NT / 4; u += WG) {
        const int r = u / (NT / 4), c = 4 * (u % (NT / 4));
        f4 s = *reinterpret_cast<const f4*>(&red[0][r][c]);
#pragma unroll
        for (int k = 1; k < NW; k++) s += *reinterpret_cast<const f4*>(&red[k][r][c]);
        *reinterpret_cast<f4*>(&red[0][r][c]) = s;
    }
    __syncthreads();

    if constexpr (MODE == kPlain) {
        half_t* __restrict__ y = static_cast<half_t*>(which == 0 ? a.y[0] : which == 1 ? a.y[1] : a.y[2]);
        for (int u = tid; u < MT * NT / 8; u += WG) {
            const int r = u / (NT / 8), c = 8 * (u % (NT / 8));
            if (row0 + r >= a.M || col0 + c >= a.N) continue;
            half_t* dst = y + size_t(row0 + r) * a.N + col0 + c;
            if (a.vec8) {
                h8 o;
#pragma unroll
                for (int e = 0; e < 8; e++) o[e] = half_t(red[0][r][c + e]);
                *reinterpret_cast<h8*>(dst) = o;
            } else {
                for (int e = 0; e < 8 && col0 + c + e < a.N; e++) dst[e] = half_t(red[0][r][c + e]);
            }
        }
        return;
    }
    // one thread: 8 columns and their 8 partners of one row
    for (int u = tid; u < MT * HALF / 8; u += WG) {
        const int r = u / (HALF / 8), c = 8 * (u % (HALF / 8));
        const int row = row0 + r;
        if (row >= a.M) continue;
        float f0[8], f1[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            f0[e] = red[0][r][c + e];
            f1[e] = red[0][r][HALF + c + e];
        }
        const int head = col0 / D, d0 = col0 % D + c;
        h8 o0, o1;
        if (which < 2) {
            const half_t* cs = static_cast<const half_t*>(a.cos_sin_cache) + rotary::clamp_pos(a.positions[row], a.max_position) * D + d0;
            const h8 c8 = *reinterpret_cast<const h8*>(cs), s8 = *reinterpret_cast<const h8*>(cs + D / 2);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                o0[e] = half_t(rotary::rot_elem(f0[e], f1[e], float(c8[e]), float(s8[e]), true));
                o1[e] = half_t(rotary::rot_elem(f1[e], f0[e], float(c8[e]), float(s8[e]), false));
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                o0[e] = half_t(f0[e]);
                o1[e] = half_t(f1[e]);
            }
        }
        half_t* dst;
        if (MODE == kRotary || which == 0) {
            dst = static_cast<half_t*>(which == 0 ? a.y[0] : which == 1 ? a.y[1] : a.y[2]) + size_t(row) * a.N + head * D + d0;
        } else {
            const int fill = a.tail_fill[row] + a.delta_tokens;
            if (fill < 0 || fill >= a.C) continue;   // the host guarantees a free row; never write outside the chunk
            dst = static_cast<half_t*>(which == 1 ? a.y[1] : a.y[2]) +
                  ((size_t(a.tail_slot[row]) * (a.N / D) + head) * a.C + fill) * D + d0;
        }
        *reinterpret_cast<h8*>(dst) = o0;
        *reinterpret_cast<h8*>(dst + D / 2) = o1;
    }
}

template <int MB, int NB, int R, int MODE>
int launch_tile(const ProjectArgs& a, hipStream_t st) {
    constexpr int MT = 16 * MB, NT = 16 * NB;
    const int64_t wgs = int64_t((a.N + NT - 1) / NT) * a.n_w * ((int64_t(a.M) + MT - 1) / MT);
    if (wgs > 0x7fffffff) return -1;
    hipLaunchKernelGGL((project_kernel<MB, NB, R, MODE>), dim3(static_cast<unsigned>(wgs)), dim3(WG), 0, st, a);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : static_cast<int>(e);
}

// Tiles.  Up to 16 rows: 16 columns a workgroup (three weights of 4096 x 4096, 8 rows: 22.7 us against 26.3 with
// 32 columns; one weight 8.4), three units on their way where a wave has more than two (otherwise they
// would only be asked for again).  More rows: 64 x 64, unless that leaves a quarter of the 256 compute units
// without a workgroup (one weight of 1024 x 1024, 252 rows: 4.7 us in 32 x 32 tiles, 13.7 in 64 x 64).
template <int MODE>
int launch_mode(const ProjectArgs& a, hipStream_t st) {
    if (a.M <= 16) {
        return a.K > 2 * NW * UNIT ? launch_tile<1, 1, 3, MODE>(a, st) : launch_tile<1, 1, 2, MODE>(a, st);
    }
    const int64_t big = int64_t((a.N + 63) / 64) * a.n_w * ((int64_t(a.M) + 63) / 64);
    return big < 192 ? launch_tile<2, 2, 2, MODE>(a, st) : launch_tile<4, 4, 2, MODE>(a, st);
}

}  // namespace

int launch_project(const ProjectArgs& a, hipStream_t st) {
    if (a.M <= 0 || a.N <= 0) return 0;
    if (a.K <= 0 || a.K % UNIT != 0 || a.n_w < 1 || a.n_w > 3 || a.M > 0x7fffff00) return -1;
    if (!a.positions) return launch_mode<kPlain>(a, st);
    if (a.N % D != 0 || a.n_w != 3) return -1;
    return a.tail_slot ? launch_mode<kAppend>(a, st) : launch_mode<kRotary>(a, st);
}

}  // namespace ca
