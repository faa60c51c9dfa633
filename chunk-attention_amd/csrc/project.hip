// Projections of a batch of token rows for gfx950 (MI355X): y = x . W^T with one to three weights in one
// launch, fp16 data, fp32 sums rounded once.  What the attention layer does around its attention call
// (the reference calls a library for each, src/chunk_attn/models/llama_hf/modeling_llama.py:52-62,111):
//
//   plain     any row-major weights [N, K]: output projection, language-model head
//   rotary    q, k and v of a layer, q and k turned by their positions' angles before they are rounded
//   append    the same for a decode step: k and v go straight to the free row of each sequence's last chunk
//   add       plain, added to other rows once rounded: output projection and residual
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "kernels.h"
#include "norm_math.h"
#include "rotary_math.h"

namespace ca {
namespace {

using rotary::half_t;
using rotary::h4;
using rotary::h8;
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int D = 128;
constexpr int NW = 8;              // waves of a workgroup: each sums its share of k for the whole tile
constexpr int WG = 64 * NW;
constexpr int UNIT = 64;           // k elements a wave takes at a time: one 128-byte line of every row

enum { kPlain = 0, kRotary = 1, kAppend = 2, kAdd = 3 };
constexpr bool turns(int mode) { return mode == kRotary || mode == kAppend; }

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
// LDS, which every wave fills and reads for itself: from there on the waves share their tiles
// (project_tile_kernel; the line is at launch_mode).
//
// Columns of a rotary tile: half of them from the first half of a head, half their partners 64 further on.
// XR: rows of x that are fetched; of a block of 16 the others' products are of whatever stands in LDS, and not stored
// (up to 8 rows a quarter of a unit's loads: q, k and v of 2048 on 1 row 9.1 -> 8.3 us, of 4096 20.9 -> 20.1, one weight
// of 1024 3.0 -> 2.8).
//
// NORM: x is normalised on its way.  Between them the eight waves hold a whole row in registers (at most R units
// each), so its squares cost one exchange over LDS, in the order in which rms_norm adds them (pieces 32, 16, ... 1
// apart, then by 512 elements: the same bits), while the weights are still on their way (q, k and v of 1024 on 8 rows 4.6 -> 5.4
// us, and the norm's launch of 2.6 in front is gone).
template <int MB, int NB, int R, int XR, int MODE, bool NORM>
__global__ __launch_bounds__(WG) void project_kernel(const ProjectArgs a) {
    constexpr int MT = 16 * MB, NT = 16 * NB, PITCH = NT + 4;
    constexpr int ROWS = MT + NT;                    // rows of a unit: the tile's columns (rows of W), then its rows
    __shared__ __attribute__((aligned(16))) union {
        half_t stage[NW][ROWS * UNIT];
        float red[NW][MT][PITCH];
    } sm;
    // squares of the x pieces of a unit: [unit of the wave][load][wave][lane]
    __shared__ float squares[NORM ? R * (XR / 8) * NW * 64 : 1];
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
    const int col0 = !turns(MODE) ? blk * NT : (blk / PER_HEAD) * D + (blk % PER_HEAD) * HALF;
    const int row0 = rb * MT;

    // Load r of a unit brings rows 8r .. 8r+7, eight lanes to the 128 bytes of a row (requested in the
    // matrix cores' layout, neighbouring lanes would lie in different rows, and every lane would cost a
    // look-up of its own).
    constexpr int NL = (NT + XR) / 8;
    const half_t* src[NL];
#pragma unroll
    for (int r = 0; r < NL; r++) {
        if (8 * r < NT) {
            const int c = 8 * r + (l >> 3);
            int n = (!turns(MODE) || c < HALF) ? col0 + c : col0 + c + D / 2 - HALF;
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
    // what is added to this thread's eight products at the end: asked for now
    static_assert(MT * NT / 8 <= WG, "one piece of the output a thread");
    h8 added;
    const bool adds = MODE == kAdd && tid < MT * NT / 8 && row0 + tid / (NT / 8) < a.M && col0 + 8 * (tid % (NT / 8)) < a.N;
    if (adds) added = *reinterpret_cast<const h8*>(static_cast<const half_t*>(a.add) + size_t(row0 + tid / (NT / 8)) * a.N + col0 + 8 * (tid % (NT / 8)));

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
    if constexpr (NORM) {                            // at most R units a wave: all of them now
        constexpr int XL = XR / 8;                   // loads of x a unit, behind those of w
        h8 weight[R];
        if (mine > 0) {
#pragma unroll
            for (int r = 0; r < R; r++) {            // x first: it is waited for first
                const int k0 = (w + NW * (r < mine ? r : mine - 1)) * UNIT;
#pragma unroll
                for (int n = 0; n < XL; n++) st[r][NL - XL + n] = *reinterpret_cast<const h8*>(src[NL - XL + n] + k0);
                weight[r] = *reinterpret_cast<const h8*>(static_cast<const half_t*>(a.norm) + k0 + 8 * (l & 7));
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                const int k0 = (w + NW * (r < mine ? r : mine - 1)) * UNIT;
#pragma unroll
                for (int n = 0; n < NL - XL; n++) st[r][n] = *reinterpret_cast<const h8*>(src[n] + k0);
            }
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
#pragma unroll
            for (int n = 0; n < XL; n++) {
                squares[((r * XL + n) * NW + w) * 64 + l] = r < mine ? norm::sum_of_squares8(st[r][NL - XL + n]) : 0.f;
            }
        }
        __syncthreads();
        float inv[XL];
#pragma unroll
        for (int n = 0; n < XL; n++) {
            float sum = 0.f;
#pragma unroll
            for (int r = 0; r < R; r++) {
                const float* s = &squares[(r * XL + n) * NW * 64 + l];
                float v = ((s[0] + s[4 * 64]) + (s[2 * 64] + s[6 * 64])) + ((s[64] + s[5 * 64]) + (s[3 * 64] + s[7 * 64]));
#pragma unroll
                for (int m = 4; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
                sum = r == 0 ? v : sum + v;
            }
            inv[n] = norm::inverse_rms(sum, a.K, a.norm_epsilon);
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (r < mine) {
#pragma unroll
                for (int n = 0; n < XL; n++) {
                    st[r][NL - XL + n] = norm::scaled8(st[r][NL - XL + n], weight[r], inv[n]);
                    if (MODE == kPlain && blockIdx.x == 0 && a.normed && 8 * n + (l >> 3) < a.M) {   // (one block of rows)
                        half_t* to = static_cast<half_t*>(a.normed) + size_t(8 * n + (l >> 3)) * a.K + (w + NW * r) * UNIT + 8 * (l & 7);
                        *reinterpret_cast<h8*>(to) = st[r][NL - XL + n];
                    }
                }
                multiply(st[r]);
            }
        }
    } else if (mine > 0) {
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

    if constexpr (!turns(MODE)) {
        half_t* y = static_cast<half_t*>(which == 0 ? a.y[0] : which == 1 ? a.y[1] : a.y[2]);
        for (int u = tid; u < MT * NT / 8; u += WG) {
            const int r = u / (NT / 8), c = 8 * (u % (NT / 8));
            if (row0 + r >= a.M || col0 + c >= a.N) continue;
            half_t* dst = y + size_t(row0 + r) * a.N + col0 + c;
            if (MODE == kAdd || a.vec8) {
                h8 o;
#pragma unroll
                for (int e = 0; e < 8; e++) o[e] = half_t(red[0][r][c + e]);
                if (MODE == kAdd) {
#pragma unroll
                    for (int e = 0; e < 8; e++) o[e] = half_t(float(o[e]) + float(added[e]));
                }
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

template <int MB, int NB, int R, int XR, int MODE, bool NORM = false>
int launch_tile(const ProjectArgs& a, hipStream_t st) {
    constexpr int MT = 16 * MB, NT = 16 * NB;
    const int64_t wgs = int64_t((a.N + NT - 1) / NT) * a.n_w * ((int64_t(a.M) + MT - 1) / MT);
    if (wgs > 0x7fffffff) return -1;
    hipLaunchKernelGGL((project_kernel<MB, NB, R, XR, MODE, NORM>), dim3(static_cast<unsigned>(wgs)), dim3(WG), 0, st, a);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : static_cast<int>(e);
}

// ---- many rows: tiles that the waves of a workgroup share --------------------------------------------------------
//
// A workgroup computes BM rows by BN columns; stages of 64 k elements of its rows of x and of w reach LDS by direct
// loads, NBUF - 1 stages ahead, and every wave reads the operands of its BM / WM x CW part from there, one k-step (32)
// ahead of its products, with one barrier a stage.
//
// What bounds it: large products, power.  With every compute unit busy the clock falls to about 1.6 GHz (matrix ops
// on registers alone then reach 1.70 PFLOP/s as 16 x 16 x 32, 1.55 as 32 x 32 x 16, which is why the operands here are
// 16 wide), and every LDS read and fetched line lowers it further: q, k and v of 4096 with their rotation on 2048
// rows 181 us, 1.14 PFLOP/s (187 to 193 on other machines; three library products and the rotary launch 209 to 212; the same stages with all of their
// loads requested in a row behind the barrier 219: a wave issues in order, and its products waited for the loads to
// be taken; with 32 x 32 x 16 195).  One weight of 4096 on 2048 rows 57.6 (the library 64.1).  Smaller ones, the fill
// of the pipeline and a stage's latency: 0.36 us a stage for 128 x 128, 0.56 for 128 x 256 (0.43 is the matrix cores').
// Waves of 64 x 128 or 128 x 64, four to a workgroup, read less from LDS but leave one wave to a SIMD: 226 to 230
// us where eight of 64 x 64 take 181; 256 x 256 tiles 210 to 218 (384 of them on 256 units).
__device__ __forceinline__ void load_to_lds16(const char* src, half_t* dst) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                     (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

constexpr int BK = 64;             // k elements of a stage: one 128-byte line of every row

template <int BM, int BN, int NBUF, int WAVES, int NB, int MODE>
__global__ __launch_bounds__(64 * WAVES, 2) void project_tile_kernel(const ProjectArgs a) {
    constexpr int CW = 16 * NB;                      // columns of a wave
    constexpr int WN = BN / CW, WM = WAVES / WN;
    constexpr int TM = BM / WM;                      // rows of a wave
    constexpr int MB = TM / 16;                      // its 16-row blocks
    constexpr int STAGE = (BM + BN) * BK;            // halves of a stage: the rows of x, then the rows of w
    constexpr int NLD = (BM + BN) / 8 / WAVES;       // loads of a wave a stage, eight rows each
    constexpr int EP = CW + 8;                       // pitch of the output's way through LDS
    __shared__ __attribute__((aligned(16))) half_t lds[NBUF * STAGE];
    static_assert(WAVES * 32 * EP <= NBUF * STAGE && NLD * 8 * WAVES == BM + BN && MB % 2 == 0 && NBUF > 2, "");

    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = w / WN, wn = w % WN;
    const int l = tid & 63, g = l >> 4, i = l & 15;
    // Tiles in groups of eight row tiles, columns inside, dealt to the XCDs (block b runs on XCD b % 8) in
    // contiguous ranges: what an XCD's 32 units work on at a time is about eight row tiles by four column tiles.
    const int per_w = (a.N + BN - 1) / BN;
    const int n_cb = per_w * a.n_w, n_rb = (a.M + BM - 1) / BM;
    const int total = n_cb * n_rb;
    const int xcd = blockIdx.x & 7, q8 = total >> 3, r8 = total & 7;
    const int u = xcd * q8 + (xcd < r8 ? xcd : r8) + (blockIdx.x >> 3);
    constexpr int GM = 8;
    const int grp = u / (GM * n_cb), in_grp = u - grp * GM * n_cb;
    const int g_rows = n_rb - grp * GM < GM ? n_rb - grp * GM : GM;
    const int cb = in_grp / g_rows, rb = grp * GM + in_grp % g_rows;
    const int which = cb / per_w, blk = cb - which * per_w;
    const half_t* __restrict__ wt = static_cast<const half_t*>(which == 0 ? a.w[0] : which == 1 ? a.w[1] : a.w[2]);
    const int row0 = rb * BM, col0 = blk * BN;
    // Column of the weight behind row c of the tile's w part.  Rotary: a wave's columns are CW / 2 of a head's first
    // half and their partners 64 further on, so that a lane holds both.
    auto column = [&](int c) {
        if (!turns(MODE)) return col0 + c;
        const int part = (col0 + c) / CW, in = c % CW;
        return part / (D / CW) * D + part % (D / CW) * (CW / 2) + in % (CW / 2) + in / (CW / 2) * (D / 2);
    };

    const char* xbase = reinterpret_cast<const char*>(static_cast<const half_t*>(a.x) + size_t(row0) * a.K);
    const char* wbase = reinterpret_cast<const char*>(wt);
    unsigned off[NLD];
#pragma unroll
    for (int r = 0; r < NLD; r++) {
        const int lb = w * NLD + r;                  // rows 8 lb .. 8 lb + 7 of the stage
        int row = 8 * lb + (l >> 3);
        const int piece = (l & 7) ^ (l >> 3);        // piece c of row r stands at place c ^ (r & 7), as above
        if (lb < BM / 8) {
            if (row0 + row >= a.M) row = a.M - 1 - row0;          // computed, not stored
        } else {
            row = column(row - BM);
            if (row >= a.N) row = a.N - 1;
        }
        off[r] = (unsigned(row) * unsigned(a.K) + 8 * piece) * 2;
    }
    // One load of stage t; `at`: the stage's buffer.
    auto load = [&](int r, int t, int at) {
        const int lb = w * NLD + r;
        load_to_lds16((lb < BM / 8 ? xbase : wbase) + size_t(t) * (BK * 2) + off[r], &lds[at + lb * 8 * BK]);
    };
    auto fetch = [&](int t, int at) {
#pragma unroll
        for (int r = 0; r < NLD; r++) load(r, t, at);
    };
    f4 acc[MB][NB];
#pragma unroll
    for (int m = 0; m < MB; m++) {
#pragma unroll
        for (int n = 0; n < NB; n++) acc[m][n] = f4{ 0.f, 0.f, 0.f, 0.f };
    }
    h8 xf[2][MB], wf[2][NB];
    const int xrow = (wm * TM + i) * BK, wrow = (BM + wn * CW + i) * BK;
    // Operand o of k-step ks, w's blocks first.
    auto operand = [&](int o, int at, int ks, int set) {
        const half_t* p = &lds[at + 8 * ((4 * ks + g) ^ (i & 7))];
        if (o < NB) wf[set][o] = *reinterpret_cast<const h8*>(p + wrow + o * 16 * BK);
        else xf[set][o - NB] = *reinterpret_cast<const h8*>(p + xrow + (o - NB) * 16 * BK);
    };
    // The products of a k-step on operand set `set`.  Spread between them: the other set's operands (k-step ks of the
    // stage at `at`, if MORE) and N loads of stage t.
    auto step = [&](int set, auto more, int at, int ks, int t, int t_at, auto count) {
        constexpr int PRODUCTS = MB * NB, OPS = MB + NB, N = decltype(count)::value;
#pragma unroll
        for (int k = 0; k < PRODUCTS; k++) {
            if constexpr (decltype(more)::value) {
#pragma unroll
                for (int o = k * OPS / PRODUCTS; o < (k + 1) * OPS / PRODUCTS; o++) operand(o, at, ks, set ^ 1);
            }
#pragma unroll
            for (int r = k * N / PRODUCTS; r < (k + 1) * N / PRODUCTS; r++) load(r, t, t_at);
            const int m = k / NB, n = k % NB;
            acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[set][n], xf[set][m], acc[m][n], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    const int n_t = a.K / BK;
    // Every wave's loads but those of the newest `left` stages have landed, and every wave holds what it has read.
    auto meet = [&](auto left) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(left)::value * NLD) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
#pragma unroll
    for (int s = 0; s < NBUF - 1; s++) {
        if (s < n_t) fetch(s, s * STAGE);
    }
    if (n_t >= NBUF - 1) meet(std::integral_constant<int, NBUF - 2>{});
    else meet(std::integral_constant<int, 0>{});
#pragma unroll
    for (int o = 0; o < MB + NB; o++) operand(o, 0, 0, 0);
    int at = 0, free_at = (NBUF - 1) * STAGE;
    // Stage t.  LOADS: there is a stage t + NBUF - 1 to request; MORE: there is a stage t + 1.
    auto stage_of = [&](int t, auto loads, auto more) {
        constexpr bool LOADS = decltype(loads)::value;
        step(0, std::true_type{}, at, 1, t + NBUF - 1, free_at, std::integral_constant<int, LOADS ? NLD : 0>{});
        // The stage's last operands are in registers: behind the barrier its buffer is free, the next stage has
        // landed, and this stage's last products cover the latency of its first operands.
        meet(std::integral_constant<int, LOADS ? NBUF - 2 : 0>{});
        free_at = at;
        at = at + STAGE == NBUF * STAGE ? 0 : at + STAGE;
        step(1, more, at, 0, 0, 0, std::integral_constant<int, 0>{});
    };
    int t = 0;
    for (; t + NBUF - 1 < n_t; t++) stage_of(t, std::true_type{}, std::true_type{});
    for (; t + 1 < n_t; t++) stage_of(t, std::false_type{}, std::true_type{});
    stage_of(t, std::false_type{}, std::false_type{});
    // the loop's last matrix ops are read behind a branch, where the compiler's own wait states do not reach
    asm volatile("s_nop 15\n\ts_nop 15");
    __builtin_amdgcn_sched_barrier(0);

    // Lane (g, i) holds row i of a 16 x 16 block, columns 4g .. 4g + 3: rounded, and through the wave's own piece of
    // LDS, 32 rows at a time, into whole lines.
    half_t* stage = &lds[w * 32 * EP];
    half_t* y = static_cast<half_t*>(which == 0 ? a.y[0] : which == 1 ? a.y[1] : a.y[2]);
#pragma unroll
    for (int m2 = 0; m2 < MB / 2; m2++) {
        const int row_base = row0 + wm * TM + 32 * m2;
        constexpr int PIECES = CW / 8;
        h8 added[CW / 16];          // asked for before the sums go through LDS
        if constexpr (MODE == kAdd) {
#pragma unroll
            for (int p = 0; p < CW / 16; p++) {
                const int row = row_base + p * (64 / PIECES) + l / PIECES, n = column(wn * CW + 8 * (l % PIECES));
                if (row < a.M && n < a.N) added[p] = *reinterpret_cast<const h8*>(static_cast<const half_t*>(a.add) + size_t(row) * a.N + n);
            }
        }
#pragma unroll
        for (int mm = 0; mm < 2; mm++) {
            const int m = 2 * m2 + mm, row = row_base + 16 * mm + i;
            const half_t* cs = nullptr;
            if (turns(MODE) && which < 2) {
                cs = static_cast<const half_t*>(a.cos_sin_cache) +
                     rotary::clamp_pos(a.positions[row < a.M ? row : a.M - 1], a.max_position) * D + (col0 + wn * CW) % D / 2;
            }
#pragma unroll
            for (int n = 0; n < NB / 2; n++) {
                const int c = 16 * n + 4 * g;
                const f4 f0 = acc[m][n], f1 = acc[m][n + NB / 2];
                h4 o0, o1;
                if (turns(MODE) && which < 2) {
                    const h4 c4 = *reinterpret_cast<const h4*>(cs + c), s4 = *reinterpret_cast<const h4*>(cs + c + D / 2);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        o0[e] = half_t(rotary::rot_elem(f0[e], f1[e], float(c4[e]), float(s4[e]), true));
                        o1[e] = half_t(rotary::rot_elem(f1[e], f0[e], float(c4[e]), float(s4[e]), false));
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        o0[e] = half_t(f0[e]);
                        o1[e] = half_t(f1[e]);
                    }
                }
                *reinterpret_cast<h4*>(&stage[(16 * mm + i) * EP + c]) = o0;
                *reinterpret_cast<h4*>(&stage[(16 * mm + i) * EP + CW / 2 + c]) = o1;
            }
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int p = 0; p < CW / 16; p++) {
            const int r = p * (64 / PIECES) + l / PIECES, c = 8 * (l % PIECES);
            const int row = row_base + r, n = column(wn * CW + c);
            if (row >= a.M || n >= a.N) continue;
            h8 o = *reinterpret_cast<const h8*>(&stage[r * EP + c]);
            if constexpr (MODE == kAdd) {
#pragma unroll
                for (int e = 0; e < 8; e++) o[e] = half_t(float(o[e]) + float(added[p][e]));
            }
            half_t* dst = y + size_t(row) * a.N + n;
            if (MODE == kAppend && which > 0) {
                const int fill = a.tail_fill[row] + a.delta_tokens;
                if (fill < 0 || fill >= a.C) continue;   // the host guarantees a free row; never write outside the chunk
                dst = y + ((size_t(a.tail_slot[row]) * (a.N / D) + n / D) * a.C + fill) * D + n % D;
            }
            if (turns(MODE) || MODE == kAdd || a.vec8) {
                *reinterpret_cast<h8*>(dst) = o;
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    if (n + e < a.N) dst[e] = o[e];
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

template <int BM, int BN, int NBUF, int WAVES, int NB, int MODE>
int launch_shared_tile(const ProjectArgs& a, hipStream_t st) {
    const int64_t wgs = int64_t((a.N + BN - 1) / BN) * a.n_w * ((int64_t(a.M) + BM - 1) / BM);
    if (wgs > 0x7fffffff) return -1;
    hipLaunchKernelGGL((project_tile_kernel<BM, BN, NBUF, WAVES, NB, MODE>), dim3(static_cast<unsigned>(wgs)), dim3(64 * WAVES), 0, st, a);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : static_cast<int>(e);
}

// ---- q, k and v of many rows: tiles of 256 x 384 and 128 x 384 -----------------------------------------------------
//
// The three weights' columns are one row of heads here, of which a workgroup takes three by 256 (MB 8) or 128 (MB 4)
// rows: q, k and v of 4096 on 2048 rows are 256 tiles of 256 x 384, one for each compute unit, where 128 x 256 makes
// three rounds of 48 KB a stage for 4 MFLOP.
// Eight waves of 128 x 96 (64 x 96), two to a SIMD: 192 accumulators of 256 registers, so that a k-step's operands do
// not fit twice.  The six of w stay for a stage and are replaced one by one behind their last product, those of x are
// read two rows of products ahead into four places in turn.  A stage's last reads lie two such rows before its end, and
// what follows them is covered by those rows' products: the barrier behind which its buffer is free and the next
// stage's first operands.  Four stages of 32 k elements fill the LDS: a load has three stages' time to land, and a stage's
// are spread over all of its products (a wave issues in order: in a row, the products wait for them to be taken).
// A wave's columns are three pairs of 16, a head's first half and the partners 64 further on; pair p of the launch is
// pair p % 4 of head p / 4, counted over the weights.
//
// What bounds it: the clock, as above, and 0.3 us of 64 k elements' 1.8 the loads.  4096 x 4096 on 2048 rows 189 -> 161
// us, 1.28 PFLOP/s; on 1024 rows (128 x 384) 118 -> 103; 2048 x 2048 on 3000 rows 87 -> 70.  Two stages of 64 took
// 166, and the results' way out as straight code for every accumulator 170 (20 KB of it, fetched once by each wave).
constexpr int HN = 384;
constexpr int HK = 32;             // k elements of a stage: one k-step

template <int MB>
__global__ __launch_bounds__(512, 2) void project_heads_kernel(const ProjectArgs a) {
#ifdef __HIP_DEVICE_COMPILE__                        // (the host's pass knows no buffer resources, and drops a template that has one)
    constexpr int HM = 32 * MB, WN = 4, NB = 6, PAIRS = NB / 2, CW = 16 * NB, TM = 16 * MB;
    constexpr int STAGE = (HM + HN) * HK * 2;        // bytes
    constexpr int NBUF = 4;
    constexpr int XL = HM / 128, WL = HN / 128;      // loads of a wave a stage, sixteen rows each
    constexpr int NLD = XL + WL, EARLY = 2;           // the first two behind the barrier, the others over the next stage
    constexpr int EP = CW + 4;                       // pitch of the sums' way through LDS
    __shared__ __attribute__((aligned(16))) char lds[NBUF * STAGE];
    static_assert(NLD >= EARLY && MB % 4 == 0 && 8 * 32 * EP * 4 + HM * 4 <= NBUF * STAGE, "");

    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = w / WN, wn = w % WN;
    const int l = tid & 63, g = l >> 4, i = l & 15;
    // tiles to XCDs as above
    const int heads = a.N / D, all_heads = 3 * heads;
    const int n_cb = heads, n_rb = (a.M + HM - 1) / HM;
    const int total = n_cb * n_rb;
    const int xcd = blockIdx.x & 7, q8 = total >> 3, r8 = total & 7;
    const int u = xcd * q8 + (xcd < r8 ? xcd : r8) + (blockIdx.x >> 3);
    constexpr int GM = 8;
    const int grp = u / (GM * n_cb), in_grp = u - grp * GM * n_cb;
    const int g_rows = n_rb - grp * GM < GM ? n_rb - grp * GM : GM;
    const int cb = in_grp / g_rows, rb = grp * GM + in_grp % g_rows;
    const int row0 = rb * HM;
    const int pair0 = cb * (HN / 32);                // the tile's first pair

    // A wave's loads of a stage: rows 16 (XL w + r) .. + 15 of x, then rows 16 (WL w + r) .. + 15 of the tile's columns.
    // As buffer loads: a lane's part of the address is 32 bits (64 would not fit beside the accumulators).  Piece c of
    // row r stands at place c ^ (r >> 2 & 1) * 2: eight rows at two neighbouring pieces lie in different banks.
    int lane_row = l >> 2;
    const int piece = (l & 3) ^ ((l >> 4 & 1) << 1);
    const unsigned last_row = a.M - 1 - row0;        // rows behind it repeat it: computed, not stored
    auto buffer = [](const void* p) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, -1, 0x00020000); };
    const auto xsrc = buffer(static_cast<const half_t*>(a.x) + size_t(row0) * a.K);
    const half_t* wsrc[WL];
#pragma unroll
    for (int r = 0; r < WL; r++) {
        const int part = WL * w + r, block = part % NB;
        const int pair = pair0 + part / NB * PAIRS + block % PAIRS, head = pair >> 2, which = head / heads;
        const int col = (head - which * heads) * D + (pair & 3) * 16 + block / PAIRS * (D / 2);
        wsrc[r] = static_cast<const half_t*>(which == 0 ? a.w[0] : which == 1 ? a.w[1] : a.w[2]) + size_t(col) * a.K;
    }
    const unsigned woff = unsigned(lane_row) * (unsigned(a.K) * 2) + 16 * piece;
    auto load = [&](int r, int t, int at) {          // `at`: the stage's buffer
        auto* dst = (__attribute__((address_space(3))) void*)(lds + at + (r < XL ? XL * w + r : HM / 16 + WL * w + r - XL) * 1024);
        if (r < XL) {
            const unsigned row = min(unsigned(lane_row + 16 * (XL * w + r)), last_row);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xsrc, dst, 16, row * (unsigned(a.K) * 2) + 16 * piece, t * (HK * 2), 0, 0);
            return;
        }
        __builtin_amdgcn_raw_ptr_buffer_load_lds(buffer(wsrc[r - XL]), dst, 16, woff, t * (HK * 2), 0, 0);
    };

    f4 acc[MB][NB];
#pragma unroll
    for (int m = 0; m < MB; m++) {
#pragma unroll
        for (int n = 0; n < NB; n++) acc[m][n] = f4{ 0.f, 0.f, 0.f, 0.f };
    }
    h8 xf[4], wf[NB];
    const int lane = i * (HK * 2) + 16 * (g ^ ((i >> 2 & 1) << 1));
    int xat = wm * TM * (HK * 2) + lane, wat = (HM + wn * CW) * (HK * 2) + lane;
    auto read = [&](int at) { return *reinterpret_cast<const h8*>(lds + at); };

    const int n_t = a.K / HK;
    // Every wave's loads but its newest `left` have landed, and every wave holds what it has read.
    auto meet = [&](auto left) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(left)::value) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
#pragma unroll
    for (int s = 0; s < NBUF; s++) {
#pragma unroll
        for (int r = 0; r < (s < NBUF - 1 ? NLD : EARLY); r++) {
            if (s < n_t) load(r, s, s * STAGE);
        }
    }
    if (n_t >= NBUF) meet(std::integral_constant<int, 2 * NLD + EARLY>{});
    else meet(std::integral_constant<int, 0>{});
#pragma unroll
    for (int n = 0; n < NB; n++) wf[n] = read(wat + n * 1024);
    xf[0] = read(xat);
    xf[1] = read(xat + 1024);
    int here = 0;
    // Stage t in the buffer at `here`.  MORE: there is a stage t + 1; LATE: a stage t + 3, whose last load is still to be
    // asked for; LOADS: a stage t + 4.
    auto stage_of = [&](int t, auto more, auto late, auto loads) {
        constexpr bool MORE = decltype(more)::value, LATE = decltype(late)::value, LOADS = decltype(loads)::value;
        const int next = here + STAGE == NBUF * STAGE ? 0 : here + STAGE, before = here == 0 ? (NBUF - 1) * STAGE : here - STAGE;
        asm volatile("" : "+v"(lane_row));           // the offsets in x are formed where they are used: kept, they are registers
#pragma unroll
        for (int m = 0; m < MB; m++) {
            if (m == MB - 2 && MORE) {
                meet(std::integral_constant<int, LATE ? 2 * NLD : 0>{});
                xat += next - here;
                wat += next - here;
            }
#pragma unroll
            for (int n = 0; n < NB; n++) {
                acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[n], xf[m & 3], acc[m][n], 0, 0, 0);
                if (n == 0 && (m + 2 < MB || MORE)) xf[(m + 2) & 3] = read(xat + (m + 2) % MB * 1024);
                if (m == MB - 1 && MORE) wf[n] = read(wat + n * 1024);
                constexpr int FREE = (MB - 2) * NB, TAIL = 2 * NB;
                const int k = m * NB + n;
#pragma unroll
                for (int r = 0; r < NLD; r++) {
                    if (LATE && r >= EARLY && k == (2 * (r - EARLY) + 1) * FREE / (2 * (NLD - EARLY > 0 ? NLD - EARLY : 1))) load(r, t + NBUF - 1, before);
                    if (LOADS && r < EARLY && k - FREE == (2 * r + 1) * TAIL / (2 * EARLY)) load(r, t + NBUF, here);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        here = next;
    };
    const auto yes = std::true_type{};
    const auto no = std::false_type{};
    int t = 0;
    for (; t + NBUF < n_t; t++) stage_of(t, yes, yes, yes);
    if (t + NBUF == n_t) stage_of(t++, yes, yes, no);
    for (; t + 1 < n_t; t++) stage_of(t, yes, no, no);
    // the rows' positions: on their way during the last stage, then where every lane finds them
    const int64_t own = tid < HM ? a.positions[row0 + tid < a.M ? row0 + tid : a.M - 1] : 0;
    stage_of(t, no, no, no);
    // the loop's last matrix ops are read behind a branch, where the compiler's own wait states do not reach
    asm volatile("s_nop 15\n\ts_nop 15");
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();                                 // every wave is done with the last stage's operands
    int* position = reinterpret_cast<int*>(lds + 8 * 32 * EP * 4);
    if (tid < HM) position[tid] = static_cast<int>(rotary::clamp_pos(own, a.max_position));
    __syncthreads();

    // Lane (g, i) holds row i of a 16 x 16 block, columns 4g .. 4g + 3: through the wave's own piece of LDS, 32 rows at a
    // time, to lanes that hold eight columns of a row and their partners.  One piece of code for all of
    // them: what is run once is fetched once, and straight code for every accumulator took 6 us longer.
    float* sums = reinterpret_cast<float*>(lds) + w * 32 * EP;
    const int pair_w = pair0 + wn * PAIRS;           // the wave's first pair
    auto put = [&](auto block) {
        constexpr int M2 = decltype(block)::value;
#pragma unroll
        for (int mm = 0; mm < 2; mm++) {
#pragma unroll
            for (int n = 0; n < NB; n++) *reinterpret_cast<f4*>(&sums[(16 * mm + i) * EP + 16 * n + 4 * g]) = acc[2 * M2 + mm][n];
        }
    };
#pragma unroll 1
    for (int m2 = 0; m2 < MB / 2; m2++) {
        if (m2 == 0) put(std::integral_constant<int, 0>{});
        if (m2 == 1) put(std::integral_constant<int, 1>{});
        if constexpr (MB > 4) {
            if (m2 == 2) put(std::integral_constant<int, 2>{});
            if (m2 == 3) put(std::integral_constant<int, 3>{});
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int p = 0; p < PAIRS; p++) {
            const int at = p * 64 + l, r = at / (2 * PAIRS), q = at % (2 * PAIRS);
            const int in_tile = wm * TM + 32 * m2 + r, pair = pair_w + (q >> 1), head = pair >> 2;
            const int which = head >= 2 * heads ? 2 : head >= heads ? 1 : 0, d0 = (pair & 3) * 16 + 8 * (q & 1);
            const half_t* cs = static_cast<const half_t*>(a.cos_sin_cache) + size_t(position[in_tile]) * D + d0;
            const h8 c8 = *reinterpret_cast<const h8*>(cs), s8 = *reinterpret_cast<const h8*>(cs + D / 2);
            const float* f = &sums[r * EP + 8 * q];
            float f0[8], f1[8];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                f0[e] = f[e];
                f1[e] = f[CW / 2 + e];
            }
            h8 o0, o1;
            if (which < 2) {
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
            if (row0 + in_tile < a.M) {
                half_t* dst = static_cast<half_t*>(which == 0 ? a.y[0] : which == 1 ? a.y[1] : a.y[2]) +
                              size_t(row0 + in_tile) * a.N + (head - which * heads) * D + d0;
                *reinterpret_cast<h8*>(dst) = o0;
                *reinterpret_cast<h8*>(dst + D / 2) = o1;
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
#endif
}

template <int MB>
int launch_heads(const ProjectArgs& a, hipStream_t st) {
    constexpr int HM = 32 * MB;
    const int64_t wgs = int64_t(a.N) / D * ((int64_t(a.M) + HM - 1) / HM);
    if (wgs > 0x7fffffff) return -1;
    hipLaunchKernelGGL(project_heads_kernel<MB>, dim3(static_cast<unsigned>(wgs)), dim3(512), 0, st, a);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : static_cast<int>(e);
}

// Which of them q, k and v take beside the tiles of 128 x 128 and 128 x 256, of which there are `square` and `wide` rounds:
// the one that the rounds make the shortest; 0 for none.  A round takes so long for each 64 k elements, and at its ends (in
// 1/64 us; the last, partial one of 256 x 384 less, for the clock is higher then).  Measured with each (us in 128 x 128 or
// 128 x 256, 128 x 384, 256 x 384): 4096 x 4096 on 500 rows 62, 96, 121, on 700 102, 97, 119, on 1024 118, 103, 126, on 1200
// 117, 188, 126, on 1500 161, 190, 132, on 2048 189, 216, 161, on 2300 221, 257, 278; 2048 x 2048 on 1000 rows 30, 38, 61, on
// 1500 53, 42, 62, on 2048 56, 51, 63, on 3000 87, 85, 70; 1024 x 1024 on 2000 rows 19, 24, 38, on 4096 35, 30, 40, on 7000
// 55, 53, 46; 5120 x 5120 on 1000 rows 159, 266, 178, on 1300 222, 259, 181.
int heads_shape(const ProjectArgs& a, int64_t square, int64_t wide) {
    constexpr int CUS = 256;
    const int64_t stages = a.K / 64, heads = a.N / D;
    if (square == 1) return 0;
    auto cost = [&](int64_t tiles, int round, int empty, int ends) {
        const int64_t full = tiles / CUS, rest = tiles % CUS;
        return full * (stages * round + ends) + (rest ? stages * (empty + (round - empty) * rest / CUS) + ends : 0);
    };
    const int64_t others = std::min(square * (stages * 39 + 160), wide * (stages * 59 + 160));
    const int64_t tall = cost(heads * ((int64_t(a.M) + 255) / 256), 160, 115, 576);
    const int64_t flat = cost(heads * ((int64_t(a.M) + 127) / 128), 105, 94, 192);
    return std::min(tall, flat) >= others ? 0 : tall < flat ? 8 : 4;
}

// Tiles.  Up to 16 rows: 16 columns a workgroup (three weights of 4096 x 4096, 8 rows: 22.7 us against 26.3 with
// 32 columns; one weight 8.4), three units on their way where a wave has more than two (otherwise they
// would only be asked for again).  More rows: 32 x 32 with k split over the waves while about one of them falls to each
// of the 256 compute units, then the smallest shared tile of which that holds, each stage of it being the shorter
// (us on the GPU, weights from memory, in 32 x 32, 64 x 64, 64 x 128, 128 x 128 tiles: one weight of 1024 on 252 rows
// 4.3, 5.3, 6.5, 7.6; q, k and v of 1024 on 252 rows 8.6, 7.2, 8.9, 11.0, on 512 rows 15.1, 9.1, 9.4, 11.3; one of 4096
// on 64 rows 11.4, 14.9, 19.1, 21.7, on 252 rows 19.6, 15.9, 19.5, 23.3; q, k and v of 4096 on 128 rows 38.8, 38.5, 32.7,
// 41.9, on 192 rows 56.7, 51.3, 57.2, 38.1).  Where even 128 x 256 leaves a second round, the rounds decide, a stage of
// 128 x 128 taking 0.36 us and one of 128 x 256 0.56 (q, k and v of 4096: 700 rows 95.5 and 99.8, 1500 rows 166 and
// 161, 2048 rows 209 and 181).
enum Tile { kRows8, kRows16, k32x32, k64x64Split, k64x64, k64x128, k128x128, k128x256, kHeads128, kHeads256 };

Tile tile_of(const ProjectArgs& a, bool rotary) {
    if (a.M <= 16) return a.M <= 8 ? kRows8 : kRows16;
    auto tiles = [&](int bm, int bn) { return int64_t((a.N + bn - 1) / bn) * a.n_w * ((int64_t(a.M) + bm - 1) / bm); };
    constexpr int CUS = 256;
    if (tiles(32, 32) <= CUS + CUS / 8) return k32x32;
    // Shared tiles reach their rows and columns with 32-bit offsets.  Beyond them the largest tile with k split over
    // the waves, where three quarters of the compute units get one (32768 x 32768 on 65, 252 and 1000 rows 779, 1544 and 6146 us; in
    // 32 x 32 tiles 1134, 2960 and 11711).
    if (int64_t(a.N) * a.K >= int64_t(1) << 30 || a.K > 1 << 22) return 4 * tiles(64, 64) < 3 * CUS ? k32x32 : k64x64Split;
    if (tiles(64, 64) <= CUS) return k64x64;
    if (tiles(64, 128) <= CUS) return k64x128;
    const int64_t square = (tiles(128, 128) + CUS - 1) / CUS, wide = (tiles(128, 256) + CUS - 1) / CUS;
    const int shape = rotary ? heads_shape(a, square, wide) : 0;
    if (shape) return shape == 8 ? kHeads256 : kHeads128;
    return square == 1 || square * 36 < wide * 56 ? k128x128 : k128x256;
}

template <int MODE>
int launch_mode(const ProjectArgs& a, hipStream_t st) {
    if constexpr (MODE == kPlain || MODE == kAppend) {
        if (a.norm) return a.M <= 8 ? launch_tile<1, 1, 2, 8, MODE, true>(a, st) : launch_tile<1, 1, 2, 16, MODE, true>(a, st);
    }
    const bool long_k = a.K > 2 * NW * UNIT;
    switch (tile_of(a, MODE == kRotary)) {
    case kRows8: return long_k ? launch_tile<1, 1, 3, 8, MODE>(a, st) : launch_tile<1, 1, 2, 8, MODE>(a, st);
    case kRows16: return long_k ? launch_tile<1, 1, 3, 16, MODE>(a, st) : launch_tile<1, 1, 2, 16, MODE>(a, st);
    case k32x32: return launch_tile<2, 2, 2, 32, MODE>(a, st);
    case k64x64Split: return launch_tile<4, 4, 2, 64, MODE>(a, st);
    // (five buffers: one weight of 4096 from memory on 100 and 200 rows 18.4 and 19.0 us with four, 16.8 and 17.0 with five, 16.9
    // to 17.5 with six to ten; the larger tiles gain nothing from a fifth)
    case k64x64: return launch_shared_tile<64, 64, 5, 4, 2, MODE>(a, st);
    case k64x128: return launch_shared_tile<64, 128, 4, 8, 2, MODE>(a, st);
    case k128x128: return launch_shared_tile<128, 128, 4, 8, 2, MODE>(a, st);
    case k128x256: return launch_shared_tile<128, 256, 3, 8, 4, MODE>(a, st);
    case kHeads128:
        if constexpr (MODE == kRotary) return launch_heads<4>(a, st);
        break;
    case kHeads256:
        if constexpr (MODE == kRotary) return launch_heads<8>(a, st);
        break;
    }
    return -1;
}

}  // namespace

void project_tile(const ProjectArgs& a, int* rows, int* cols) {
    constexpr int shape[][2] = { { 16, 16 }, { 16, 16 }, { 32, 32 }, { 64, 64 }, { 64, 64 }, { 64, 128 }, { 128, 128 }, { 128, 256 }, { 128, HN }, { 256, HN } };
    const Tile t = tile_of(a, a.positions && !a.tail_slot);
    *rows = shape[t][0];
    *cols = shape[t][1];
}

// One block of rows, two units a wave.
bool project_norms(int M, int K) { return M <= 16 && K <= 2 * NW * UNIT; }

int launch_project(const ProjectArgs& a, hipStream_t st) {
    if (a.M <= 0 || a.N <= 0) return 0;
    if (a.K <= 0 || a.K % UNIT != 0 || a.n_w < 1 || a.n_w > 3 || a.M > 0x7fffff00) return -1;
    if (a.norm && (!project_norms(a.M, a.K) || a.add || (a.positions && !a.tail_slot))) return -1;
    if (a.normed && (!a.norm || a.positions)) return -1;
    if (a.add && (a.n_w != 1 || a.positions || !a.vec8)) return -1;
    if (!a.positions) return a.add ? launch_mode<kAdd>(a, st) : launch_mode<kPlain>(a, st);
    if (a.N % D != 0 || a.n_w != 3) return -1;
    return a.tail_slot ? launch_mode<kAppend>(a, st) : launch_mode<kRotary>(a, st);
}

}  // namespace ca
