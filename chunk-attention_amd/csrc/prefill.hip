// Causal attention over whole prompts for gfx950 (MI355X): the prefill branch of the attention layer
// (the reference computes it with an external attention library,
// src/chunk_attn/models/llama_hf/modeling_llama.py:64-84).  fp16 q/k/v [batch, n, heads, 128], fp32
// scores, softmax and sums, fp16 output rounded once; d_head 128.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "kernels.h"

namespace ca {
namespace {

typedef _Float16 half_t;
typedef half_t h2 __attribute__((ext_vector_type(2)));
typedef half_t h4 __attribute__((ext_vector_type(4)));
typedef half_t h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));

constexpr int D = 128;
constexpr int WG = 256;
constexpr int NW = WG / 64;
constexpr int ROWS = 64;            // query rows of a workgroup
constexpr float NEG_INF = -__builtin_huge_valf();
constexpr float kShift = 8.f;       // probabilities are kept as 2^8 times their value (see below)
constexpr float kSlack = 7.f;       // a row's maximum moves when it grows by more than 2^7 (see below)

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ h4 lds_read_tr(const half_t* p) {
    typedef short s4v __attribute__((ext_vector_type(4)));
    const s4v raw = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s4v __attribute__((address_space(3)))*)p);
    return __builtin_bit_cast(h4, raw);
}

// what fp16 leaves of p: p - a, a the lower or upper half of a register (one instruction; written out, the
// compiler widens the half first)
template <bool UPPER>
__device__ __forceinline__ float rest_of(float p, h2 a) {
    float r;
    if constexpr (UPPER) asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(a), "v"(p));
    else asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(a), "v"(p));
    return r;
}

// IEEE maximum: unlike fmaxf it needs no canonical inputs, and three of them fit one instruction
__device__ __forceinline__ float max2(float a, float b) { return __builtin_elementwise_maximum(a, b); }

// maximum over lanes l, l^16, l^32, l^48 (the four 16-lane groups), in all four
__device__ __forceinline__ float max_over_groups(float v) {
    const unsigned u = __builtin_bit_cast(unsigned, v);
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const unsigned a0 = a[0], a1 = a[1];
    const float m16 = max2(__builtin_bit_cast(float, a0), __builtin_bit_cast(float, a1));
    const unsigned w = __builtin_bit_cast(unsigned, m16);
    const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    const unsigned b0 = b[0], b1 = b[1];
    return max2(__builtin_bit_cast(float, b0), __builtin_bit_cast(float, b1));
}

// K and V tiles in LDS, rows of 256 B without padding (the direct global -> LDS loads write 64
// consecutive 16-byte pieces): piece c of row r stands at place c ^ swizzle(r).  A 16-byte read is served for
// eight lanes of two neighbouring 16-lane groups at a time, i.e. eight rows at two neighbouring pieces, a
// transposed read for eight rows at two pieces too: the swizzle leaves the lowest bit of the piece alone within
// eight rows, so that those sixteen places are all different.
template <int TILE>
struct CausalLds {
    half_t k[2][TILE * D];
    half_t v[2][TILE * D];
};
__device__ __forceinline__ int swizzle(int row) { return ((row & 7) << 1) | ((row >> 3) & 1); }
__device__ __forceinline__ int place(int row, int piece) { return row * D + ((piece ^ swizzle(row)) << 3); }
__device__ __forceinline__ void load_to_lds16(const char* src, half_t* dst) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                     (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

// Up to N chunks' rows of k and v for a cache's pools, copied in the attention's launch by the workgroups behind its own:
// they need the memory, which the attention leaves idle, and start as its first workgroups end.  As a launch of their own
// the rows of 2048 tokens of 32 heads took 11.2 us behind the attention's 64.2, together they take 65 to 70.
template <int N>
struct CopyIn {
    u4* kpool;
    u4* vpool;
    int C, chunk_wgs;                                          // workgroups of a chunk
    CopyChunk chunk[N];
};
template <>
struct CopyIn<0> {};

// Threads that copy one chunk: a thread one piece of 16 bytes of up to four neighbouring tokens.
constexpr int COPY_TOKENS = 4, PIECES = D / 8;
__host__ __device__ __forceinline__ int copy_threads(int H, int C) { return (C + COPY_TOKENS - 1) / COPY_TOKENS * H * PIECES; }

// Workgroup u of those that copy.  All of a thread's loads are on request before its first store.
template <int N>
__device__ __forceinline__ void copy_rows(const half_t* __restrict__ k, const half_t* __restrict__ v, int H, const CopyIn<N>& in, int u) {
    const int e = u / in.chunk_wgs;
    const unsigned id = unsigned(u - e * in.chunk_wgs) * WG + threadIdx.x, row_pieces = unsigned(H) * PIECES;
    const unsigned quad = id / row_pieces, at = id - quad * row_pieces;
    const int t0 = int(quad) * COPY_TOKENS, n = in.chunk[e].n;
    if (t0 >= n) return;
    const u4* __restrict__ ks = reinterpret_cast<const u4*>(k) + (size_t(in.chunk[e].row) + t0) * row_pieces + at;
    const u4* __restrict__ vs = reinterpret_cast<const u4*>(v) + (size_t(in.chunk[e].row) + t0) * row_pieces + at;
    const size_t to = ((size_t(in.chunk[e].slot) * H + at / PIECES) * in.C + t0) * PIECES + at % PIECES;
    u4 kr[COPY_TOKENS], vr[COPY_TOKENS];
#pragma unroll
    for (int j = 0; j < COPY_TOKENS; j++) {          // past the last row that one again: no branch between the loads
        const size_t row = size_t(t0 + j < n ? j : n - 1 - t0) * row_pieces;
        kr[j] = ks[row];
        vr[j] = vs[row];
    }
    asm volatile("" ::: "memory");                   // (a load that only a branch below needs would move there)
#pragma unroll
    for (int j = 0; j < COPY_TOKENS; j++) {
        if (t0 + j < n) {
            in.kpool[to + j * PIECES] = kr[j];
            in.vpool[to + j * PIECES] = vr[j];
        }
    }
}

// The chunks that the attention's launch has no room for.
template <int N>
__global__ __launch_bounds__(WG) void copy_in_kernel(const half_t* __restrict__ k, const half_t* __restrict__ v, int H,
                                                     const CopyIn<N> in) {
    copy_rows(k, v, H, in, blockIdx.x);
}

// A workgroup attends 64 query rows of one (sequence, head): wave w owns 16 of them and keeps their Q^T
// operands and output accumulators in registers; TILE-key tiles of K and V go through LDS, the next tile on
// its way into a second buffer.  S^T = K.Q^T leaves each lane with four keys of one row, which is the operand
// layout O^T = V^T.P^T needs, so probabilities never leave registers.
//
// What bounds it: matrix ops (half of them the second P.V product below) and the vector ops of the softmax are
// about equal, and each wave's run of them is one dependent chain; what hides a chain is another wave.  TILE 32
// holds four workgroups a compute unit (110 registers, 32 KB), 64 two.  32 heads, 2048 tokens: 63.4 us (66.2 with the
// places of the tiles and the clamps at the prompt's end computed in every tile), 3000 tokens 120 (126), 8 x 300
// tokens 21.8 us; 16 heads, 8 x 1000 tokens 62.6 (64.5).  Two blocks of 16 rows a wave, which halve the reads from LDS,
// leave two waves to a SIMD: 67 to 85, 114 to 150, 21 to 30 and 62 to 87.  Long runs of large ones are held back by
// the clock, which falls with what they draw (about 1.7 GHz).
//
// The probabilities are fp32; the matrix cores take fp16.  p = hi + lo with hi = fp16(p) and
// lo = fp16(p - hi) carries 21 bits of p at the price of a second P.V product, and p is scaled by 2^8
// (the row sum likewise, so it cancels) to keep lo of small p above fp16's smallest step.  Against 64
// bits the output is as far off as with fp32 products: its own rounding to fp16 is what remains.
// The maximum a row's scores are taken relative to moves only when it would grow by more than 2^7 (p stays
// below 2^15, inside fp16): the accumulators are rescaled a few times a row instead of at most tiles.
template <int TILE, int N>
__global__ __launch_bounds__(WG, TILE == 32 ? 4 : 2) void causal_attention_kernel(
    const half_t* __restrict__ q, const half_t* __restrict__ k, const half_t* __restrict__ v, half_t* __restrict__ out,
    int n, int H, int n_bh, int n_blocks, float scale_log2, const CopyIn<N> in) {
    const int n_wgs = n_bh * n_blocks;
    if constexpr (N > 0) {
        if (int(blockIdx.x) >= n_wgs) {
            copy_rows(k, v, H, in, blockIdx.x - n_wgs);
            return;
        }
    }
    constexpr int TB = TILE / 16;                              // 16-key blocks of a tile
    constexpr int TP = TILE / 32;                              // pairs of them
    constexpr int RPW = TILE / NW;                             // rows of a tile that a wave brings
    __shared__ __attribute__((aligned(16))) CausalLds<TILE> sm;
    // Query blocks in descending order (the last ones attend most).  Workgroup b runs on XCD b % 8:
    // with a multiple of 8 heads every head stays on one XCD, whose L2 then holds its K and V.
    // Every second 256 workgroups (one per compute unit) are taken in reverse, in steps of 8 so that the
    // XCD does not change: a compute unit gets a long and a short block instead of two long ones.
    int b = blockIdx.x;
    if (((b >> 8) & 1) && (b | 255) < n_wgs) b = (b & ~255) | ((31 - ((b >> 3) & 31)) << 3) | (b & 7);
    const int bh = b % n_bh;
    const int block = n_blocks - 1 - b / n_bh;
    const int seq = bh / H, h = bh - seq * H;
    const size_t stride = size_t(H) * D;                       // halves between tokens
    const size_t base = size_t(seq) * n * stride + size_t(h) * D;

    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l = tid & 63, g = l >> 4, i = l & 15;
    const int q0 = block * ROWS;                               // first row of the workgroup
    const int row0 = q0 + 16 * w;                              // first row of the wave
    const int row = row0 + i;                                  // the lane's row

    h8 qreg[4];
#pragma unroll
    for (int ks = 0; ks < 4; ks++) {
        qreg[ks] = (row < n) ? *reinterpret_cast<const h8*>(q + base + size_t(row) * stride + 32 * ks + 8 * g)
                             : h8{ 0, 0, 0, 0, 0, 0, 0, 0 };
    }
    float m_run = NEG_INF, l_lane = 0.f;
    f4 oacc[8];
#pragma unroll
    for (int db = 0; db < 8; db++) oacc[db] = f4{ 0.f, 0.f, 0.f, 0.f };

    // Wave w brings rows RPW * w and on of a tile, four per load: lane l writes piece l of those 1024 B,
    // i.e. place l & 15 of row l >> 4, and therefore reads piece (l & 15) ^ swizzle(row).  Rows past the last
    // token repeat it (valid memory; their scores are masked for every row).
    unsigned whole[RPW / 4];                                   // bytes from the tile's first row
#pragma unroll
    for (int r = 0; r < RPW / 4; r++) {
        const int kr = RPW * w + 4 * r + g;
        whole[r] = (unsigned(kr) * unsigned(stride) + 8 * (i ^ swizzle(kr))) * 2;
    }
    auto fetch_tile = [&](int t, int buf) {
        const char* __restrict__ kg = reinterpret_cast<const char*>(k + base + size_t(TILE * t) * stride);
        const char* __restrict__ vg = reinterpret_cast<const char*>(v + base + size_t(TILE * t) * stride);
        const int left = n - 1 - TILE * t;
        if (left >= TILE - 1) {
#pragma unroll
            for (int r = 0; r < RPW / 4; r++) {
                load_to_lds16(kg + whole[r], &sm.k[buf][(RPW * w + 4 * r) * D]);
                load_to_lds16(vg + whole[r], &sm.v[buf][(RPW * w + 4 * r) * D]);
            }
            return;
        }
#pragma unroll
        for (int r = 0; r < RPW / 4; r++) {
            unsigned off = whole[r];
            const int kr = RPW * w + 4 * r + g;
            if (kr > left) off -= unsigned(kr - left) * unsigned(stride) * 2;
            load_to_lds16(kg + off, &sm.k[buf][(RPW * w + 4 * r) * D]);
            load_to_lds16(vg + off, &sm.v[buf][(RPW * w + 4 * r) * D]);
        }
    };

    const int last = (q0 + ROWS < n ? q0 + ROWS : n) - 1;      // last query row of the workgroup
    const int n_tiles = last / TILE + 1;

    auto tile_body = [&](int t, const half_t* __restrict__ kt, const half_t* __restrict__ vt, auto masked_tag) {
        constexpr bool MASKED = decltype(masked_tag)::value;   // some key of the tile lies after some row of the wave
        // The places of a row's pieces differ in a few bits of the address: one base a lane, the others by
        // exclusive or, formed where they are used (hoisted out of the loop they cost twelve registers); in bytes, so
        // that nothing but the exclusive or is left of them.
        int kbase = 2 * place(i, g), vbase = 2 * place(4 * g + (i >> 2), (i >> 1) & 1) + 8 * (i & 1);   // bytes
        asm volatile("" : "+v"(kbase), "+v"(vbase));
        f4 sc[TB];
#pragma unroll
        for (int tb = 0; tb < TB; tb++) {
            h8 kop[4];
#pragma unroll
            for (int ks = 0; ks < 4; ks++) kop[ks] = *reinterpret_cast<const h8*>(reinterpret_cast<const char*>(kt) + (kbase ^ (64 * ks)) + 32 * D * tb);
            f4 acc = f4{ 0.f, 0.f, 0.f, 0.f };
#pragma unroll
            for (int ks = 0; ks < 4; ks++) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(kop[ks], qreg[ks], acc, 0, 0, 0);
            sc[tb] = acc;
        }
        if constexpr (MASKED) {  // selects, not branches, between a matrix op and its first reader
#pragma unroll
            for (int tb = 0; tb < TB; tb++) {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    if (TILE * t + 16 * tb + 4 * g + r > row) sc[tb][r] = NEG_INF;
                }
            }
        }
        // online softmax: the scale is positive and rides in the exponent's multiply-add
        float mx = sc[0][0];
#pragma unroll
        for (int e = 1; e < 4 * TB - 1; e += 2) mx = max2(max2(mx, sc[e >> 2][e & 3]), sc[(e + 1) >> 2][(e + 1) & 3]);
        mx = max_over_groups(max2(mx, sc[TB - 1][3]));
        const float m_new = max2(m_run, mx * scale_log2);
        const bool grew = m_new > m_run + kSlack;
        if (__builtin_amdgcn_ballot_w64(grew) != 0) {
            // only the rows that grew: what a row gives must not depend on the rows behind it
            const float alpha = !grew ? 1.f : (m_run == NEG_INF) ? 0.f : fast_exp2(m_run - m_new);
            m_run = grew ? m_new : m_run;
            l_lane *= alpha;
#pragma unroll
            for (int db = 0; db < 8; db++) oacc[db] *= alpha;
        }
        // a row whose scores are all -inf so far has no maximum to subtract
        const float nm = kShift - (m_run == NEG_INF ? 0.f : m_run);
#pragma unroll
        for (int tp = 0; tp < TP; tp++) {
            h8 hi, lo;
            float sum = 0.f;
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                const float p0 = fast_exp2(__builtin_fmaf(sc[2 * tp + (e >> 2)][e & 3], scale_log2, nm));
                const float p1 = fast_exp2(__builtin_fmaf(sc[2 * tp + (e >> 2)][(e & 3) + 1], scale_log2, nm));
                const h2 a = __builtin_bit_cast(h2, __builtin_amdgcn_cvt_pkrtz(p0, p1));
                const h2 c = __builtin_bit_cast(h2, __builtin_amdgcn_cvt_pkrtz(rest_of<false>(p0, a), rest_of<true>(p1, a)));
                hi[e] = a[0];
                hi[e + 1] = a[1];
                lo[e] = c[0];
                lo[e + 1] = c[1];
                sum += p0 + p1;
            }
            l_lane += sum;
#pragma unroll
            for (int half = 0; half < 2; half++) {             // V operands of four dim blocks at a time
                __builtin_amdgcn_sched_barrier(0);
                h8 a[4];
#pragma unroll
                for (int d = 0; d < 4; d++) {                  // rows key and key + 16 are swizzled alike
                    const half_t* p0 = reinterpret_cast<const half_t*>(reinterpret_cast<const char*>(vt) + (vbase ^ (32 * (4 * half + d))) + 64 * D * tp);
                    const h4 x = lds_read_tr(p0), y = lds_read_tr(p0 + 16 * D);
                    a[d] = h8{ x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3] };
                }
#pragma unroll
                for (int d = 0; d < 4; d++) oacc[4 * half + d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[d], hi, oacc[4 * half + d], 0, 0, 0);
#pragma unroll
                for (int d = 0; d < 4; d++) oacc[4 * half + d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[d], lo, oacc[4 * half + d], 0, 0, 0);
            }
        }
    };

    // this wave's pieces of tile t have landed; behind the barrier everyone's have, and everyone is done
    // with the other buffer
    auto arrive = [&](int t) {
        __builtin_amdgcn_s_waitcnt(0x0f70);                    // vmcnt(0)
        __syncthreads();
        if (t + 1 < n_tiles) fetch_tile(t + 1, (t + 1) & 1);
    };
    fetch_tile(0, 0);
    const int n_whole = q0 / TILE;                             // tiles that lie before every row of the workgroup
    int t = 0;
    for (; t + 1 < n_whole; t += 2) {                          // by two: the buffers' places are constants
        arrive(t);
        tile_body(t, sm.k[0], sm.v[0], std::false_type{});
        arrive(t + 1);
        tile_body(t + 1, sm.k[1], sm.v[1], std::false_type{});
    }
    if (t < n_whole) {
        arrive(t);
        tile_body(t, sm.k[0], sm.v[0], std::false_type{});
        t++;
    }
    // The diagonal: waves whose rows all lie before a tile skip it.  Waves begin at multiples of 16, which
    // divides the tile: a wave that takes part has the tile's first key before or at every one of its rows.
    for (; t < n_tiles; t++) {
        arrive(t);
        if (TILE * t <= row0) tile_body(t, sm.k[t & 1], sm.v[t & 1], std::true_type{});
    }

    float sum = l_lane;
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    const float r = 1.f / sum;
    if (row < n) {
        half_t* dst = out + base + size_t(row) * stride + 4 * g;
#pragma unroll
        for (int db = 0; db < 8; db++) {
            const f4 o = oacc[db];
            *reinterpret_cast<h4*>(dst + 16 * db) = h4{ half_t(o[0] * r), half_t(o[1] * r), half_t(o[2] * r), half_t(o[3] * r) };
        }
    }
}

template <int N>
CopyIn<N> copies(const CausalArgs& a) {
    CopyIn<N> in;
    in.kpool = static_cast<u4*>(a.kpool);
    in.vpool = static_cast<u4*>(a.vpool);
    in.C = a.C;
    in.chunk_wgs = (copy_threads(a.n_heads, a.C) + WG - 1) / WG;
    for (int i = 0; i < N; i++) in.chunk[i] = i < a.n_chunks ? a.chunks[i] : CopyChunk{ 0, 0, 0 };
    return in;
}

template <int N>
int launch(const CausalArgs& a, hipStream_t st) {
    const int n_bh = a.batch * a.n_heads, blocks = (a.n_tokens + ROWS - 1) / ROWS;
    const half_t* q = static_cast<const half_t*>(a.q);
    const half_t* k = static_cast<const half_t*>(a.k);
    const half_t* v = static_cast<const half_t*>(a.v);
    half_t* out = static_cast<half_t*>(a.out);
    CopyIn<N> in;
    int64_t wgs = int64_t(n_bh) * blocks;
    if constexpr (N > 0) {
        in = copies<N>(a);
        wgs += int64_t(a.n_chunks) * in.chunk_wgs;
        if (wgs > 0x7fffffff) return -1;
    }
    const dim3 grid(static_cast<unsigned>(wgs)), block(WG);
    // Tiles of 32 keys let four workgroups share a compute unit, tiles of 64 two, with half as many barriers: worth
    // more while few workgroups are left over from two a unit, the longer the prompt the more (us with 64 and 32 keys
    // a tile, workgroups in brackets: 1004 tokens x 16 heads [256] 21.9, 24.8; 1516 x 16 [384] 33.5, 37.6; 1004 x 32
    // [512] 23.5, 25.8; 4 x 236 x 32 [512] 9.5, 9.3; 4 x 556 x 16 [576] 15.8, 17.1; 4 x 300 x 32 [640] 12.4, 11.8;
    // 4 x 620 x 16 [640] 17.6, 18.9; 4 x 364 x 32 [768] 15.9, 14.3; 1516 x 32 [768] 37.7, 42.0; 2028 x 32 [1024]
    // 64.0, 61.5).
    if (int64_t(n_bh) * blocks > (a.n_tokens < 600 ? 576 : 768)) {
        hipLaunchKernelGGL((causal_attention_kernel<32, N>), grid, block, 0, st, q, k, v, out, a.n_tokens, a.n_heads, n_bh, blocks,
                           a.scale_log2, in);
    } else {
        hipLaunchKernelGGL((causal_attention_kernel<64, N>), grid, block, 0, st, q, k, v, out, a.n_tokens, a.n_heads, n_bh, blocks,
                           a.scale_log2, in);
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : static_cast<int>(e);
}

}  // namespace

bool causal_attention_fits(int batch, int n_tokens, int n_heads) {
    const int64_t blocks = (int64_t(n_tokens) + ROWS - 1) / ROWS;
    return int64_t(batch) * n_heads <= 0x7fffff00 / blocks && n_tokens <= 0x7fffff00 - ROWS;
}

int launch_causal_attention(const CausalArgs& a, hipStream_t st) {
    if (a.batch <= 0 || a.n_tokens <= 0 || a.n_heads <= 0) return 0;
    if (!causal_attention_fits(a.batch, a.n_tokens, a.n_heads) || a.n_chunks > kCausalChunks) return -1;
    if (a.n_chunks == 0) return launch<0>(a, st);
    return a.n_chunks <= 8 ? launch<8>(a, st) : launch<kCausalChunks>(a, st);
}

int launch_copy_in(const CausalArgs& a, hipStream_t st) {
    if (a.n_chunks <= 0 || a.n_heads <= 0) return 0;
    if (a.n_chunks > kCausalChunks) return -1;
    const CopyIn<kCausalChunks> in = copies<kCausalChunks>(a);
    const int64_t wgs = int64_t(a.n_chunks) * in.chunk_wgs;
    if (wgs > 0x7fffffff) return -1;
    hipLaunchKernelGGL(copy_in_kernel<kCausalChunks>, dim3(static_cast<unsigned>(wgs)), dim3(WG), 0, st, static_cast<const half_t*>(a.k),
                       static_cast<const half_t*>(a.v), a.n_heads, in);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : static_cast<int>(e);
}

}  // namespace ca
