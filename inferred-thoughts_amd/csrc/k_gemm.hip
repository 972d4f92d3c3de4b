// Batched (prefill) matmuls on the int8 matrix cores.
//
// out[t][j] = sum_b (float)isum(t, j, b) * (dw[j][b] * dx[t][b]), b ascending: the per-block
// integer dot of the reference's Q8_0 x Q8_0 product (src/quant/dot.rs), formed by one
// v_mfma_i32_16x16x32_i8 per 32-element block with a zero accumulator, then scaled and added
// in f32 in block order.  The arithmetic and its order are the GEMV kernels' and the CPU
// path's, so results are bit-identical; what changes is that a weight row is read once per
// 128 tokens instead of once per token.
//
// MFMA operand layout (16x16x32, i8): lane l supplies 8 consecutive k of row (l % 16) at
// k = 8 * (l / 16) for both A (weight rows) and B (tokens); it receives D for token l % 16
// and weight rows 4 * (l / 16) + {0,1,2,3}.
#include <algorithm>
#include <type_traits>

#include "it_device.h"
#include "it_dot.h"
#include "it_launch.h"
#include "kernels.h"

namespace itk {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
constexpr int GT = 256;    // four waves: four groups of 16 weight rows
constexpr int SLAB = 128;  // k per staging step: four Q8_0 blocks
constexpr int LSTR = SLAB + 8;  // LDS row stride in bytes (padded)

// A block owns 64 weight rows x NT*16 tokens.  Each step stages a 128-wide k slab of both
// operands and their block scales into LDS with coalesced 16-byte loads (the next slab's
// loads are in flight while the current one is multiplied), then every wave runs its 16 rows
// against all token tiles: one MFMA per (block, tile), four scaled adds per lane after it.
template <int NT, bool FMA = false>
__global__ __launch_bounds__(GT) void q8_gemm_k(const int8_t* __restrict__ wq, const uint16_t* __restrict__ ws,
                                                const int8_t* __restrict__ xq, const float* __restrict__ xs,
                                                float* __restrict__ out, int n_in, int n_out, int n_tok,
                                                float out_scale) {
    constexpr int TOK = NT * 16;
    constexpr int BL = (TOK * 8 + GT - 1) / GT;      // 16-byte loads per thread for the token slab
    constexpr int BS = (TOK * 4 + GT - 1) / GT;      // scale loads per thread for the token slab
    __shared__ __align__(16) int8_t As[2][64 * LSTR];
    __shared__ __align__(16) int8_t Bs[2][TOK * LSTR];
    __shared__ uint16_t Asc[2][64 * 4];
    __shared__ float Bsc[2][TOK * 4];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 15, g = lane >> 4;
    const int row0 = blockIdx.x * 64, tok0 = blockIdx.y * TOK;
    const int nb = n_in >> 5;
    const int nslab = (n_in + SLAB - 1) / SLAB;

    uint4 ra[2], rb[BL];
    uint16_t rsa;
    float rsb[BS];
    auto fetch = [&](int s) {
        const int k0 = s * SLAB;
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const int idx = tid + p * GT, row = idx >> 3, seg = idx & 7;
            const int k = k0 + seg * 16;
            ra[p] = k < n_in ? *(const uint4*)(wq + (int64_t)min(row0 + row, n_out - 1) * n_in + k) : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int p = 0; p < BL; p++) {
            const int idx = tid + p * GT, tok = idx >> 3, seg = idx & 7;
            const int k = k0 + seg * 16;
            rb[p] = (tok < TOK && k < n_in) ? *(const uint4*)(xq + (int64_t)min(tok0 + tok, n_tok - 1) * n_in + k)
                                            : make_uint4(0, 0, 0, 0);
        }
        {
            const int row = tid >> 2, bi = tid & 3, bb = s * 4 + bi;
            rsa = bb < nb ? ws[(int64_t)min(row0 + row, n_out - 1) * nb + bb] : (uint16_t)0;
        }
#pragma unroll
        for (int p = 0; p < BS; p++) {
            const int idx = tid + p * GT, tok = idx >> 2, bi = idx & 3, bb = s * 4 + bi;
            rsb[p] = (tok < TOK && bb < nb) ? xs[(int64_t)min(tok0 + tok, n_tok - 1) * nb + bb] : 0.0f;
        }
    };
    auto stash = [&](int buf) {
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const int idx = tid + p * GT, row = idx >> 3, seg = idx & 7;
            *(uint4*)(As[buf] + row * LSTR + seg * 16) = ra[p];
        }
#pragma unroll
        for (int p = 0; p < BL; p++) {
            const int idx = tid + p * GT, tok = idx >> 3, seg = idx & 7;
            if (tok < TOK) *(uint4*)(Bs[buf] + tok * LSTR + seg * 16) = rb[p];
        }
        Asc[buf][tid] = rsa;
#pragma unroll
        for (int p = 0; p < BS; p++) {
            const int idx = tid + p * GT;
            if (idx < TOK * 4) Bsc[buf][idx] = rsb[p];
        }
    };

    float acc[NT][4];
#pragma unroll
    for (int tt = 0; tt < NT; tt++)
#pragma unroll
        for (int i = 0; i < 4; i++) acc[tt][i] = 0.0f;

    fetch(0);
    stash(0);
    __syncthreads();
    for (int s = 0; s < nslab; s++) {
        const int buf = s & 1;
        if (s + 1 < nslab) fetch(s + 1);
        const int nblk = min(4, nb - s * 4);
        for (int bi = 0; bi < nblk; bi++) {
            const long a = *(const long*)(As[buf] + (wave * 16 + m) * LSTR + bi * 32 + g * 8);
            float dw[4];
#pragma unroll
            for (int i = 0; i < 4; i++) dw[i] = it_f16_to_f32(Asc[buf][(wave * 16 + 4 * g + i) * 4 + bi]);
#pragma unroll
            for (int tt = 0; tt < NT; tt++) {
                const long bv = *(const long*)(Bs[buf] + (tt * 16 + m) * LSTR + bi * 32 + g * 8);
                const float dx = Bsc[buf][(tt * 16 + m) * 4 + bi];
                const v4i z = {0, 0, 0, 0};
                const v4i d = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, bv, z, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if (FMA) acc[tt][i] = fmaf((float)d[i], dw[i] * dx, acc[tt][i]);
                    else acc[tt][i] += (float)d[i] * (dw[i] * dx);
                }
            }
        }
        if (s + 1 < nslab) stash(buf ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int tt = 0; tt < NT; tt++) {
        const int t = tok0 + tt * 16 + m;
        if (t >= n_tok) continue;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int j = row0 + wave * 16 + 4 * g + i;
            if (j < n_out) out[(int64_t)t * n_out + j] = out_scale != 1.0f ? acc[tt][i] * out_scale : acc[tt][i];
        }
    }
}

// ------------------------------------------------------------------ rows of whole 256-wide slabs
// The same products where n_in is a multiple of 256, staged by loads that go from memory straight to LDS.  A block owns 64
// weight rows x 16 NT tokens; a stage is 256 k (eight blocks' scales are one 16-byte load), two of them in LDS.  The kernel
// above has one slab of 128 in flight, in registers, and stores it between the products of two slabs: on a batch of some
// dozen to some hundred tokens every slab waits out most of a trip to memory.  Here a stage is asked for as soon as its
// buffer has been read and costs no register, no store and one barrier for 256 k.  Such a load writes its lanes' 16 bytes
// side by side, so a row's sixteen pieces are permuted by the row's number instead of being padded apart: sixteen rows' reads
// of a piece start in different banks.  The arithmetic is the same, product by product, in the same order.
// For the few-token end, where it is bound by the stages' latency (from some 500 tokens on by the twelve vector operations per
// product, for which there is the kernel below).  8192 x 2048 over 64 tokens: 18.1 -> 11.2 us; 4096 x 2048 over 64 / 201: 16.0 -> 9.3,
// 24.9 -> 15.4; 2048 x 4096 over 64 / 201 / 512: 28.5 -> 15.8, 32.4 -> 18.7, 41.2 -> 27.4.  Three or four stages: 0 to 50 % slower everywhere, fewer
// blocks fit a CU.  The f16 matrix cores with the activations as an f16 pair and no scale per token, 128 x 256 tiles: 437 us for 8192 x 2048 over
// 5,700, and 20 % behind on everything smaller.
typedef _Float16 hv8 __attribute__((ext_vector_type(8)));

template <int NT> constexpr int tile_stage_bytes() { return 64 * 256 + NT * 16 * 256 + 1024 + 1024; }

template <int NT, bool FMA>
__global__ __launch_bounds__(256) void q8_tile_k(const int8_t* __restrict__ wq, const uint16_t* __restrict__ ws,
                                                 const int8_t* __restrict__ xq, const float* __restrict__ xs,
                                                 float* __restrict__ out, int n_in, int n_out, int n_tok, float out_scale) {
    constexpr int STAGE = tile_stage_bytes<NT>(), X_AT = 64 * 256, WS_AT = X_AT + NT * 16 * 256, XS_AT = WS_AT + 1024;
    extern __shared__ __align__(1024) uint8_t tlds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 15, g = lane >> 4;
    const int row0 = blockIdx.x * 64, tok0 = blockIdx.y * NT * 16;
    const int nb = n_in >> 5, n_stage = n_in >> 8;
    const uint32_t at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lptr)tlds);

    // what this lane fetches every stage: four weight rows, NT token rows, and for the first waves a row's scales
    const int8_t* wp[4];
    const int8_t* xp[NT];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int row = (wave * 4 + i) * 4 + (lane >> 4);
        wp[i] = wq + (int64_t)min(row0 + row, n_out - 1) * n_in + (((lane & 15) ^ (row & 15)) << 4);
    }
#pragma unroll
    for (int i = 0; i < NT; i++) {
        const int row = (wave * NT + i) * 4 + (lane >> 4);
        xp[i] = xq + (int64_t)min(tok0 + row, n_tok - 1) * n_in + (((lane & 15) ^ (row & 15)) << 4);
    }
    const bool has_scales = wave < 2;
    const uint8_t* sp = wave == 0 ? (const uint8_t*)(ws + (int64_t)min(row0 + lane, n_out - 1) * nb)
                                  : (const uint8_t*)(xs + (int64_t)min(tok0 + min(lane >> 1, NT * 16 - 1), n_tok - 1) * nb + 4 * (lane & 1));
    const int s_step = wave == 0 ? 16 : 32;
    auto ask = [&](int s, int buf) __attribute__((always_inline)) {
        const uint32_t d = at + buf * STAGE;
#pragma unroll
        for (int i = 0; i < 4; i++) to_lds(wp[i] + s * 256, d + (wave * 4 + i) * 1024);
#pragma unroll
        for (int i = 0; i < NT; i++) to_lds(xp[i] + s * 256, d + X_AT + (wave * NT + i) * 1024);
        if (has_scales) to_lds(sp + s * s_step, d + WS_AT + wave * 1024);
    };
    float acc[NT][4];
#pragma unroll
    for (int tt = 0; tt < NT; tt++)
#pragma unroll
        for (int i = 0; i < 4; i++) acc[tt][i] = 0.0f;

    ask(0, 0);
    for (int s = 0; s < n_stage; s++) {
        const int buf = s & 1;
        __builtin_amdgcn_s_waitcnt(0x0070);      // stage s has landed (vmcnt 0), and this wave has what it read of the last one (lgkmcnt 0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (s + 1 < n_stage) ask(s + 1, buf ^ 1);      // (every wave has read that buffer)
        const uint8_t* const d = tlds + buf * STAGE;
        hv8 dw[4];
#pragma unroll
        for (int i = 0; i < 4; i++) dw[i] = *(const hv8*)(d + WS_AT + (wave * 16 + 4 * g + i) * 16);
#pragma unroll
        for (int b4 = 0; b4 < 2; b4++) {
            float4 dx[NT];
#pragma unroll
            for (int tt = 0; tt < NT; tt++) dx[tt] = *(const float4*)(d + XS_AT + (tt * 16 + m) * 32 + b4 * 16);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int b = 4 * b4 + q, piece = ((2 * b + (g >> 1)) ^ m) << 4;
                const long a = *(const long*)(d + (wave * 16 + m) * 256 + piece + 8 * (g & 1));
                float w[4];
#pragma unroll
                for (int i = 0; i < 4; i++) w[i] = (float)dw[i][b];
#pragma unroll
                for (int tt = 0; tt < NT; tt++) {
                    const long bv = *(const long*)(d + X_AT + (tt * 16 + m) * 256 + piece + 8 * (g & 1));
                    const float x = q == 0 ? dx[tt].x : q == 1 ? dx[tt].y : q == 2 ? dx[tt].z : dx[tt].w;
                    const v4i z = {0, 0, 0, 0};
                    const v4i c = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, bv, z, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        if (FMA) acc[tt][i] = fmaf((float)c[i], w[i] * x, acc[tt][i]);
                        else acc[tt][i] += (float)c[i] * (w[i] * x);
                    }
                }
            }
        }
    }
#pragma unroll
    for (int tt = 0; tt < NT; tt++) {
        const int t = tok0 + tt * 16 + m, j = row0 + wave * 16 + 4 * g;
        if (t >= n_tok) continue;
        float* o = out + (int64_t)t * n_out + j;
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (out_scale != 1.0f) acc[tt][i] *= out_scale;
        if (j + 3 < n_out && !(n_out & 3)) {
            *(float4*)o = make_float4(acc[tt][0], acc[tt][1], acc[tt][2], acc[tt][3]);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (j + i < n_out) o[i] = acc[tt][i];
        }
    }
}

// ------------------------------------------------------------------ ... and enough of them: 32 x 32 products, 128 rows a block
// A block owns 128 weight rows x 32 TT tokens; each of its four waves takes 32 rows against all the tokens by MFMA 32x32x32, so a
// block of 32 k of two tiles is one instruction with a lane's sixteen results behind it.  Lane l supplies 16 k, of its half
// l / 32, of row (or token) l % 32 and receives D[8 (i / 4) + 4 (l / 32) + i % 4][l % 32], i = 0..15.  The sixteen factors dw * dx are a
// product of the matrix cores too: both are f16, so that a 32x32x16_f16 with the row's scale and the token's as its one k
// gives the exact products in the same lanes (operands: one 8-byte read a row and a token a stage, a mask a product).  A
// stage is 128 k and there are two; what of the next one a wave brings is asked for between the products of this one, a request a
// product.
// Bound by the two vector operations (convert, multiply-add; three in exact mode) of every product and the matrix cores' two
// instructions, which two waves of a SIMD overlap in part: 8192 x 2048 over 5,700 tokens 293 us, of which 271 remain without
// loads and 250 without the factors' product (312 with the factors on the vector ALU); 4096 x 2048: 163 -> 153; 2048 x 4096: 176 -> 160;
// 8192 x 2048 over 512 and 1,500: 37.5 -> 36, 94 -> 87.  The product of a tile is started before the last tile's is scaled (the
// compiler alone waited for each), and the outputs go through LDS to be stored 512 bytes a token.  Where in a unit the factors'
// product stands, and two or four requests a product, made no difference.  The arithmetic is the CPU path's, product by
// product, in the same order.
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
constexpr int WIDE_ROWS = 128, WIDE_K = 128;
template <int TT> constexpr int wide_stage_bytes() { return (WIDE_ROWS + 32 * TT) * (WIDE_K + 8); }

template <int TT, bool FMA>
__global__ __launch_bounds__(256, 2) void q8_wide_k(const int8_t* __restrict__ wq, const uint16_t* __restrict__ ws,
                                                    const int8_t* __restrict__ xq, const float* __restrict__ xs,
                                                    float* __restrict__ out, int n_in, int n_out, int n_tok, float out_scale) {
    constexpr int STAGE = wide_stage_bytes<TT>(), X_AT = WIDE_ROWS * WIDE_K, WS_AT = X_AT + 32 * TT * WIDE_K, XS_AT = WS_AT + WIDE_ROWS * 8;
    extern __shared__ __align__(1024) uint8_t tlds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c32 = lane & 31, half = lane >> 5, turn = (c32 >> 1) & 7;
    const int row0 = blockIdx.x * WIDE_ROWS, tok0 = blockIdx.y * 32 * TT;
    const int nb = n_in >> 5, n_stage = n_in / WIDE_K;
    const uint32_t at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lptr)tlds);
    const int8_t* const wbase = wq + (int64_t)row0 * n_in;
    const int8_t* const xbase = xq + (int64_t)tok0 * n_in;

    // what this lane fetches every stage: a piece of four weight rows and of TT token rows, and four scales of a row
    uint32_t wo[4], xo[TT];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int row = (wave * 4 + i) * 8 + (lane >> 3);
        wo[i] = (uint32_t)min(row, n_out - 1 - row0) * n_in + (((lane & 7) ^ ((row >> 1) & 7)) << 4);
    }
#pragma unroll
    for (int i = 0; i < TT; i++) {
        const int row = (wave * TT + i) * 8 + (lane >> 3);
        xo[i] = (uint32_t)min(row, n_tok - 1 - tok0) * n_in + (((lane & 7) ^ ((row >> 1) & 7)) << 4);
    }
    const bool of_w = wave < 2;       // which scales: of the 128 rows, or of the tokens
    const int s_row = of_w ? tid : min(tid - 128, 32 * TT - 1);
    const uint8_t* const sp = of_w ? (const uint8_t*)(ws + (int64_t)min(row0 + s_row, n_out - 1) * nb) : (const uint8_t*)(xs + (int64_t)min(tok0 + s_row, n_tok - 1) * nb);
    auto ask = [&](int s, int buf, int i) __attribute__((always_inline)) {
        const uint32_t d = at + buf * STAGE;
        if (i < 4) to_lds_at(wbase + s * WIDE_K, wo[i & 3], d + (wave * 4 + i) * 1024);
        else to_lds_at(xbase + s * WIDE_K, xo[(i - 4) % TT], d + X_AT + (wave * TT + i - 4) * 1024);
    };
    uint2 sc;                                     // four blocks' scales, f16
    auto load_scales = [&](int s) __attribute__((always_inline)) {
        if (of_w) {
            sc = *(const uint2*)(sp + s * 8);
        } else {
            typedef _Float16 hv4 __attribute__((ext_vector_type(4)));
            const float4 v = *(const float4*)(sp + s * 16);       // (f16 values)
            sc = __builtin_bit_cast(uint2, hv4{(_Float16)v.x, (_Float16)v.y, (_Float16)v.z, (_Float16)v.w});
        }
    };
    auto put_scales = [&](int buf) __attribute__((always_inline)) {
        if (of_w || tid - 128 < 32 * TT) *(uint2*)(tlds + buf * STAGE + (of_w ? WS_AT : XS_AT) + 8 * s_row) = sc;
    };
    const uint32_t lo16 = half ? 0u : 0xffffu, hi16 = half ? 0u : 0xffff0000u;   // lanes of the first half supply k 0 .. 7
    float acc[TT][16];
#pragma unroll
    for (int tt = 0; tt < TT; tt++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[tt][i] = 0.0f;

#pragma unroll
    for (int i = 0; i < 4 + TT; i++) ask(0, 0, i);
    load_scales(0);
    auto stage = [&](int s, auto more_of) __attribute__((always_inline)) {
        constexpr bool more = decltype(more_of)::value;
        const int buf = s & 1;
        put_scales(buf);                          // (the other buffer's are still read)
        __builtin_amdgcn_s_waitcnt(0x0070);      // stage s has landed, and this wave's scales
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (more) load_scales(s + 1);
        const uint8_t* const d = tlds + buf * STAGE;
        // unit u: block u / TT of the stage, token tile u % TT.  Its product is started before the one before it is scaled and added, its
        // operands are read one unit earlier.
        constexpr int UNITS = 4 * TT;
        v4i a[2], bv[2];
        v16i c[2];
        v16f sp2[2];                              // the scales' products
        // Block b's scale alone, as k = b of an f16 operand: of this lane's row, or of its token.
        uint2 ws4, xs4[TT];
        auto one_scale = [&](uint2 v, int b) __attribute__((always_inline)) {
            const uint32_t e = (b & 2 ? v.y : v.x) & (b & 1 ? hi16 : lo16);
            return __builtin_bit_cast(hv8, b & 2 ? make_uint4(0, e, 0, 0) : make_uint4(e, 0, 0, 0));
        };
        auto read = [&](int u) __attribute__((always_inline)) {
            const int b = u / TT, tt = u % TT, piece = ((2 * b + half) ^ turn) << 4;
            if (tt == 0) a[b & 1] = *(const v4i*)(d + (wave * 32 + c32) * WIDE_K + piece);
            bv[u & 1] = *(const v4i*)(d + X_AT + (tt * 32 + c32) * WIDE_K + piece);
        };
        auto start = [&](int u) __attribute__((always_inline)) {
            v16i z;
#pragma unroll
            for (int i = 0; i < 16; i++) z[i] = 0;
            c[u & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[(u / TT) & 1], bv[u & 1], z, 0, 0, 0);
            v16f zf;
#pragma unroll
            for (int i = 0; i < 16; i++) zf[i] = 0.0f;
            sp2[u & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(one_scale(ws4, u / TT), one_scale(xs4[u % TT], u / TT), zf, 0, 0, 0);
        };
        ws4 = *(const uint2*)(d + WS_AT + 8 * (wave * 32 + c32));
#pragma unroll
        for (int tt = 0; tt < TT; tt++) xs4[tt] = *(const uint2*)(d + XS_AT + 8 * (tt * 32 + c32));
        read(0);
        start(0);
        read(1);
#pragma unroll
        for (int u = 0; u < UNITS; u++) {
            __builtin_amdgcn_sched_barrier(0);
            if (u + 1 < UNITS) start(u + 1);
            if (u + 2 < UNITS) read(u + 2);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int tt = u % TT;
                if (FMA) acc[tt][i] = fmaf((float)c[u & 1][i], sp2[u & 1][i], acc[tt][i]);
                else acc[tt][i] += (float)c[u & 1][i] * sp2[u & 1][i];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 16; i++) asm volatile("" : "+v"(acc[u % TT][i]));      // (done here: kept for later they fill the registers)
            constexpr int PER = (4 + TT + UNITS - 1) / UNITS;
            if (more) {
#pragma unroll
                for (int k = 0; k < PER; k++)
                    if (u * PER + k < 4 + TT) ask(s + 1, buf ^ 1, u * PER + k);
            }
        }
    };
    for (int s = 0; s + 1 < n_stage; s++) stage(s, std::true_type{});
    stage(n_stage - 1, std::false_type{});
    // through LDS, so that a token's 128 outputs are stored side by side
    constexpr int OSTR = WIDE_ROWS + 4;
    static_assert(32 * TT * OSTR * 4 <= 2 * STAGE);
    float* const o_lds = (float*)tlds;
    __syncthreads();
#pragma unroll
    for (int tt = 0; tt < TT; tt++)
#pragma unroll
        for (int i4 = 0; i4 < 4; i4++) {
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = out_scale != 1.0f ? acc[tt][4 * i4 + i] * out_scale : acc[tt][4 * i4 + i];
            *(float4*)(o_lds + (tt * 32 + c32) * OSTR + wave * 32 + 8 * i4 + 4 * half) = make_float4(v[0], v[1], v[2], v[3]);
        }
    __syncthreads();
    const int j = row0 + 4 * (tid & 31);
    for (int tt = tid >> 5; tt < 32 * TT && tok0 + tt < n_tok; tt += 8) {
        const float4 v = *(const float4*)(o_lds + tt * OSTR + 4 * (tid & 31));
        float* const o = out + (int64_t)(tok0 + tt) * n_out + j;
        if (j + 3 < n_out && !(n_out & 3)) {
            *(float4*)o = v;
        } else {
            const float f[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (j + i < n_out) o[i] = f[i];
        }
    }
}

}  // namespace

bool q8_gemm(const WView& w, const float* act_scales, const int8_t* act_quants, int n_tok, float* out, float out_scale,
             hipStream_t s, bool fma) {
    if (w.fmt != W_Q8_0 || n_tok < 16 || w.n_in % 32 || w.n_in <= 0 || w.n_out <= 0) return false;
    if ((reinterpret_cast<uintptr_t>(w.q) & 15) || (reinterpret_cast<uintptr_t>(act_quants) & 15)) return false;
    const int tiles = (n_tok + 15) / 16;
    const int gx = (w.n_out + 63) / 64;
    const int8_t* wq = (const int8_t*)w.q;
    const uint16_t* ws = (const uint16_t*)w.scales;
#define IT_GEMM(NT)                                                                                                  \
    do {                                                                                                             \
        if (fma) hipLaunchKernelGGL((q8_gemm_k<NT, true>), dim3(gx, (tiles + NT - 1) / NT), dim3(GT), 0, s, wq, ws, act_quants, act_scales, \
                                    out, w.n_in, w.n_out, n_tok, out_scale);                                        \
        else hipLaunchKernelGGL((q8_gemm_k<NT, false>), dim3(gx, (tiles + NT - 1) / NT), dim3(GT), 0, s, wq, ws, act_quants, act_scales, \
                                out, w.n_in, w.n_out, n_tok, out_scale);                                            \
    } while (0)
    const bool slabs = w.n_in % 256 == 0 && !((reinterpret_cast<uintptr_t>(ws) | reinterpret_cast<uintptr_t>(act_scales) | reinterpret_cast<uintptr_t>(out)) & 15);
    if (slabs) {
        auto launch = [&](auto kernel, int rows, int toks, size_t lds) {
            if (!lds_allowed<decltype(kernel)::value>(lds)) return false;
            hipLaunchKernelGGL(decltype(kernel)::value, dim3((w.n_out + rows - 1) / rows, (n_tok + toks - 1) / toks), dim3(256), lds, s, wq, ws, act_quants, act_scales,
                               out, w.n_in, w.n_out, n_tok, out_scale);
            return true;
        };
        auto tile = [&](auto nt) {
            constexpr int NT = decltype(nt)::value;
            constexpr size_t lds = 2 * tile_stage_bytes<NT>();
            return fma ? launch(KernelIs<&q8_tile_k<NT, true>>{}, 64, 16 * NT, lds) : launch(KernelIs<&q8_tile_k<NT, false>>{}, 64, 16 * NT, lds);
        };
        auto wide = [&](auto tt) {
            constexpr int TT = decltype(tt)::value;
            constexpr size_t lds = 2 * wide_stage_bytes<TT>();
            return fma ? launch(KernelIs<&q8_wide_k<TT, true>>{}, WIDE_ROWS, 32 * TT, lds) : launch(KernelIs<&q8_wide_k<TT, false>>{}, WIDE_ROWS, 32 * TT, lds);
        };
        using std::integral_constant;
        // 64 rows x 16 tokens a block up to 640 of them (2.5 a CU).  Above, the shape that takes least by the blocks a CU gets, b, from
        // what rows of 2,048 measure (in us; a block alone on its CU is quicker): 64 x 32 2.5 + 6.2 b; 128 x 32, three a CU at a time,
        // 19, 24 and 31; 128 x 64 25 and 37 for two; 128 x 128 38 and 66: what they took with the scales' products on the vector ALU, 4 to 9 %
        // more than now.  (4096 x 2048 over 300 / 400 / 512 / 1,100 / 1,500 / 5,700 tokens, now: 64 x 32 21.6, 27.8, 29.3, 54.1, 70.0, 239; 128 x 32
        // 20.8, 21.9, 23.0, 46.3, 53.5, 200; 128 x 64 24.1, 25.2, 26.0, 43.1, 46.0, 162; 128 x 128 35.9, 36.7, 37.3, 51.4, 55.1, 161.  The third
        // 128 x 64 block of a CU costs less than the sum says: at 1,100 and 1,500 tokens the shape taken, 128 x 32, is the second best.)
        // It served other row lengths as it is: 1,024 to 8,192 rows of 512 to 8,192 over 100 to 2,500 tokens, 90 shapes, none more than 3 %
        // behind 16, 32 or 64 tokens a block by their number alone.
        const int64_t units = (int64_t)gx * tiles;
        if (units <= 640) {
            if (tile(integral_constant<int, 1>{})) return true;
        } else {
            const int64_t gw = (w.n_out + WIDE_ROWS - 1) / WIDE_ROWS;
            auto per_cu = [&](int64_t rows, int toks) { return (rows * ((n_tok + toks - 1) / toks) + 255) / 256; };
            const int64_t b1 = per_cu(gw, 32), b2 = per_cu(gw, 64), b4 = per_cu(gw, 128);
            const int64_t cost[4] = {25 + 62 * per_cu(gx, 32), 306 * (b1 / 3) + (b1 % 3 == 2 ? 240 : b1 % 3 * 190), 369 * (b2 / 2) + b2 % 2 * 250,
                                     656 * (b4 / 2) + b4 % 2 * 380};
            const int64_t* const best = std::min_element(cost, cost + 4);
            if (best == cost ? tile(integral_constant<int, 2>{}) : best == cost + 1 ? wide(integral_constant<int, 1>{})
                             : best == cost + 2 ? wide(integral_constant<int, 2>{}) : wide(integral_constant<int, 4>{}))
                return true;
        }
    }
    // 64 tokens per block at most: four blocks fit a CU (38 KB of LDS, 98 VGPRs) and hide each other's LDS and
    // barrier waits; 128 tokens per block (two blocks per CU) measured 20 % slower despite reading the weights half as often
    // ... unless that leaves fewer than two blocks per CU (a short batch, few rows): then narrower blocks, which re-read
    // the weights (from the cache) but fill the chip (the dense matmuls of an 8-layer model over a 96-token prompt:
    // 1.57 against 2.16 ms); the arithmetic per output is the same for every width
    int nt = tiles >= 4 ? 4 : tiles >= 2 ? 2 : 1;
    while (nt > 1 && (int64_t)gx * ((tiles + nt - 1) / nt) < 512) nt >>= 1;
    if (nt == 4) IT_GEMM(4);
    else if (nt == 2) IT_GEMM(2);
    else IT_GEMM(1);
#undef IT_GEMM
    return true;
}

}  // namespace itk

// =====================================================================================
// Grouped expert matmuls for a batch of (token, pick) pairs.
//
// The per-pair GEMV reads an expert's matrix once per pair.  Here the pairs are first sorted
// into per-expert lists ("expert-sorted token lists": moe_group_k), the lists are cut into
// tiles of up to 16 pairs, and one block multiplies 64 rows of that expert's matrix with the
// tile's 16 activation rows on the matrix cores (Q8_0 int8, NVFP4 f16), so a matrix is read
// once per tile.  Per pair and row the arithmetic is the GEMV's: per-block integer dots, scaled
// and added in block order (Q8_0: (float)isum * (dw * dx); NVFP4: (dy * dA) * (float)sa then
// (dy * dB) * (float)sb per 32-element chunk of two sub-blocks), then the expert's second scale,
// then silu-mul for the gate/up pair.
namespace itk {
namespace {

// One block.  work layout: [0] = number of tiles; tiles as int4 {expert, first slot, pairs, 0};
// order[slot] = pair index.  The order of pairs inside an expert's list depends on the atomics'
// arrival order; it only decides which lane computes which pair, never a value.
// tile_pairs: most pairs of one tile (16 for the int8 kernels, 128 for the f16 kernel).
__global__ __launch_bounds__(1024) void moe_group_k(const int32_t* __restrict__ ids, int n_picks, int n_expert,
                                                    int tile_pairs, int32_t* __restrict__ n_tiles,
                                                    int4* __restrict__ tiles, int32_t* __restrict__ order) {
    __shared__ int cnt[1024], off[1024], toff[1024], cur[1024];
    const int tid = threadIdx.x;
    cnt[tid] = 0;
    __syncthreads();
    // eight picks' ids in flight per thread: the walk is bound by the latency of these loads
    for (int p0 = tid; p0 < n_picks; p0 += 8 * 1024) {
        int e[8];
#pragma unroll
        for (int u = 0; u < 8; u++) e[u] = p0 + u * 1024 < n_picks ? ids[p0 + u * 1024] : -1;
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (e[u] >= 0) atomicAdd(&cnt[e[u]], 1);
    }
    __syncthreads();
    // exclusive prefix sums of the pair counts and of the tile counts, all 1024 slots at once
    const int mine = tid < n_expert ? cnt[tid] : 0;
    const int my_tiles = (mine + tile_pairs - 1) / tile_pairs;
    off[tid] = mine;
    toff[tid] = my_tiles;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1) {
        const int a = tid >= d ? off[tid - d] : 0, b = tid >= d ? toff[tid - d] : 0;
        __syncthreads();
        off[tid] += a;
        toff[tid] += b;
        __syncthreads();
    }
    if (tid == 1023) *n_tiles = toff[1023];
    const int my_off = off[tid] - mine, my_toff = toff[tid] - my_tiles;
    cur[tid] = my_off;
    __syncthreads();
    for (int p0 = tid; p0 < n_picks; p0 += 8 * 1024) {
        int e[8];
#pragma unroll
        for (int u = 0; u < 8; u++) e[u] = p0 + u * 1024 < n_picks ? ids[p0 + u * 1024] : -1;
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (e[u] >= 0) order[atomicAdd(&cur[e[u]], 1)] = p0 + u * 1024;
    }
    for (int k = 0; k < my_tiles; k++)
        tiles[my_toff + k] = make_int4(tid, my_off + tile_pairs * k, min(tile_pairs, mine - tile_pairs * k), 0);
}

struct ExpertsGemmP {
    const uint8_t *q, *s, *q2, *s2;
    const uint8_t* const *q_tab, *const *s_tab, *const *q2_tab, *const *s2_tab;  // expert placement tables or null
    int64_t q_stride, s_stride;
    const float *scale2, *scale2_up;
    const float* act_scales;
    const int8_t* act_quants;
    float* out;
    int n_in, n_out, x_mode, n_used;
    const int32_t* n_tiles;
    const int4* tiles;
    const int32_t* order;
};

// the block's results: pair m's rows j0 .. j0 + 3
template <bool GLU>
IT_DEV void put_pairs(const ExpertsGemmP& p, int64_t e, int cnt, const int* pair_s, int j0, int m, const float (&acc)[GLU ? 2 : 1][4]) {
    if (m >= cnt) return;
    const int64_t pair = pair_s[m];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int j = j0 + i;
        if (j >= p.n_out) continue;
        float a0 = acc[0][i];
        if (p.scale2) a0 *= p.scale2[e];
        if (GLU) {
            float a1 = acc[GLU ? 1 : 0][i];
            if (p.scale2_up) a1 *= p.scale2_up[e];
            a0 = it_silu(a0) * a1;
        }
        p.out[pair * p.n_out + j] = a0;
    }
}

template <bool GLU>
__global__ __launch_bounds__(GT) void experts_gemm_k(ExpertsGemmP p) {
    constexpr int NM = GLU ? 2 : 1;
    __shared__ __align__(16) int8_t As[2][NM][64 * LSTR];
    __shared__ float Asc[2][NM][64 * 4];
    __shared__ __align__(16) int8_t Bs[2][16 * LSTR];
    __shared__ float Bsc[2][16 * 4];
    __shared__ int xrow_s[16], pair_s[16];
    const int tile = blockIdx.x;
    if (tile >= *p.n_tiles) return;
    const int4 td = p.tiles[tile];
    const int64_t e = td.x;
    const int cnt = td.z;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 15, g = lane >> 4;
    const int row0 = blockIdx.y * 64;
    const int n_in = p.n_in, nb = n_in >> 5;
    const int nslab = n_in / SLAB;
    if (tid < 16) {
        const int pair = p.order[td.y + min(tid, cnt - 1)];
        pair_s[tid] = pair;
        xrow_s[tid] = p.x_mode == 0 ? pair : (p.x_mode == 1 ? pair / p.n_used : 0);
    }
    __syncthreads();
    const uint8_t* wq[2] = {it_expert_at(p.q, p.q_tab, e, p.q_stride), GLU ? it_expert_at(p.q2, p.q2_tab, e, p.q_stride) : nullptr};
    const uint8_t* ws[2] = {it_expert_at(p.s, p.s_tab, e, p.s_stride), GLU ? it_expert_at(p.s2, p.s2_tab, e, p.s_stride) : nullptr};

    uint4 ra[NM][2], rb;
    float rsa[NM], rsb;
    rb = make_uint4(0, 0, 0, 0);
    rsb = 0.0f;
#pragma unroll
    for (int mt = 0; mt < NM; mt++)
#pragma unroll
        for (int q = 0; q < 2; q++) {
            ra[mt][q] = rb;
            rsa[mt] = 0.0f;
        }
    auto fetch = [&](int s) {
#pragma unroll
        for (int mt = 0; mt < NM; mt++) {
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const int idx = tid + q * GT, row = idx >> 3, seg = idx & 7;
                ra[mt][q] = *(const uint4*)(wq[mt] + (int64_t)min(row0 + row, p.n_out - 1) * n_in + s * SLAB + seg * 16);
            }
            const int row = tid >> 2, bi = tid & 3;
            rsa[mt] = it_f16_to_f32(((const uint16_t*)ws[mt])[(int64_t)min(row0 + row, p.n_out - 1) * nb + s * 4 + bi]);
        }
        if (tid < 128) {
            const int pr = tid >> 3, seg = tid & 7;
            rb = *(const uint4*)(p.act_quants + (int64_t)xrow_s[pr] * n_in + s * SLAB + seg * 16);
        }
        if (tid < 64) rsb = p.act_scales[(int64_t)xrow_s[tid >> 2] * nb + s * 4 + (tid & 3)];
    };
    auto stash = [&](int buf) {
#pragma unroll
        for (int mt = 0; mt < NM; mt++) {
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const int idx = tid + q * GT, row = idx >> 3, seg = idx & 7;
                *(uint4*)(As[buf][mt] + row * LSTR + seg * 16) = ra[mt][q];
            }
            Asc[buf][mt][tid] = rsa[mt];
        }
        if (tid < 128) *(uint4*)(Bs[buf] + (tid >> 3) * LSTR + (tid & 7) * 16) = rb;
        if (tid < 64) Bsc[buf][tid] = rsb;
    };

    float acc[NM][4];
#pragma unroll
    for (int mt = 0; mt < NM; mt++)
#pragma unroll
        for (int i = 0; i < 4; i++) acc[mt][i] = 0.0f;
    const v4i z = {0, 0, 0, 0};

    fetch(0);
    stash(0);
    __syncthreads();
    for (int s = 0; s < nslab; s++) {
        const int buf = s & 1;
        if (s + 1 < nslab) fetch(s + 1);
#pragma unroll
        for (int bi = 0; bi < 4; bi++) {
            const long bv = *(const long*)(Bs[buf] + m * LSTR + bi * 32 + g * 8);
            const float dx = Bsc[buf][m * 4 + bi];
#pragma unroll
            for (int mt = 0; mt < NM; mt++) {
                const long a = *(const long*)(As[buf][mt] + (wave * 16 + m) * LSTR + bi * 32 + g * 8);
                const v4i d = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, bv, z, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float dw = Asc[buf][mt][(wave * 16 + 4 * g + i) * 4 + bi];
                    acc[mt][i] += (float)d[i] * (dw * dx);
                }
            }
        }
        if (s + 1 < nslab) stash(buf ^ 1);
        __syncthreads();
    }
    put_pairs<GLU>(p, e, cnt, pair_s, row0 + wave * 16 + 4 * g, m, acc);
}

// NVFP4, the CPU path's bits: a sub-block's dot is a sum of whole numbers, and the f16 matrix instruction forms it exactly (doubled
// e2m1 by quants: 16 products below 1,524, in f32); so is the product of the activation's f16 step and the weight's e4m3 scale, a
// second instruction of which one term is not 0.  Left to the vector ALU are gfx950's own conversion of the nibbles, the product of the
// two results and its addition, sub-blocks in order.  On the int8 instructions that were also the nibbles' expansion, the halves'
// selection, the dots' conversion and the scales' product, 2.7 times the instructions, which bounded it: 333 tokens, ten of 512 experts
// of 512 x 2,048: gate and up 356 -> 194 us; a request of 333 tokens and eight more on two layers 3.50 -> 3.08 ms.
// A lane takes bytes 2 g and 2 g + 1 of each sub-block (k order: low and high nibble of the one, of the other), so a row of a slab lies in
// LDS as four groups of eight sub-blocks' two bytes, 16 bytes a lane and slab; the quants, as f16, in the same order.
constexpr int NROW = 64 + 16, NCOL = 256 + 16;   // LDS bytes of a row's nibbles, of a pair's quants: sixteen rows at once hit different banks
template <bool GLU>
__global__ __launch_bounds__(GT, 4) void experts_nvfp4_k(ExpertsGemmP p) {
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    typedef float v4f __attribute__((ext_vector_type(4)));
    constexpr int NM = GLU ? 2 : 1;
    __shared__ __align__(16) uint8_t As[2][NM][64 * NROW];
    __shared__ __align__(16) uint32_t Asc[2][NM][64 * 4];   // eight f16 a row
    __shared__ __align__(16) uint8_t Bs[2][16 * NCOL];
    __shared__ __align__(16) uint32_t Bsc[2][16 * 4];       // an f16 each
    __shared__ int xrow_s[16], pair_s[16];
    const int tile = blockIdx.x;
    if (tile >= *p.n_tiles) return;
    const int4 td = p.tiles[tile];
    const int64_t e = td.x;
    const int cnt = td.z;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 15, g = lane >> 4;
    const int row0 = blockIdx.y * 64;
    const int n_in = p.n_in, nb = n_in >> 5;
    const int nslab = n_in / SLAB;
    if (tid < 16) {
        const int pair = p.order[td.y + min(tid, cnt - 1)];
        pair_s[tid] = pair;
        xrow_s[tid] = p.x_mode == 0 ? pair : (p.x_mode == 1 ? pair / p.n_used : 0);
    }
    __syncthreads();
    const int row = tid >> 2, seg = tid & 3, pr = tid >> 3, sub = tid & 7;   // what a thread brings: of a row two sub-blocks, of a pair one
    const int64_t wrow = min(row0 + row, p.n_out - 1);
    const uint8_t *wq[NM], *ws[NM];
    wq[0] = it_expert_at(p.q, p.q_tab, e, p.q_stride) + wrow * (n_in >> 1) + seg * 16;
    ws[0] = it_expert_at(p.s, p.s_tab, e, p.s_stride) + wrow * (n_in >> 4) + seg * 2;
    if (GLU) {
        wq[NM - 1] = it_expert_at(p.q2, p.q2_tab, e, p.q_stride) + wrow * (n_in >> 1) + seg * 16;
        ws[NM - 1] = it_expert_at(p.s2, p.s2_tab, e, p.s_stride) + wrow * (n_in >> 4) + seg * 2;
    }
    const int8_t* const xq = p.act_quants + (int64_t)xrow_s[pr & 15] * n_in + sub * 16;
    const float* const xs = p.act_scales + (int64_t)xrow_s[row & 15] * nb + seg;

    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    u4 ra[NM] = {}, rb = {};
    uint32_t rsa[NM] = {};
    float rsb = 0.0f;
    auto fetch = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < NM; mt++) {
            ra[mt] = *(const u4*)(wq[mt] + s * 64);
            rsa[mt] = *(const uint16_t*)(ws[mt] + s * 8);
        }
        if (tid < 128) rb = *(const u4*)(xq + s * SLAB);
        if (tid < 64) rsb = xs[s * 4];
    };
    auto stash = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < NM; mt++) {
            // sub-blocks 2 seg (words 0, 1) and 2 seg + 1 (words 2, 3): group q's bytes 2 q, 2 q + 1 of each
#pragma unroll
            for (int q = 0; q < 4; q++)
                *(uint32_t*)(As[buf][mt] + row * NROW + q * 16 + seg * 4) =
                    __builtin_amdgcn_perm(ra[mt][2 + q / 2], ra[mt][q / 2], q & 1 ? 0x07060302u : 0x05040100u);
            const _Float16 s0 = (_Float16)it_ue4m3_to_f32(rsa[mt] & 0xffu), s1 = (_Float16)it_ue4m3_to_f32(rsa[mt] >> 8);
            Asc[buf][mt][row * 4 + seg] = __builtin_bit_cast(uint16_t, s0) | (uint32_t)__builtin_bit_cast(uint16_t, s1) << 16;
        }
        if (tid < 128) {
            auto quant = [&](int i) __attribute__((always_inline)) { return (_Float16)(float)(int8_t)(rb[i >> 2] >> (8 * (i & 3))); };
#pragma unroll
            for (int q = 0; q < 4; q++)
                *(h4*)(Bs[buf] + pr * NCOL + q * 64 + sub * 8) = h4{quant(2 * q), quant(2 * q + 8), quant(2 * q + 1), quant(2 * q + 9)};
        }
        if (tid < 64) Bsc[buf][tid] = __builtin_bit_cast(uint16_t, (_Float16)rsb);
    };

    float acc[NM][4];
#pragma unroll
    for (int mt = 0; mt < NM; mt++)
#pragma unroll
        for (int i = 0; i < 4; i++) acc[mt][i] = 0.0f;
    const v4f z = {0.0f, 0.0f, 0.0f, 0.0f};

    fetch(0);
    stash(0);
    __syncthreads();
    for (int s = 0; s < nslab; s++) {
        const int buf = s & 1;
        if (s + 1 < nslab) fetch(s + 1);
        // the pair's quants, and its step of chunk c in the k slot that holds the scale of the sub-block (slots 4 g ..: sub-blocks 4 g ..)
        h4 bq[8];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const u4 x = *(const u4*)(Bs[buf] + m * NCOL + g * 64 + c * 16);
            bq[2 * c] = __builtin_bit_cast(h4, (uint64_t)x[1] << 32 | x[0]);
            bq[2 * c + 1] = __builtin_bit_cast(h4, (uint64_t)x[3] << 32 | x[2]);
        }
        u4 dx = *(const u4*)(Bsc[buf] + m * 4);
#pragma unroll
        for (int c = 0; c < 4; c++) dx[c] = g == c >> 1 ? dx[c] : 0u;
#pragma unroll
        for (int mt = 0; mt < NM; mt++) {
            const u4 nib = *(const u4*)(As[buf][mt] + (wave * 16 + m) * NROW + g * 16);
            const h4 sc = *(const h4*)(Asc[buf][mt] + (wave * 16 + m) * 4 + 2 * (g & 1));   // (g of 2 and 3: their slots' steps are 0)
            v4f dot[2], by[2];                       // (a sub-block's two results are on their way while the last one's are added)
#pragma unroll
            for (int j = 0; j <= 8; j++) {
                if (j < 8) {
                    const h2 lo = j & 1 ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(nib[j / 2], 2.0f, 2) : __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(nib[j / 2], 2.0f, 0);
                    const h2 hi = j & 1 ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(nib[j / 2], 2.0f, 3) : __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(nib[j / 2], 2.0f, 1);
                    const uint64_t step = (uint64_t)dx[j / 2] << (16 * (j & 3));
                    dot[j & 1] = __builtin_amdgcn_mfma_f32_16x16x16f16(h4{lo[0], lo[1], hi[0], hi[1]}, bq[j], z, 0, 0, 0);
                    by[j & 1] = __builtin_amdgcn_mfma_f32_16x16x16f16(sc, __builtin_bit_cast(h4, step), z, 0, 0, 0);
                }
                if (j > 0) {
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[mt][i] += by[(j - 1) & 1][i] * dot[(j - 1) & 1][i];
                    // (here, not behind all products, whose results would fill the registers)
                    asm volatile("" : "+v"(acc[mt][0]), "+v"(acc[mt][1]), "+v"(acc[mt][2]), "+v"(acc[mt][3]));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (s + 1 < nslab) stash(buf ^ 1);
        __syncthreads();
    }
    put_pairs<GLU>(p, e, cnt, pair_s, row0 + wave * 16 + 4 * g, m, acc);
}

}  // namespace

size_t experts_group_work_ints(int n_picks, int n_expert) {
    // sized for the smallest tiles any kernel groups for (eight pairs)
    return 16 + (size_t)(n_expert + n_picks / 8 + 2) * 4 + (size_t)n_picks;
}

bool experts_gemm(const ExpertsView& w, const ExpertsView* up, const int32_t* ids, int n_picks, int n_used, int x_mode,
                  const float* act_scales, const int8_t* act_quants, float* out, int32_t* work, size_t work_ints,
                  bool grouped, hipStream_t s) {
    if (n_picks < 32 || !work || w.n_expert > 1024 || w.n_in % SLAB || (w.fmt != W_Q8_0 && w.fmt != W_NVFP4)) return false;
    if (work_ints < experts_group_work_ints(n_picks, w.n_expert)) return false;
    if ((reinterpret_cast<uintptr_t>(w.q) & 15) || w.q_stride % 16 || (reinterpret_cast<uintptr_t>(act_quants) & 15)) return false;
    if (up && (up->fmt != w.fmt || up->n_in != w.n_in || up->n_out != w.n_out || (reinterpret_cast<uintptr_t>(up->q) & 15)))
        return false;
    const int max_tiles = w.n_expert + n_picks / 16 + 1;
    int32_t* n_tiles = work;
    int4* tiles = (int4*)(work + 16);
    int32_t* order = work + 16 + (size_t)(max_tiles + 1) * 4;
    if (!grouped) hipLaunchKernelGGL(moe_group_k, dim3(1), dim3(1024), 0, s, ids, n_picks, w.n_expert, 16, n_tiles, tiles, order);
    ExpertsGemmP p{};
    p.q = (const uint8_t*)w.q;
    p.s = (const uint8_t*)w.scales;
    p.q2 = up ? (const uint8_t*)up->q : nullptr;
    p.s2 = up ? (const uint8_t*)up->scales : nullptr;
    p.q_stride = w.q_stride;
    p.s_stride = w.s_stride;
    p.q_tab = w.q_tab;
    p.s_tab = w.s_tab;
    p.q2_tab = up ? up->q_tab : nullptr;
    p.s2_tab = up ? up->s_tab : nullptr;
    p.scale2 = w.scale2;
    p.scale2_up = up ? up->scale2 : nullptr;
    p.act_scales = act_scales;
    p.act_quants = act_quants;
    p.out = out;
    p.n_in = w.n_in;
    p.n_out = w.n_out;
    p.x_mode = x_mode;
    p.n_used = n_used < 1 ? 1 : n_used;
    p.n_tiles = n_tiles;
    p.tiles = tiles;
    p.order = order;
    dim3 grid(max_tiles, (w.n_out + 63) / 64);
    if (w.fmt == W_Q8_0) {
        if (up) hipLaunchKernelGGL(experts_gemm_k<true>, grid, dim3(GT), 0, s, p);
        else hipLaunchKernelGGL(experts_gemm_k<false>, grid, dim3(GT), 0, s, p);
    } else {
        if (up) hipLaunchKernelGGL(experts_nvfp4_k<true>, grid, dim3(GT), 0, s, p);
        else hipLaunchKernelGGL(experts_nvfp4_k<false>, grid, dim3(GT), 0, s, p);
    }
    return true;
}


void moe_group(const int32_t* ids, int n_picks, int n_expert, int tile_pairs, int32_t* n_tiles, int4* tiles,
               int32_t* order, hipStream_t s) {
    hipLaunchKernelGGL(moe_group_k, dim3(1), dim3(1024), 0, s, ids, n_picks, n_expert, tile_pairs, n_tiles, tiles, order);
}

}  // namespace itk
