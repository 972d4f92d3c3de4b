// Dense Q8_0 products of a short batch on the int8 matrix cores (fast mode).
//
// The tiles of k_gemm.hip walk the k range slab by slab, a round trip through LDS each, for matrices whose bytes take 2 us and
// whose arithmetic takes one.  Here the k range is cut over the waves of a
// block and every wave asks at once for all it will read, 16 RT weight rows and up to 32 tokens of its 256 (or 512) k, straight
// into registers: one trip to memory.  The waves' sums meet in LDS behind one barrier.
// The products are those of k_gemm.hip (an exact int32 sum per 32 terms, scaled and added in f32 with one rounding); the f32
// sums of the waves are added at the end instead of one running over the whole row.
// Bound by that trip's latency; 2048 x 4096 over 23 tokens 32.0 -> 16.6 us, 4096 x 2048 19.2 -> 10.6, 512 x 2048 18.4 -> 10.2
// (cold caches, between two events, whose own 5 us are in both).  Not kept: further tokens in a loop over the same weights
// (5 us for every 32 of them, each load instruction of the tokens touching sixteen lines for 32 bytes each).
//
// MFMA 16x16x32 i8: lane l supplies 8 consecutive k of row l % 16 at k = 8 (l / 16) for A (weights) and B (tokens) and
// receives weight rows 4 (l / 16) + {0..3} of token l % 16.
#include <algorithm>

#include "it_device.h"
#include "kernels.h"

namespace itk {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));

template <int KW, int U, int RT>
__global__ __launch_bounds__(64 * KW) void q8_short_k(const int8_t* __restrict__ wq, const uint16_t* __restrict__ ws,
                                                      const int8_t* __restrict__ xq, const float* __restrict__ xs,
                                                      float* __restrict__ out, int n_out, int n_tok, float out_scale) {
    constexpr int n_in = 256 * KW * U, nb = n_in / 32;
    __shared__ float4 red[KW][2 * RT][64];     // [wave][token tile, row tile][lane]
    const int lane = threadIdx.x & 63;
    const int kw = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int row0 = blockIdx.x * 16 * RT;

    // everything this wave reads, asked for at once: its part of the weight rows, of the tokens, and their scales (the
    // weights' for the four rows that a lane receives)
    long a[U][RT][8], x[U][2][8];
    uint4 dw[U][RT][4];
    float4 dx[U][2][2];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int k = (u * KW + kw) * 256;
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            const int8_t* p = wq + (int64_t)min(row0 + rt * 16 + r, n_out - 1) * n_in + k + g * 8;
#pragma unroll
            for (int b = 0; b < 8; b++) a[u][rt][b] = *(const long*)(p + b * 32);
#pragma unroll
            for (int i = 0; i < 4; i++) dw[u][rt][i] = *(const uint4*)(ws + (int64_t)min(row0 + rt * 16 + 4 * g + i, n_out - 1) * nb + k / 32);
        }
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int64_t tok = min(16 * t + r, n_tok - 1);
            const int8_t* p = xq + tok * n_in + k + g * 8;
#pragma unroll
            for (int b = 0; b < 8; b++) x[u][t][b] = *(const long*)(p + b * 32);
            const float4* d = (const float4*)(xs + tok * nb + k / 32);
            dx[u][t][0] = d[0];
            dx[u][t][1] = d[1];
        }
    }
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int u = 0; u < U; u++) {
                const float d8[8] = {dx[u][t][0].x, dx[u][t][0].y, dx[u][t][0].z, dx[u][t][0].w, dx[u][t][1].x, dx[u][t][1].y, dx[u][t][1].z, dx[u][t][1].w};
#pragma unroll
                for (int b = 0; b < 8; b++) {
                    const v4i z = {0, 0, 0, 0};
                    const v4i d = __builtin_amdgcn_mfma_i32_16x16x32_i8(a[u][rt][b], x[u][t][b], z, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float w = (float)__builtin_bit_cast(h8, dw[u][rt][i])[b];
                        acc[i] = fmaf((float)d[i], w * d8[b], acc[i]);
                    }
                }
            }
            red[kw][t * RT + rt][lane] = make_float4(acc[0], acc[1], acc[2], acc[3]);
        }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 2 * RT; c++) {
        if (c % KW != kw) continue;
        float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
        for (int k = 0; k < KW; k++) {
            const float4 v = red[k][c][lane];
            s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
        }
        const int tok = 16 * (c / RT) + r, row = row0 + 16 * (c % RT) + 4 * g;
        if (tok >= n_tok) continue;
        s.x *= out_scale; s.y *= out_scale; s.z *= out_scale; s.w *= out_scale;
        float* o = out + (int64_t)tok * n_out + row;
        if (row + 3 < n_out && n_out % 4 == 0) {
            *(float4*)o = s;
        } else {
            if (row < n_out) o[0] = s.x;
            if (row + 1 < n_out) o[1] = s.y;
            if (row + 2 < n_out) o[2] = s.z;
            if (row + 3 < n_out) o[3] = s.w;
        }
    }
}

}  // namespace

bool q8_short(const WView& w, const float* act_scales, const int8_t* act_quants, int n_tok, float* out, float out_scale, hipStream_t s) {
    const int kw = w.n_in / 256;
    if (w.fmt != W_Q8_0 || n_tok < 2 || w.n_out < 1 || w.n_in % 256 || (kw != 1 && kw != 2 && kw != 4 && kw != 8 && kw != 16)) return false;
    auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    if (!al16(w.q) || !al16(w.scales) || !al16(act_quants) || !al16(act_scales) || !al16(out)) return false;
    // Up to 32 tokens and a block of 32 rows per CU; half as many leave room for blocks of 16 rows.  (The tiles of k_gemm.hip
    // are 1 to 2 us behind at 16 tokens, level at 32 and ahead above.)
    if (n_tok > 32 || w.n_out > 8192) return false;
    const int rt = w.n_out > 4096 ? 2 : 1;
    // below 16 tokens against one GEMV each: from 16,384 results on (4096 rows: 9.1 against 9.7 us for 3 tokens, 9.0 against 12.6
    // for 5; 512 rows: behind, 9.0 against 7.1 for 12)
    if (n_tok < 16 && (int64_t)n_tok * w.n_out < 16384) return false;
    const dim3 grid((w.n_out + 16 * rt - 1) / (16 * rt)), block(64 * std::min(kw, 8));
#define IT_QS(KW, U)                                                                                                                  \
    do {                                                                                                                              \
        if (rt == 2) hipLaunchKernelGGL((q8_short_k<KW, U, 2>), grid, block, 0, s, (const int8_t*)w.q, (const uint16_t*)w.scales,     \
                                        act_quants, act_scales, out, w.n_out, n_tok, out_scale);                                      \
        else hipLaunchKernelGGL((q8_short_k<KW, U, 1>), grid, block, 0, s, (const int8_t*)w.q, (const uint16_t*)w.scales, act_quants, \
                                act_scales, out, w.n_out, n_tok, out_scale);                                                          \
    } while (0)
    switch (kw) {
        case 1: IT_QS(1, 1); break;
        case 2: IT_QS(2, 1); break;
        case 4: IT_QS(4, 1); break;
        case 8: IT_QS(8, 1); break;
        default: IT_QS(8, 2); break;
    }
#undef IT_QS
    return true;
}

}  // namespace itk
