// Unquantized (F32 / F16 / BF16) weights: what a real file keeps its router, shared-expert gate and ssm alpha / beta in.
//
// Exact mode: the CPU path's serial f32 fold over the row (/root/reference src/ops/naive.rs:843-861).  Fast mode: the
// same products summed by the f32 matrix instruction, whose inputs, products and sums are f32 as well.
#include <cstdint>

#include "it_device.h"
#include "kernels.h"
#include "it_dot.h"

namespace itk {
namespace {

template <int FMT>
IT_DEV float4 load_w4(const uint8_t* row, int i) {
    if (FMT == W_F32) return *(const float4*)((const float*)row + i);
    const uint2 h = *(const uint2*)((const uint16_t*)row + i);
    if (FMT == W_F16)
        return make_float4(it_f16_to_f32(h.x & 0xffffu), it_f16_to_f32(h.x >> 16), it_f16_to_f32(h.y & 0xffffu), it_f16_to_f32(h.y >> 16));
    return make_float4(it_bf16_to_f32(h.x & 0xffffu), it_bf16_to_f32(h.x >> 16), it_bf16_to_f32(h.y & 0xffffu), it_bf16_to_f32(h.y >> 16));
}
template <int FMT>
IT_DEV float load_w1(const uint8_t* row, int i) {
    if (FMT == W_F32) return ((const float*)row)[i];
    const uint16_t h = ((const uint16_t*)row)[i];
    return FMT == W_F16 ? it_f16_to_f32(h) : it_bf16_to_f32(h);
}
// row j of the two matrices of a launch; rows past the end repeat the last one (their results are not stored)
template <int FMT>
IT_DEV const uint8_t* float_row(const FloatMats& m, int j, int n_in) {
    constexpr int ESZ = FMT == W_F32 ? 4 : 2;
    const int last = m.n0 + m.n1 - 1;
    j = j < last ? j : last;
    return j < m.n0 ? m.w0 + (int64_t)j * n_in * ESZ : m.w1 + (int64_t)(j - m.n0) * n_in * ESZ;
}
IT_DEV void float_store(const FloatMats& m, int t, int j, float v) {
    if (j < m.n0) m.out0[(int64_t)t * m.n0 + j] = v;
    else if (j < m.n0 + m.n1) m.out1[(int64_t)t * m.n1 + (j - m.n0)] = v;
}

// ------------------------------------------------------------------ exact mode, a few tokens
// A block: EX_ROWS rows of one token.  All its threads form products, coalesced, into LDS; a lane per row then folds them
// in order.  Bound by the serial chain: n_in dependent additions (2,048: 6 us), where one thread per output, which also
// waited for its own uncoalesced loads, took 127 to 190 us.
constexpr int EX_ROWS = 8, EX_K = 2048;
template <int FMT>
__global__ __launch_bounds__(256) void float_fold_exact_k(FloatMats m, const float* __restrict__ x, int n_in, float out_scale) {
    __shared__ __align__(16) float prod[EX_ROWS][EX_K + 4];   // + 4: the rows' 16-byte reads fall on different banks
    const int row0 = blockIdx.x * EX_ROWS, t = blockIdx.y, tid = threadIdx.x;
    const float* xt = x + (int64_t)t * n_in;
    const uint8_t* rows[EX_ROWS];
#pragma unroll
    for (int r = 0; r < EX_ROWS; r++) rows[r] = float_row<FMT>(m, row0 + r, n_in);
    float sum = 0.0f;
    for (int k0 = 0; k0 < n_in; k0 += EX_K) {
        const int kn = min(EX_K, n_in - k0);
        if (k0) __syncthreads();
        // (the activation once, every row's loads of a step together)
#pragma unroll 2
        for (int i = tid; i < kn; i += 256) {
            const float xv = xt[k0 + i];
            float wv[EX_ROWS];
#pragma unroll
            for (int r = 0; r < EX_ROWS; r++) wv[r] = load_w1<FMT>(rows[r], k0 + i);
#pragma unroll
            for (int r = 0; r < EX_ROWS; r++) prod[r][i] = wv[r] * xv;
        }
        __syncthreads();
        if (tid < EX_ROWS) {
            sum = fold_terms_from(sum, prod[tid], kn);
        }
    }
    if (tid < EX_ROWS) float_store(m, t, row0 + tid, out_scale != 1.0f ? sum * out_scale : sum);
}

// ------------------------------------------------------------------ exact mode, a batch
// TILE rows x TILE tokens per block, an R x R tile of sums per thread; k in slabs of 32 through LDS, the next slab's loads
// in flight meanwhile.  Product and addition are rounded apart (-ffp-contract=off) and k ascends, so every sum is the serial
// fold's.  A slab that reaches past the row is padded with zero products, which change no bit (the sum, which starts at
// +0, is never -0).  Bound by the vector ALU; R = 2 while R = 4 would leave the chip short of blocks.
template <int FMT, int R>
__global__ __launch_bounds__(256) void float_tile_exact_k(FloatMats m, const float* __restrict__ x, int n_in, int n_tok, float out_scale) {
    constexpr int KS = 32, TILE = 16 * R, NL = TILE / 32;   // NL float4 loads of each operand per thread and slab
    __shared__ __align__(16) float Ws[KS][TILE + 4], Xs[KS][TILE + 4];
    const int tid = threadIdx.x, tr = tid & 15, tc = tid >> 4;
    const int row0 = blockIdx.x * TILE, tok0 = blockIdx.y * TILE;
    const int lr = tid >> 3, lk = (tid & 7) * 4;            // staging: rows (tokens) lr, lr + 32; k lk .. + 3
    const uint8_t* wp[NL];
    const float* xp[NL];
#pragma unroll
    for (int h = 0; h < NL; h++) {
        wp[h] = float_row<FMT>(m, row0 + lr + 32 * h, n_in);
        xp[h] = x + (int64_t)min(tok0 + lr + 32 * h, n_tok - 1) * n_in;
    }
    float acc[R][R];
#pragma unroll
    for (int a = 0; a < R; a++)
#pragma unroll
        for (int b = 0; b < R; b++) acc[a][b] = 0.0f;
    float4 wv[NL], xv[NL];
    auto load = [&](int k) {
#pragma unroll
        for (int h = 0; h < NL; h++) {
            const bool in = k + lk < n_in;                  // n_in is a multiple of 4
            wv[h] = in ? load_w4<FMT>(wp[h], k + lk) : make_float4(0.f, 0.f, 0.f, 0.f);
            xv[h] = in ? *(const float4*)(xp[h] + k + lk) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    load(0);
    for (int k0 = 0; k0 < n_in; k0 += KS) {
        __syncthreads();
#pragma unroll
        for (int h = 0; h < NL; h++) {
            const int c = lr + 32 * h;
            Ws[lk][c] = wv[h].x; Ws[lk + 1][c] = wv[h].y; Ws[lk + 2][c] = wv[h].z; Ws[lk + 3][c] = wv[h].w;
            Xs[lk][c] = xv[h].x; Xs[lk + 1][c] = xv[h].y; Xs[lk + 2][c] = xv[h].z; Xs[lk + 3][c] = xv[h].w;
        }
        __syncthreads();
        if (k0 + KS < n_in) load(k0 + KS);
#pragma unroll
        for (int k = 0; k < KS; k++) {
            float av[R], bv[R];
#pragma unroll
            for (int e = 0; e < R; e++) {
                av[e] = Ws[k][R * tr + e];
                bv[e] = Xs[k][R * tc + e];
            }
#pragma unroll
            for (int ia = 0; ia < R; ia++)
#pragma unroll
                for (int ib = 0; ib < R; ib++) acc[ia][ib] += av[ia] * bv[ib];
        }
    }
#pragma unroll
    for (int ib = 0; ib < R; ib++) {
        const int t = tok0 + R * tc + ib;
        if (t >= n_tok) continue;
#pragma unroll
        for (int ia = 0; ia < R; ia++) float_store(m, t, row0 + R * tr + ia, out_scale != 1.0f ? acc[ia][ib] * out_scale : acc[ia][ib]);
    }
}

// rows of any length at any alignment: one thread per output
template <int FMT>
__global__ void float_any_k(FloatMats m, const float* __restrict__ x, int n_in, int n_tok, float out_scale) {
    const int rows = m.n0 + m.n1;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)rows * n_tok) return;
    const int j = (int)(idx % rows), t = (int)(idx / rows);
    const float* xt = x + (int64_t)t * n_in;
    const uint8_t* row = float_row<FMT>(m, j, n_in);
    float sum = 0.0f;
    for (int i = 0; i < n_in; i++) sum += load_w1<FMT>(row, i) * xt[i];
    float_store(m, t, j, out_scale != 1.0f ? sum * out_scale : sum);
}

// ------------------------------------------------------------------ fast mode, one token: a wave per row
template <int FMT>
__global__ __launch_bounds__(256) void float_gemv_fast_k(FloatMats m, const float* __restrict__ x, int n_in, float out_scale) {
    const int lane = threadIdx.x & 63;
    const int j = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (j >= m.n0 + m.n1) return;
    const uint8_t* row = float_row<FMT>(m, j, n_in);
    float v = 0.0f;
    for (int i = lane * 4; i < n_in; i += 256) {
        const float4 wv = load_w4<FMT>(row, i);
        const float4 xv = *(const float4*)(x + i);
        v = fmaf(wv.x, xv.x, fmaf(wv.y, xv.y, fmaf(wv.z, xv.z, fmaf(wv.w, xv.w, v))));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if (lane == 0) float_store(m, 0, j, out_scale != 1.0f ? v * out_scale : v);
}

// ------------------------------------------------------------------ fast mode, several tokens: f32 matrix instructions
// A block is KW waves on one tile of 16 RT rows x 16 TT tokens, each with its share of k; the shares are added through LDS
// in wave order.  Per 16 k a lane loads one float4 of its row and one of its token for each 16-wide tile and issues four
// v_mfma_f32_16x16x4_f32 per pair of tiles, instruction j taking element j of both (k = 4 (lane / 16) + j: the same k on
// both sides, in whatever order).  Operands come straight from L2: no LDS, no barrier in the loop.  513 x 2,048 F32 rows
// (router + gate logit): 9 us for 23 tokens (9 blocks of a 64 x 64 tile on the vector ALU: 100 us), 152 us for 5,700 (369).
// (Asking for two or four steps at a time, twice buffered, is 10 to 60 % slower: not the latency of a step bounds it but the
// rate at which loads of sixteen rows' 64 bytes are served.)
typedef float f32x4_t __attribute__((ext_vector_type(4)));
template <int FMT, int RT, int TT, int KW>
__global__ __launch_bounds__(64 * KW) void float_mfma_k(FloatMats m, const float* __restrict__ x, int n_in, int n_tok, float out_scale) {
    __shared__ f32x4_t part[KW][RT * TT][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row0 = blockIdx.x * 16 * RT, tok0 = blockIdx.y * 16 * TT;
    const int steps = n_in / 16;
    const int s0 = steps * wave / KW, s1 = steps * (wave + 1) / KW;
    const uint8_t* wp[RT];
    const float* xp[TT];
    const int kl = 4 * (lane >> 4);
#pragma unroll
    for (int r = 0; r < RT; r++) wp[r] = float_row<FMT>(m, row0 + 16 * r + (lane & 15), n_in);
#pragma unroll
    for (int t = 0; t < TT; t++) xp[t] = x + (int64_t)min(tok0 + 16 * t + (lane & 15), n_tok - 1) * n_in;
    f32x4_t acc[RT][TT];
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int t = 0; t < TT; t++) acc[r][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float4 wv[RT], xv[TT];
    auto load = [&](int s) {
#pragma unroll
        for (int r = 0; r < RT; r++) wv[r] = load_w4<FMT>(wp[r], 16 * s + kl);
#pragma unroll
        for (int t = 0; t < TT; t++) xv[t] = *(const float4*)(xp[t] + 16 * s + kl);
    };
    if (s0 < s1) load(s0);
#pragma unroll 4
    for (int s = s0; s < s1; s++) {
        float4 wc[RT], xc[TT];
#pragma unroll
        for (int r = 0; r < RT; r++) wc[r] = wv[r];
#pragma unroll
        for (int t = 0; t < TT; t++) xc[t] = xv[t];
        load(min(s + 1, s1 - 1));
#pragma unroll
        for (int r = 0; r < RT; r++)
#pragma unroll
            for (int t = 0; t < TT; t++) acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wc[r].x, xc[t].x, acc[r][t], 0, 0, 0);
#pragma unroll
        for (int r = 0; r < RT; r++)
#pragma unroll
            for (int t = 0; t < TT; t++) acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wc[r].y, xc[t].y, acc[r][t], 0, 0, 0);
#pragma unroll
        for (int r = 0; r < RT; r++)
#pragma unroll
            for (int t = 0; t < TT; t++) acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wc[r].z, xc[t].z, acc[r][t], 0, 0, 0);
#pragma unroll
        for (int r = 0; r < RT; r++)
#pragma unroll
            for (int t = 0; t < TT; t++) acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wc[r].w, xc[t].w, acc[r][t], 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int t = 0; t < TT; t++) part[wave][r * TT + t][lane] = acc[r][t];
    __syncthreads();
    // result register e of lane l: row 4 (l / 16) + e, token l % 16
    for (int i = threadIdx.x; i < RT * TT * 64; i += 64 * KW) {
        const int tile = i >> 6, l = i & 63;
        f32x4_t v = part[0][tile][l];
#pragma unroll
        for (int w = 1; w < KW; w++) v += part[w][tile][l];
        const int t = tok0 + 16 * (tile % TT) + (l & 15), j = row0 + 16 * (tile / TT) + 4 * (l >> 4);
        if (t >= n_tok) continue;
#pragma unroll
        for (int e = 0; e < 4; e++) float_store(m, t, j + e, out_scale != 1.0f ? v[e] * out_scale : v[e]);
    }
}

template <int FMT, int RT, int TT, int KW>
void launch_mfma(const FloatMats& m, const float* x, int n_in, int n_tok, float out_scale, hipStream_t s) {
    const int rows = m.n0 + m.n1;
    hipLaunchKernelGGL((float_mfma_k<FMT, RT, TT, KW>), dim3((rows + 16 * RT - 1) / (16 * RT), (n_tok + 16 * TT - 1) / (16 * TT)), dim3(64 * KW), 0,
                       s, m, x, n_in, n_tok, out_scale);
}

template <int FMT>
void run(const FloatMats& m, const float* x, int n_in, int n_tok, float out_scale, int exact, hipStream_t s) {
    const int rows = m.n0 + m.n1;
    auto al = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    const bool vec = n_in % 4 == 0 && al(m.w0) && al(m.w1) && al(x);
    if (exact && n_tok <= 8) {
        // (at eight tokens the folds' blocks still run side by side; a tile of 32 tokens would be three quarters padding)
        hipLaunchKernelGGL(float_fold_exact_k<FMT>, dim3((rows + EX_ROWS - 1) / EX_ROWS, n_tok), dim3(256), 0, s, m, x, n_in, out_scale);
    } else if (exact && vec) {
        const int64_t blocks4 = (int64_t)((rows + 63) / 64) * ((n_tok + 63) / 64);
        if (blocks4 >= 512)
            hipLaunchKernelGGL((float_tile_exact_k<FMT, 4>), dim3((rows + 63) / 64, (n_tok + 63) / 64), dim3(256), 0, s, m, x, n_in, n_tok, out_scale);
        else
            hipLaunchKernelGGL((float_tile_exact_k<FMT, 2>), dim3((rows + 31) / 32, (n_tok + 31) / 32), dim3(256), 0, s, m, x, n_in, n_tok, out_scale);
    } else if (!exact && vec && n_tok == 1) {
        hipLaunchKernelGGL(float_gemv_fast_k<FMT>, dim3((rows + 3) / 4), dim3(256), 0, s, m, x, n_in, out_scale);
    } else if (!exact && vec && n_in % 16 == 0) {
        // A CU is served operands at 30 GB/s whatever it holds: the tile that leaves the busiest of 256 CUs the fewest rows to read, its
        // blocks' times the rows and tokens of a tile (0.28 to 0.30 us each at 2,048 k with eight waves, 0.30 to 0.34 with four).  513 x
        // 2,048 over 201 / 333 / 512 / 1,024 / 5,700 tokens, the largest tile of 16 x 16, 32 x 32 and 32 x 64 that gives every SIMD a wave:
        // 17.6, 25.8, 33.1, 48.9, 163 us; so 14.1, 19.1, 28.2, 34.0, 152.
        struct Tile { int rt, tt; };
        constexpr Tile tile[] = {{1, 1}, {1, 2}, {2, 2}, {2, 4}, {3, 3}, {3, 4}};
        int best = 0;
        int64_t least = INT64_MAX, best_blocks = 0;
        for (int i = 0; i < 6; i++) {
            const int r = 16 * tile[i].rt, t = 16 * tile[i].tt;
            const int64_t blocks = (int64_t)((rows + r - 1) / r) * ((n_tok + t - 1) / t), cost = (blocks + 255) / 256 * (r + t);
            if (cost < least) least = cost, best = i, best_blocks = blocks;
        }
        switch (best) {
            case 0: launch_mfma<FMT, 1, 1, 8>(m, x, n_in, n_tok, out_scale, s); break;
            case 1: launch_mfma<FMT, 1, 2, 8>(m, x, n_in, n_tok, out_scale, s); break;
            case 2: launch_mfma<FMT, 2, 2, 8>(m, x, n_in, n_tok, out_scale, s); break;
            case 3:   // (with a second block on a CU four waves do: 129 x 2,048 over 5,700 tokens 64 and 59 us; alone 33 and 38)
                if (best_blocks > 256) launch_mfma<FMT, 2, 4, 4>(m, x, n_in, n_tok, out_scale, s);
                else launch_mfma<FMT, 2, 4, 8>(m, x, n_in, n_tok, out_scale, s);
                break;
            case 4: launch_mfma<FMT, 3, 3, 4>(m, x, n_in, n_tok, out_scale, s); break;
            default: launch_mfma<FMT, 3, 4, 4>(m, x, n_in, n_tok, out_scale, s); break;
        }
    } else {
        const int64_t total = (int64_t)rows * n_tok;
        hipLaunchKernelGGL(float_any_k<FMT>, dim3((unsigned)((total + 127) / 128)), dim3(128), 0, s, m, x, n_in, n_tok, out_scale);
    }
}

}  // namespace

void float_matmul(const FloatMats& m, int fmt, const float* x, int n_in, int n_tok, float out_scale, int exact, hipStream_t s) {
    if (m.n0 + m.n1 <= 0 || n_tok <= 0) return;
    if (fmt == W_F32) run<W_F32>(m, x, n_in, n_tok, out_scale, exact, s);
    else if (fmt == W_F16) run<W_F16>(m, x, n_in, n_tok, out_scale, exact, s);
    else run<W_BF16>(m, x, n_in, n_tok, out_scale, exact, s);
}

// matmul_pair with two unquantized matrices of one element type: one launch for both
bool float_matmul_pair(const WView& a, const WView& b, const float* x, int n_tok, float* out_a, float* out_b, int exact, hipStream_t s) {
    if (a.fmt != b.fmt || a.n_in != b.n_in || a.n_out <= 0 || b.n_out <= 0) return false;
    if (a.fmt != W_F32 && a.fmt != W_F16 && a.fmt != W_BF16) return false;
    float_matmul(FloatMats{(const uint8_t*)a.q, (const uint8_t*)b.q, out_a, out_b, a.n_out, b.n_out}, a.fmt, x, a.n_in, n_tok, 1.0f, exact, s);
    return true;
}

}  // namespace itk
