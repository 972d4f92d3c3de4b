// Quantized matmuls: weight repack, the decode GEMV (dense, per-expert, fused
// gate/up), and the tiled batch kernel.
//
// Arithmetic is the reference CPU path's (/root/reference src/ops/naive.rs):
//   Q8_0  (naive.rs:691-704): per 32-block  sumf += (float)isum * (dw * dx)
//   NVFP4 (naive.rs:714-734): per 16-sub-block sumf += (dy * d) * (float)(lo + hi)
// with the f32 chain walked serially in ascending block order.  Every per-block
// term is computed by its own lane (integer dot via v_dot4_i32_i8, exact), written
// to LDS, and one lane per output row folds the terms in order — so the result is
// the CPU result bit for bit while the HBM stream stays 128-bit coalesced.
#include "it_device.h"
#include "kernels.h"
#include "it_dot.h"

namespace itk {

// ------------------------------------------------------------------ repack
// file Q8_0 block = [f16 d][32 x i8]  ->  quants[row][n_in] + scales[row][n_in/32]
__global__ void repack_q8_0_k(const uint8_t* __restrict__ raw, int8_t* __restrict__ q,
                              uint16_t* __restrict__ scales, int64_t n_blocks) {
    // 8 lanes per block, 4 bytes each
    int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t b = gid >> 3;
    int sub = (int)(gid & 7);
    if (b >= n_blocks) return;
    const uint8_t* blk = raw + b * 34;
    // 34-byte blocks are only 2-byte aligned: assemble from u16 loads
    const uint16_t* p = (const uint16_t*)(blk + 2 + sub * 4);
    uint32_t v = (uint32_t)p[0] | ((uint32_t)p[1] << 16);
    *(uint32_t*)(q + b * 32 + sub * 4) = v;
    if (sub == 0) scales[b] = *(const uint16_t*)blk;
}
void repack_q8_0(const uint8_t* raw, int8_t* q, uint16_t* scales, int64_t n_rows, int n_in, hipStream_t s) {
    int64_t n_blocks = n_rows * (n_in / 32);
    if (n_blocks <= 0) return;
    int64_t threads = n_blocks * 8;
    hipLaunchKernelGGL(repack_q8_0_k, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, raw, q, scales,
                       n_blocks);
}

// file NVFP4 block = [4 x ue4m3][32 nibble bytes] -> nibbles[row][n_in/2] + scales[row][n_in/16]
__global__ void repack_nvfp4_k(const uint8_t* __restrict__ raw, uint8_t* __restrict__ nib,
                               uint8_t* __restrict__ scales, int64_t n_blocks) {
    // 9 dwords per block; 8 lanes move nibbles, lane 0 also moves the scales
    int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t b = gid >> 3;
    int sub = (int)(gid & 7);
    if (b >= n_blocks) return;
    const uint32_t* blk = (const uint32_t*)(raw + b * 36);
    ((uint32_t*)nib)[b * 8 + sub] = blk[1 + sub];
    if (sub == 0) ((uint32_t*)scales)[b] = blk[0];
}
void repack_nvfp4(const uint8_t* raw, uint8_t* nib, uint8_t* scales, int64_t n_rows, int n_in, hipStream_t s) {
    int64_t n_blocks = n_rows * (n_in / 64);
    if (n_blocks <= 0) return;
    int64_t threads = n_blocks * 8;
    hipLaunchKernelGGL(repack_nvfp4_k, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, raw, nib,
                       scales, n_blocks);
}

// ------------------------------------------------------------------ GEMV
struct GemvP {
    const uint8_t *q, *s;     // weights (gate when GLU)
    const uint8_t *q2, *s2;   // up weights when GLU
    int64_t q_stride, s_stride;  // bytes per expert (0 for a dense matrix)
    const uint8_t* const *q_tab, *const *s_tab, *const *q2_tab, *const *s2_tab;  // expert placement tables or null
    const int32_t* ids;       // expert id per y, or null
    const float *scale2, *scale2_up;  // per-expert second scales or null
    const float* act_scales;  // [x_rows][n_in/32]
    const int8_t* act_quants; // [x_rows][n_in]
    float* out;               // [n_y][n_out]
    int n_in, n_out, rows_per_wave;
    int x_mode, n_used;       // 0: row per y, 1: row y / n_used, 2: row 0
    float out_scale;
};

constexpr int GEMV_WAVES = 4;

template <int FMT, bool GLU>
__global__ __launch_bounds__(64 * GEMV_WAVES) void gemv_k(GemvP p) {
    extern __shared__ __align__(16) float lds[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int U = p.n_in >> 5;                     // 32-element units per row
    const int TPU = (FMT == W_NVFP4) ? 2 : 1;      // terms per unit
    const int T = U * TPU;                         // terms per row
    const int R = p.rows_per_wave;
    const int tstride = T + 4;
    float* terms = lds + (size_t)wave * R * tstride * (GLU ? 2 : 1);
    float* terms2 = terms + (size_t)R * tstride;

    const int y = blockIdx.y;
    const int row0 = (blockIdx.x * GEMV_WAVES + wave) * R;
    if (row0 >= p.n_out) return;
    const int nrows = min(R, p.n_out - row0);

    int64_t e = p.ids ? (int64_t)p.ids[y] : 0;
    const uint8_t* wq = it_expert_at(p.q, p.q_tab, e, p.q_stride);
    const uint8_t* ws = it_expert_at(p.s, p.s_tab, e, p.s_stride);
    const uint8_t* wq2 = GLU ? it_expert_at(p.q2, p.q2_tab, e, p.q_stride) : nullptr;
    const uint8_t* ws2 = GLU ? it_expert_at(p.s2, p.s2_tab, e, p.s_stride) : nullptr;
    int xr = p.x_mode == 0 ? y : (p.x_mode == 1 ? y / p.n_used : 0);
    const int8_t* aq = p.act_quants + (int64_t)xr * p.n_in;
    const float* as = p.act_scales + (int64_t)xr * U;

    const int items = nrows * U;
    for (int base = 0; base < items; base += 64) {
        int it = base + lane;
        if (it < items) {
            int r = it / U, u = it - r * U;
            int64_t row = row0 + r;
            const uint4* ap = (const uint4*)(aq + u * 32);
            uint4 a0 = ap[0], a1 = ap[1];
            float dx = as[u];
            if (FMT == W_Q8_0) {
                const uint4* wp = (const uint4*)(wq + row * p.n_in + u * 32);
                uint16_t dw = ((const uint16_t*)ws)[row * U + u];
                terms[r * tstride + u] = unit_q8_0(wp[0], wp[1], dw, a0, a1, dx);
                if (GLU) {
                    const uint4* wp2 = (const uint4*)(wq2 + row * p.n_in + u * 32);
                    uint16_t dw2 = ((const uint16_t*)ws2)[row * U + u];
                    terms2[r * tstride + u] = unit_q8_0(wp2[0], wp2[1], dw2, a0, a1, dx);
                }
            } else {
                uint4 w = *(const uint4*)(wq + row * (p.n_in >> 1) + u * 16);
                uint32_t sc = ((const uint16_t*)ws)[row * U + u];
                float tA, tB;
                unit_nvfp4(w, sc, a0, a1, dx, &tA, &tB);
                terms[r * tstride + 2 * u] = tA;
                terms[r * tstride + 2 * u + 1] = tB;
                if (GLU) {
                    uint4 w2 = *(const uint4*)(wq2 + row * (p.n_in >> 1) + u * 16);
                    uint32_t sc2 = ((const uint16_t*)ws2)[row * U + u];
                    unit_nvfp4(w2, sc2, a0, a1, dx, &tA, &tB);
                    terms2[r * tstride + 2 * u] = tA;
                    terms2[r * tstride + 2 * u + 1] = tB;
                }
            }
        }
    }
    // the wave's own LDS region: a wave-level barrier is enough
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    if (lane < nrows) {
        float acc = fold_terms(terms + lane * tstride, T);
        float* o = p.out + (int64_t)y * p.n_out + row0 + lane;
        if (GLU) {
            float acc2 = fold_terms(terms2 + lane * tstride, T);
            if (p.scale2) acc *= p.scale2[e];
            if (p.scale2_up) acc2 *= p.scale2_up[e];
            *o = it_silu(acc) * acc2;
        } else {
            if (p.scale2) acc *= p.scale2[e];
            if (p.out_scale != 1.0f) acc *= p.out_scale;
            *o = acc;
        }
    }
}

static int pick_rows_per_wave(int n_out, int n_y) {
    // aim for >= ~2048 waves in flight, cap the fold's idle lanes at 16 rows per wave
    int64_t want_waves = 2048;
    int64_t r = ((int64_t)n_out * n_y) / want_waves;
    int R = 1;
    while (R < 16 && R * 2 <= r) R *= 2;
    return R;
}

template <int FMT, bool GLU>
static void launch_gemv(GemvP p, int n_y, hipStream_t s) {
    int R = pick_rows_per_wave(p.n_out, n_y);
    int T = (p.n_in / 32) * (FMT == W_NVFP4 ? 2 : 1);
    auto lds_for = [&](int r) { return (size_t)GEMV_WAVES * r * (T + 4) * sizeof(float) * (GLU ? 2 : 1); };
    while (R > 1 && lds_for(R) > 48 * 1024) R /= 2;
    p.rows_per_wave = R;
    size_t lds = lds_for(R);
    int gx = (p.n_out + R * GEMV_WAVES - 1) / (R * GEMV_WAVES);
    hipLaunchKernelGGL((gemv_k<FMT, GLU>), dim3(gx, n_y), dim3(64 * GEMV_WAVES), lds, s, p);
}

void matmul(const WView& w, const float* x, const float* act_scales, const int8_t* act_quants, int n_tok,
            float* out, float out_scale, int exact, hipStream_t s) {
    if (n_tok <= 0 || w.n_out <= 0) return;
    if (!exact && q8_short(w, act_scales, act_quants, n_tok, out, out_scale, s)) return;
    // (fast mode adds each scaled block sum with one rounding: 4 ms of a 174 ms prefill pass)
    if (q8_gemm(w, act_scales, act_quants, n_tok, out, out_scale, s, !exact)) return;
    if (w.fmt == W_Q8_0 || w.fmt == W_NVFP4) {
        GemvP p{};
        p.q = (const uint8_t*)w.q;
        p.s = (const uint8_t*)w.scales;
        p.act_scales = act_scales;
        p.act_quants = act_quants;
        p.out = out;
        p.n_in = w.n_in;
        p.n_out = w.n_out;
        p.x_mode = 0;
        p.n_used = 1;
        p.out_scale = out_scale;
        if (w.fmt == W_Q8_0) launch_gemv<W_Q8_0, false>(p, n_tok, s);
        else launch_gemv<W_NVFP4, false>(p, n_tok, s);
        return;
    }
    const FloatMats m{(const uint8_t*)w.q, nullptr, out, nullptr, w.n_out, 0};
    float_matmul(m, w.fmt, x, w.n_in, n_tok, out_scale, exact, s);
}

static GemvP experts_params(const ExpertsView& w, const int32_t* ids, int n_used, int x_mode,
                            const float* act_scales, const int8_t* act_quants, float* out) {
    GemvP p{};
    p.q = (const uint8_t*)w.q;
    p.s = (const uint8_t*)w.scales;
    p.q_stride = w.q_stride;
    p.s_stride = w.s_stride;
    p.ids = ids;
    p.q_tab = w.q_tab;
    p.s_tab = w.s_tab;
    p.scale2 = w.scale2;
    p.act_scales = act_scales;
    p.act_quants = act_quants;
    p.out = out;
    p.n_in = w.n_in;
    p.n_out = w.n_out;
    p.x_mode = x_mode;
    p.n_used = n_used < 1 ? 1 : n_used;
    p.out_scale = 1.0f;
    return p;
}

void matmul_experts(const ExpertsView& w, const int32_t* ids, int n_picks, int n_used, int x_mode,
                    const float* act_scales, const int8_t* act_quants, float* out, hipStream_t s) {
    if (n_picks <= 0) return;
    GemvP p = experts_params(w, ids, n_used, x_mode, act_scales, act_quants, out);
    if (w.fmt == W_Q8_0) launch_gemv<W_Q8_0, false>(p, n_picks, s);
    else launch_gemv<W_NVFP4, false>(p, n_picks, s);
}

void moe_glu(const ExpertsView& gate, const ExpertsView& up, const int32_t* ids, int n_picks, int n_used,
             int x_mode, const float* act_scales, const int8_t* act_quants, float* out, hipStream_t s) {
    if (n_picks <= 0) return;
    GemvP p = experts_params(gate, ids, n_used, x_mode, act_scales, act_quants, out);
    p.q2 = (const uint8_t*)up.q;
    p.s2 = (const uint8_t*)up.scales;
    p.q2_tab = up.q_tab;
    p.s2_tab = up.s_tab;
    p.scale2_up = up.scale2;
    if (gate.fmt == W_Q8_0) launch_gemv<W_Q8_0, true>(p, n_picks, s);
    else launch_gemv<W_NVFP4, true>(p, n_picks, s);
}

}  // namespace itk
