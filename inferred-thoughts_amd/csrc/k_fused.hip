// Fused single-token kernels.
//
// A decode pass issues ~35 seam ops per layer, each a microsecond-scale kernel, so the
// pass is bound by launch latency rather than HBM.  When a decode pass is captured
// into a graph the backend rewrites runs of seam ops into the kernels below.  Each
// one performs exactly the arithmetic of the ops it replaces, in the same order
// (the `exact` flag keeps the serial f64 norm sums), so results do not change by a bit.
//
//   fused_gemv      [rms_norm] + quantize_q8_0 + up to 4 matmuls on one activation
//                   (+ causal conv + silu on the first output, or += into the output)
//   gdn_core        gather q/k/v + l2_norm(q,k) + delta_rule + rms_norm_heads + silu_mul
//   moe_glu_fused   [rms_norm + router + shared gate logit +] softmax + top-k + quantize + expert gate/up + shared gate/up + silu_mul
//   moe_down_fused  quantize + expert down + shared down + moe_finish + add_assign
//   attn_prep       gather q/gate + rms_norm_heads(q,k) + rope(q,k) + kv_write(k,v)
//   attn_merge_gate split-K merge + sigmoid_mul
#include <algorithm>
#include "it_device.h"
#include "it_dot.h"
#include "it_fast.h"
#include "it_launch.h"
#include "it_reduce.h"
#include "kernels.h"
#include "kernels_fused.h"

namespace itk {

// Q8_0 quantization of `n` floats in LDS (naive.rs:652-675), 8 lanes per 32-block.
__device__ void lds_quantize_q8_0(const float* xf, int n, float* xs, int8_t* xq) {
    const int nb = n >> 5;
    const int tid = threadIdx.x, sub = tid & 7;
    for (int base = 0; base < nb; base += (int)blockDim.x >> 3) {
        int b = base + (tid >> 3);
        bool live = b < nb;
        float4 v = live ? *(const float4*)(xf + b * 32 + sub * 4) : make_float4(0.f, 0.f, 0.f, 0.f);
        float amax = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
        amax = fmaxf(amax, __shfl_xor(amax, 1, 64));
        amax = fmaxf(amax, __shfl_xor(amax, 2, 64));
        amax = fmaxf(amax, __shfl_xor(amax, 4, 64));
        if (live) {
            float d = amax / 127.0f;
            float id = d != 0.0f ? 1.0f / d : 0.0f;
            float r[4] = {roundf(v.x * id), roundf(v.y * id), roundf(v.z * id), roundf(v.w * id)};
            uint32_t packed = 0;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float c = fminf(fmaxf(r[i], -128.0f), 127.0f);
                int q = (r[i] != r[i]) ? 0 : (int)c;
                packed |= ((uint32_t)(q & 0xff)) << (8 * i);
            }
            *(uint32_t*)(xq + b * 32 + sub * 4) = packed;
            if (sub == 0) xs[b] = it_f16_to_f32(it_f32_to_f16(d));
        }
    }
}

// The Q8_0 form of four values, eight neighbouring lanes a block (naive.rs:652-675): the quants and, in every lane, the f16 scale.
IT_DEV void quantize_quad(float4 v, uint32_t* packed, float* scale) {
    float amax = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
    amax = fmaxf(amax, dpp_xor1(amax));
    amax = fmaxf(amax, dpp_xor2(amax));
    amax = fmaxf(amax, dpp_half_mirror(amax));
    const float d = amax / 127.0f;
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    const float r[4] = {roundf(v.x * id), roundf(v.y * id), roundf(v.z * id), roundf(v.w * id)};
    uint32_t q = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float c = fminf(fmaxf(r[i], -128.0f), 127.0f);
        q |= ((uint32_t)(((r[i] != r[i]) ? 0 : (int)c) & 0xff)) << (8 * i);
    }
    *packed = q;
    *scale = it_f16_to_f32(it_f32_to_f16(d));
}

// Terms of `nrows` rows starting at `row0` of one matrix against the LDS activation.
// Two phases so every HBM load of the group is in flight before the first dot: a lane
// owns IPL (row, 32-element unit) items, loads them all, then computes.
// row of item `it` where a row has U units, inv = 1 / U: items are below 2^20, so the product is never within its rounding of
// a whole number (an integer division is some forty instructions, eight of them ahead of a wave's first loads)
IT_DEV int row_of(int it, float inv) { return (int)(((float)it + 0.5f) * inv); }
IT_DEV float inv_of(int n) { return __builtin_amdgcn_rcpf((float)n); }

template <int IPL>
struct RowRegs {
    uint4 wa[IPL], wb[IPL];
    uint32_t sc[IPL];
};

template <int FMT, int IPL>
__device__ __forceinline__ void load_items(RowRegs<IPL>& rr, const uint8_t* wq, const uint8_t* ws, int n_in, int row0,
                                           int nrows, int lane) {
    const int U = n_in >> 5;
    const int items = nrows * U;
    const float inv = inv_of(U);
#pragma unroll
    for (int k = 0; k < IPL; k++) {
        if (k * 64 >= items) break;
        int it = k * 64 + lane;
        if (it < items) {
            int r = row_of(it, inv), u = it - r * U;
            int64_t row = row0 + r;
            if (FMT == W_Q8_0) {
                const uint4* wp = (const uint4*)(wq + row * n_in + u * 32);
                rr.wa[k] = wp[0];
                rr.wb[k] = wp[1];
            } else {
                rr.wa[k] = *(const uint4*)(wq + row * (n_in >> 1) + u * 16);
            }
            rr.sc[k] = ((const uint16_t*)ws)[row * U + u];
        }
    }
}

template <int FMT, int IPL>
__device__ __forceinline__ void compute_items(const RowRegs<IPL>& rr, int n_in, int nrows, const int8_t* xq,
                                              const float* xs, float* terms, int tstride, int lane) {
    const int U = n_in >> 5;
    const int items = nrows * U;
    const float inv = inv_of(U);
#pragma unroll
    for (int k = 0; k < IPL; k++) {
        if (k * 64 >= items) break;
        int it = k * 64 + lane;
        if (it < items) {
            int r = row_of(it, inv), u = it - r * U;
            const uint4* ap = (const uint4*)(xq + u * 32);
            uint4 a0 = ap[0], a1 = ap[1];
            float dx = xs[u];
            if (FMT == W_Q8_0) {
                terms[r * tstride + u] = unit_q8_0(rr.wa[k], rr.wb[k], (uint16_t)rr.sc[k], a0, a1, dx);
            } else {
                float tA, tB;
                unit_nvfp4(rr.wa[k], rr.sc[k], a0, a1, dx, &tA, &tB);
                terms[r * tstride + 2 * u] = tA;
                terms[r * tstride + 2 * u + 1] = tB;
            }
        }
    }
}

template <int FMT, int IPL>
__device__ __forceinline__ void wave_row_terms_n(const uint8_t* wq, const uint8_t* ws, int n_in, int row0, int nrows,
                                                 const int8_t* xq, const float* xs, float* terms, int tstride,
                                                 int lane) {
    RowRegs<IPL> rr;
    load_items<FMT, IPL>(rr, wq, ws, n_in, row0, nrows, lane);
    compute_items<FMT, IPL>(rr, n_in, nrows, xq, xs, terms, tstride, lane);
}

// nrows * (n_in / 32) must not exceed 512 (the launchers size rows_per_wave for that)
template <int FMT>
__device__ void wave_row_terms(const uint8_t* wq, const uint8_t* ws, int n_in, int row0, int nrows,
                               const int8_t* xq, const float* xs, float* terms, int tstride, int lane) {
    const int items = nrows * (n_in >> 5);
    if (items <= 64) wave_row_terms_n<FMT, 1>(wq, ws, n_in, row0, nrows, xq, xs, terms, tstride, lane);
    else if (items <= 128) wave_row_terms_n<FMT, 2>(wq, ws, n_in, row0, nrows, xq, xs, terms, tstride, lane);
    else if (items <= 256) wave_row_terms_n<FMT, 4>(wq, ws, n_in, row0, nrows, xq, xs, terms, tstride, lane);
    else wave_row_terms_n<FMT, 8>(wq, ws, n_in, row0, nrows, xq, xs, terms, tstride, lane);
}

// ------------------------------------------------------------------ fused_gemv
// prologue modes: 0 = the activation as is; 1 = rms_norm(x, norm_w); 3 = that, and x left in x_raw; 2 = per-head
// rms_norm of x (weight norm_w[head_dim]) gated by silu(gate): silu(g) * ((x*scale)*w)
// ------------------------------------------------------------------ router in one wave
// softmax over up to 64 experts, then n_used rounds of arg-max with ties to the lower id, the
// picked probabilities summed in pick order (src/ops/mod.rs:1191-1216, naive.rs:362-376).
// Called by one wave; probs (LDS, n_expert floats) holds the logits on entry.  Lane e keeps expert e's probability; a round is one
// reduction over the wave for the value and a ballot for the lowest id that has it.
__device__ void wave_route(float* probs, int n_expert, int n_used, int* ids, float* weights, int lane, const uint64_t* etab) {
    const bool live = lane < n_expert;
    float v = live ? probs[lane] : -INFINITY;
    const float m = group_max<64>(v);
    v = live ? it_expf_by(v - m, etab) : -1.0f;
    if (live) probs[lane] = v;
    wave_lds_sync();
    const float sum = fold_terms(probs, n_expert);   // (every lane: the same reads)
    if (live) v = v / sum;
    float picked_p = 0.0f;  // lane r keeps pick r's probability
    int picked_id = -1;
    for (int r = 0; r < n_used; r++) {
        const float best = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, group_max_tail<64>(v)), 63));
        int id = best >= 0.0f ? -1 : r;   // (probabilities that are not numbers: some expert)
        const unsigned long long has = __ballot(v == best);   // taken and absent experts hold -1
        if (id < 0 && has) id = __builtin_ctzll(has);
        if (lane == r) {
            picked_p = best;
            picked_id = id;
        }
        if (lane == id) v = -1.0f;
    }
    // sum in pick order, serial f32
    float s = 0.0f;
    for (int r = 0; r < n_used; r++) s += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, picked_p), r));
    float denom = fmaxf(s, 6.103515625e-5f);
    if (lane < n_used) {
        ids[lane] = picked_id;
        weights[lane] = picked_p / denom;
    }
    wave_lds_sync();
}
constexpr int ROUTE_ITEMS = 4;
// LDS of the exponentials of a route by a whole block
__host__ IT_DEV size_t route_terms(int n_expert) { return ((size_t)n_expert * 4 + 15) & ~(size_t)15; }

constexpr int FG_THREADS = 512, FG_LDS_MAX = 128 * 1024, FG_MAX_IN = 8 * 64 * 32;

IT_DEV int mat_index(const FusedGemvP& p, int g) {
    int mi = 0;
#pragma unroll
    for (int k = 1; k < 4; k++)
        if (k < p.n_mats && g >= p.m[k].group0) mi = k;
    return mi;
}

// A router's logits are read by another block of the same launch: they go past the caches that the XCDs do not share.
IT_DEV void put_out(const FusedGemvP& p, const FusedMat& m, int j, float v) {
    if (p.route_counter) __hip_atomic_store(m.out + j, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else m.out[j] = v;
}
// what a row's epilogue reads, asked for long before: the conv window and taps (epi 1), the value it is added to (epi 2)
struct Epi {
    float p0, p1, p2, w0, w1, w2, w3;
};
IT_DEV Epi ask_epi(const FusedGemvP& p, const FusedMat& m, int row0, int nrows, int lane) {
    Epi e{};
    if (lane >= nrows) return e;
    const int64_t j = row0 + lane;
    if (m.epi == 2) {
        e.p0 = m.out[j];
    } else if (m.epi == 1) {
        const float *past = p.conv_state + j * 3, *w = p.conv_w + j * 4;
        e.p0 = past[0]; e.p1 = past[1]; e.p2 = past[2];
        e.w0 = w[0]; e.w1 = w[1]; e.w2 = w[2]; e.w3 = w[3];
    }
    return e;
}
// fold each row's terms in order and apply the matrix's epilogue
IT_DEV void finish_rows(const FusedGemvP& p, const FusedMat& m, int row0, int nrows, const float* terms, int tstride,
                        int nb, int lane, const Epi& e, const uint64_t* etab) {
    if (lane >= nrows) return;
    const int T = m.fmt == W_NVFP4 ? nb * 2 : nb;
    float acc = fold_terms(terms + lane * tstride, T);
    const int j = row0 + lane;
    if (m.epi == 0) {
        put_out(p, m, j, acc);
    } else if (m.epi == 2) {
        m.out[j] = e.p0 + acc;
    } else if (m.epi == 3) {
        m.out[j] = it_silu_by(acc, etab);
    } else {
        // causal conv (kernel 4) + silu on channel j, state [channel][3] oldest first
        float* past = p.conv_state + (int64_t)j * 3;
        float sum = 0.0f;
        sum += e.p0 * e.w0;
        sum += e.p1 * e.w1;
        sum += e.p2 * e.w2;
        sum += acc * e.w3;
        m.out[j] = it_silu_by(sum, etab);
        past[0] = e.p1;
        past[1] = e.p2;
        past[2] = acc;
    }
}

typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));   // four floats, wherever they start
IT_DEV float4 load4(const float* p) {
    const f4u v = *(const f4u*)p;
    return make_float4(v.x, v.y, v.z, v.w);
}
IT_DEV void store4(float* p, float4 v) { *(f4u*)p = f4u{v.x, v.y, v.z, v.w}; }

// Blocks 0 .. q_blocks - 1 take the quantized rows, the rest the unquantized ones, whose fold is a chain of n_in additions (eight
// cycles each: 2,048 take 7.5 us) that nothing else should wait for.
// Bound by the chain activation -> norm -> Q8_0 -> dots -> fold -> epilogue of dependent instructions between two launches.  So a
// thread keeps its four values of the activation (and of norm weight and gate) in registers from the load to the quants, one
// barrier for the norm's sum and one for the quants; what a row's epilogue reads is asked for ahead of it, the exponential's
// table sits in LDS, and a wave's row, scalar, is found without integer divisions.  512 values, 1,552 rows: 6.4 -> 5.0 us;
// 2,048 values, 12,288 Q8_0 and 64 F32 rows 28.6 -> 11.7 (the F32 rows' LDS left one quantized row a pass), 513 F32 rows and
// the route 24.9 -> 24.5.
template <int NQ>
__global__ __launch_bounds__(FG_THREADS) void fused_gemv_k(FusedGemvP p) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ double red[FG_THREADS / 64 + 1];
    __shared__ uint64_t etab[32];
    constexpr int W = FG_THREADS / 64;
    const int n_in = p.n_in, nb = n_in >> 5;
    float* xf = (float*)smem;
    float* xs = xf + n_in;
    int8_t* xq = (int8_t*)(xs + ((nb + 3) & ~3));
    float* terms_all = (float*)(xq + n_in);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool quantized = (int)blockIdx.x < p.q_blocks;

    // the activation first, then the first row group's weights: they move while the prologue runs
    float4 xv[NQ], wv[NQ], gv[NQ];
#pragma unroll
    for (int j = 0; j < NQ; j++) {
        const int i = 4 * (tid + FG_THREADS * j);
        xv[j] = wv[j] = gv[j] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (i < n_in) {
            xv[j] = load4(p.x + i);
            if (p.mode & 1) wv[j] = load4(p.norm_w + i);
            if (p.mode == 2) {
                wv[j] = load4(p.norm_w + i % p.head_dim);
                gv[j] = load4(p.gate + i);
            }
        }
    }
    if (tid < 32) etab[tid] = IT_EXP2F_TAB[tid];
    const int R = p.rows_per_wave;
    const int tstride = nb * 2 + 4;
    float* terms = terms_all + (size_t)wave * (quantized ? p.terms_stride : n_in);
    const int g0 = blockIdx.x * W + wave;
    const bool has0 = quantized && g0 < p.total_groups;
    const FusedMat& m0 = p.m[has0 ? mat_index(p, g0) : 0];
    const int row00 = has0 ? (g0 - m0.group0) * R : 0;
    const int nrows0 = has0 ? min(R, m0.n_out - row00) : 0;
    RowRegs<8> rr;
    Epi epi{};
    if (has0) {
        if (m0.fmt == W_NVFP4) load_items<W_NVFP4, 8>(rr, m0.q, m0.s, n_in, row00, nrows0, lane);
        else load_items<W_Q8_0, 8>(rr, m0.q, m0.s, n_in, row00, nrows0, lane);
        epi = ask_epi(p, m0, row00, nrows0, lane);
    }
    // unquantized rows: one a wave at a time, dealt out over the blocks first
    const int f_blocks = gridDim.x - p.q_blocks;
    auto frow = [&](int fr) __attribute__((always_inline)) {   // (matrix, row)
        int k = p.n_mats;
        while (fr >= p.m[k].n_out) fr -= p.m[k++].n_out;
        return make_int2(k, fr);
    };
    constexpr int FW = 8;                            // of 256 floats each: what is asked for ahead of the prologue
    float4 fw[FW];
    const int fr0 = wave * f_blocks + (int)blockIdx.x - p.q_blocks;
    if (!quantized && fr0 < p.total_frows) {
        const int2 at = frow(fr0);
        const float* row = (const float*)p.m[at.x].q + (int64_t)at.y * n_in;
#pragma unroll
        for (int c = 0; c < FW; c++)
            if (c * 256 < n_in) fw[c] = *(const float4*)(row + c * 256 + lane * 4);
    }

    auto squares = [](float4 v) __attribute__((always_inline)) {
        double s = (double)(v.x * v.x);
        s += (double)(v.y * v.y);
        s += (double)(v.z * v.z);
        s += (double)(v.w * v.w);
        return s;
    };
    if (p.mode & 1) {
        double part = 0.0;
#pragma unroll
        for (int j = 0; j < NQ; j++) {
            const int i = 4 * (tid + FG_THREADS * j);
            part += squares(xv[j]);
            if (i < n_in) *(float4*)(xf + i) = xv[j];      // for the serial sum, should it be needed
        }
        part = wave_sum_f64_tail(part);
        if (lane == 63) red[wave] = part;
        __syncthreads();
        double sum = 0.0;
        for (int w = 0; w < W; w++) sum += red[w];
        float mean = (float)over(sum, n_in);
        if (p.exact && !mean_is_certain(sum, n_in, n_in, &mean)) {   // (the same answer in every thread)
            __syncthreads();
            if (tid == 0) {
                sum = 0.0;
                for (int i = 0; i < n_in; i++) sum += (double)(xf[i] * xf[i]);
                red[0] = sum;
            }
            __syncthreads();
            mean = (float)over(red[0], n_in);
        }
        const float scale = 1.0f / sqrtf(mean + p.eps);
#pragma unroll
        for (int j = 0; j < NQ; j++) {
            xv[j].x = xv[j].x * scale * wv[j].x;
            xv[j].y = xv[j].y * scale * wv[j].y;
            xv[j].z = xv[j].z * scale * wv[j].z;
            xv[j].w = xv[j].w * scale * wv[j].w;
        }
    } else if (p.mode == 2) {
        const int hd = p.head_dim, lph = hd / 4;     // 16 or 32 lanes a head
#pragma unroll
        for (int j = 0; j < NQ; j++) {
            double sum = squares(xv[j]);
            sum += dpp_f64(sum, 0);
            sum += dpp_f64(sum, 1);
            sum += dpp_f64(sum, 2);
            sum += dpp_f64(sum, 3);
            if (lph == 32) sum += __shfl_xor(sum, 16, 64);
            float mean = (float)over(sum, hd);
            if (p.exact && !mean_is_certain(sum, hd, hd, &mean)) {   // (the same answer in every lane of the head)
                sum = 0.0;
                for (int l = 0; l < lph; l++) {
                    const int from = (lane & ~(lph - 1)) + l;
                    const float a = __shfl(xv[j].x, from, 64), b = __shfl(xv[j].y, from, 64), c = __shfl(xv[j].z, from, 64), d = __shfl(xv[j].w, from, 64);
                    sum += (double)(a * a);
                    sum += (double)(b * b);
                    sum += (double)(c * c);
                    sum += (double)(d * d);
                }
                mean = (float)over(sum, hd);
            }
            const float scale = 1.0f / sqrtf(mean + p.eps);
            xv[j].x = gv[j].x * (xv[j].x * scale * wv[j].x);
            xv[j].y = gv[j].y * (xv[j].y * scale * wv[j].y);
            xv[j].z = gv[j].z * (xv[j].z * scale * wv[j].z);
            xv[j].w = gv[j].w * (xv[j].w * scale * wv[j].w);
        }
    }
#pragma unroll
    for (int j = 0; j < NQ; j++) {
        const int i = 4 * (tid + FG_THREADS * j);
        const bool live = i < n_in;
        if (blockIdx.x == 0 && live) {
            if (p.x_copy) store4(p.x_copy + i, xv[j]);
            if (p.x_copy2) store4(p.x_copy2 + i, xv[j]);
        }
        if (quantized) {
            uint32_t packed;
            float d;
            quantize_quad(xv[j], &packed, &d);
            if (live) {
                *(uint32_t*)(xq + i) = packed;
                if ((tid & 7) == 0) xs[i >> 5] = d;
            }
        } else if (live) {
            *(float4*)(xf + i) = xv[j];
        }
    }
    __syncthreads();

    if (has0) {
        if (m0.fmt == W_NVFP4) compute_items<W_NVFP4, 8>(rr, n_in, nrows0, xq, xs, terms, tstride, lane);
        else compute_items<W_Q8_0, 8>(rr, n_in, nrows0, xq, xs, terms, tstride, lane);
        wave_lds_sync();
        finish_rows(p, m0, row00, nrows0, terms, tstride, nb, lane, epi, etab);
        wave_lds_sync();
    }
    if (quantized) {
        for (int g = g0 + p.q_blocks * W; g < p.total_groups; g += p.q_blocks * W) {
            const FusedMat& m = p.m[mat_index(p, g)];
            const int row0 = (g - m.group0) * R;
            const int nrows = min(R, m.n_out - row0);
            const Epi e = ask_epi(p, m, row0, nrows, lane);
            if (m.fmt == W_NVFP4) wave_row_terms<W_NVFP4>(m.q, m.s, n_in, row0, nrows, xq, xs, terms, tstride, lane);
            else wave_row_terms<W_Q8_0>(m.q, m.s, n_in, row0, nrows, xq, xs, terms, tstride, lane);
            wave_lds_sync();
            finish_rows(p, m, row0, nrows, terms, tstride, nb, lane, e, etab);
            wave_lds_sync();
        }
    } else {
        // the wave forms a row's products, one lane folds them in order (naive.rs:843-861)
        for (int fr = fr0; fr < p.total_frows; fr += W * f_blocks) {
            const int2 at = frow(fr);
            const FusedMat& m = p.m[at.x];
            const float* row = (const float*)m.q + (int64_t)at.y * n_in;
            auto products = [&](int i, float4 w) __attribute__((always_inline)) {
                const float4 x = *(const float4*)(xf + i);
                *(float4*)(terms + i) = make_float4(w.x * x.x, w.y * x.y, w.z * x.z, w.w * x.w);
            };
#pragma unroll
            for (int c = 0; c < FW; c++)
                if (c * 256 < n_in) products(c * 256 + lane * 4, fr == fr0 ? fw[c] : *(const float4*)(row + c * 256 + lane * 4));
#pragma unroll 8
            for (int i = FW * 256 + lane * 4; i < n_in; i += 256) products(i, *(const float4*)(row + i));
            wave_lds_sync();
            const float sum = fold_terms(terms, n_in);   // (every lane: reads of one address by all cost less than by one lane)
            if (lane == 0) put_out(p, m, at.y, sum);
            wave_lds_sync();
        }
    }
    if (p.mode == 3 && blockIdx.x == gridDim.x - 1)   // (behind everything: in the prologue it cost every launch, this one or not, 0.1 us)
        for (int i = 4 * tid; i < n_in; i += 4 * FG_THREADS) store4(p.x_raw + i, load4(p.x + i));
    if (p.route_counter) {
        // The block that finishes last turns the router logits (matrix 0's output) into the
        // token's expert choice, so the next kernel starts with the ids in hand.
        __shared__ int is_last;
        __builtin_amdgcn_s_waitcnt(0);   // the logits went past the caches (put_out): they are there, no fence needed
        __syncthreads();
        if (tid == 0 && gridDim.x == 1) {
            is_last = 1;
        } else if (tid == 0) {
            unsigned prev = __hip_atomic_fetch_add(p.route_counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            is_last = prev == gridDim.x - 1;
        }
        __syncthreads();
        if (is_last) {
            // By the whole block: 512 experts took one wave 10.9 us (exponentials eight a lane, ten rounds of arg-max over
            // eight registers), this 3.5.  (The activation and the terms are done with: their LDS holds the experts' exponentials and the
            // pick's candidates.)
            __shared__ int rids[16];
            __shared__ __align__(16) float rwts[16];
            auto& sh = *(fastk::RouteLds<FG_THREADS>*)(smem + route_terms(p.n_expert));
            float l[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int e = tid + k * FG_THREADS;
                l[k] = e < p.n_expert ? __hip_atomic_load(p.route_logits + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : -INFINITY;
            }
            const float denom = fastk::block_route<FG_THREADS, true>(l, p.n_expert, p.n_used, sh, rids, rwts, etab, (float*)smem);
            if (tid < p.n_used) {
                p.route_ids[tid] = rids[tid];
                p.route_w[tid] = rwts[tid] / denom;
            }
            if (tid == 0) *p.route_counter = 0u;
        }
    }
}

// LDS of a block: the activation (f32, scales, quants) and the terms of r rows a wave
static size_t fg_base(int n_in) { return (size_t)n_in * 4 + (size_t)((n_in / 32 + 3) & ~3) * 4 + n_in; }
static size_t fg_lds(int n_in, int r) { return fg_base(n_in) + (size_t)(FG_THREADS / 64) * r * (n_in / 32 * 2 + 4) * 4; }

void fused_gemv(FusedGemvP p, hipStream_t s) {
    if (fused_gemv_fast(p, s)) return;
    constexpr int W = FG_THREADS / 64;
    // unquantized matrices behind the quantized ones
    p.route_logits = p.m[0].out;
    FusedMat all[4];
    int nq = 0, nf = 0, total_rows = 0;
    for (int i = 0; i < p.n_mats; i++)
        if (p.m[i].fmt != W_F32) all[nq++] = p.m[i];
    for (int i = 0; i < p.n_mats; i++)
        if (p.m[i].fmt == W_F32) all[nq + nf++] = p.m[i];
    p.total_frows = 0;
    for (int i = 0; i < nq + nf; i++) {
        p.m[i] = all[i];
        if (i < nq) total_rows += all[i].n_out;
        else p.total_frows += all[i].n_out;
    }
    p.n_mats = nq;
    p.n_fmats = nf;
    const int nb = p.n_in / 32;
    // enough waves to cover HBM latency: aim for ~4096 row groups, at most 512 items per wave pass
    // fewest passes per wave over 256 blocks of W waves, then the fewest rows per pass
    int R = 1;
    {
        int best = 1 << 30;
        for (int r = 1; r <= 16 && r * nb <= 512; r *= 2) {
            int passes = ((total_rows + r - 1) / r + 256 * W - 1) / (256 * W);
            if (passes < best) {
                best = passes;
                R = r;
            }
        }
    }
    // a router whose rows one block can take in one pass: nothing has to be handed from block to block
    if (p.route_counter && !nf)
        for (int r = 1; r <= 16 && r * nb <= 512; r *= 2)
            if ((total_rows + r - 1) / r <= W) {
                R = r;
                break;
            }
    while (R > 1 && fg_lds(p.n_in, R) > 60 * 1024) R /= 2;
    p.rows_per_wave = R;
    p.terms_stride = R * (nb * 2 + 4);
    int g = 0;
    for (int i = 0; i < nq; i++) {
        p.m[i].group0 = g;
        g += (p.m[i].n_out + R - 1) / R;
    }
    p.total_groups = g;
    // one block per CU: every block pays the activation prologue, so more blocks than CUs
    // only repeats it (measured: 256 blocks 12 us, 772 blocks 22 us for norm + 12k rows of 2048)
    p.q_blocks = std::min((g + W - 1) / W, 256);
    // the unquantized rows on what CUs are left, or eight to a block
    const int f_blocks = nf ? std::min(p.total_frows, std::max(256 - p.q_blocks, (p.total_frows + W - 1) / W)) : 0;
    const int f_waves = nf ? std::min(W, (p.total_frows + f_blocks - 1) / f_blocks) : 0;
    const int blocks = std::max(1, p.q_blocks + f_blocks);
    size_t lds = std::max(nq ? fg_lds(p.n_in, R) : fg_base(p.n_in), fg_base(p.n_in) + (size_t)f_waves * p.n_in * 4);
    if (p.route_counter) lds = std::max(lds, route_terms(p.n_expert) + sizeof(fastk::RouteLds<FG_THREADS>));
    auto launch = [&](auto kernel) {
        if (lds > 64 * 1024) (void)lds_allowed<decltype(kernel)::value>(FG_LDS_MAX);   // (refused: the launch reports it)
        hipLaunchKernelGGL(decltype(kernel)::value, dim3(blocks), dim3(FG_THREADS), lds, s, p);
    };
    if (p.n_in <= 4 * FG_THREADS) launch(KernelIs<&fused_gemv_k<1>>{});
    else if (p.n_in <= 8 * FG_THREADS) launch(KernelIs<&fused_gemv_k<2>>{});
    else if (p.n_in <= 16 * FG_THREADS) launch(KernelIs<&fused_gemv_k<4>>{});
    else launch(KernelIs<&fused_gemv_k<8>>{});   // (fused_gemv_takes admits no more)
}
// F32 rows beside (or in place of) quantized ones, in the kernel that keeps the CPU path's order
static bool fused_gemv_exact_takes(const FusedGemvP& p) {
    for (int i = 0; i < p.n_mats; i++) {
        if (p.m[i].fmt == W_Q8_0 || p.m[i].fmt == W_NVFP4) continue;
        if (p.m[i].fmt != W_F32 || p.m[i].epi != 0 || (reinterpret_cast<uintptr_t>(p.m[i].q) & 15)) return false;
    }
    return p.n_in % 256 == 0 && p.n_in <= FG_MAX_IN && std::max(fg_lds(p.n_in, 1), fg_base(p.n_in) + (size_t)(FG_THREADS / 64) * p.n_in * 4) <= FG_LDS_MAX;
}
// (A wave takes a row's 32-value units at once, eight a lane, and a thread holds its quads of the activation: rows of more than
// 16,384 values are left to the ops one by one.  Every block reads the whole activation, at its own time: what block 0 leaves and
// what the rows' waves write lies elsewhere.)
bool fused_gemv_takes(const FusedGemvP& p) {
    if (p.x_copy == p.x || p.x_copy2 == p.x || (p.mode == 3 && p.x_raw == p.x)) return false;
    for (int i = 0; i < p.n_mats; i++)
        if (p.m[i].out == p.x || p.m[i].out == p.gate) return false;   // (mode 3: or x_raw)
    if (p.mode == 2 && ((p.head_dim != 64 && p.head_dim != 128) || p.n_in % p.head_dim)) return false;   // (a head is a row of 16 lanes, or two)
    bool floats = false;
    for (int i = 0; i < p.n_mats; i++) floats |= p.m[i].fmt != W_Q8_0 && p.m[i].fmt != W_NVFP4;
    if (floats) return p.exact ? fused_gemv_exact_takes(p) : fused_gemv_fast_takes(p);
    return p.n_in <= FG_MAX_IN;
}

// ------------------------------------------------------------------ gdn rows
// Fast form for a block of 256 threads: thread t < DK holds k[t], thread DK + t holds q[t]; each
// vector's sum of squares is reduced in its own waves, two barriers in all.
// `v` is the thread's element, loaded by the caller (ahead of its other loads: loads return in order).
template <int DK>
__device__ __forceinline__ void l2_kq_fast(float v, float eps, float* kq, double* red) {
    static_assert(DK == 64 || DK == 128, "one or two waves per vector");
    constexpr int WPV = DK / 64;  // waves per vector
    const int tid = threadIdx.x, wave = tid >> 6;
    const bool live = tid < 2 * DK;
    const bool is_q = tid >= DK;
    const int i = is_q ? tid - DK : tid;
    const double part = wave_sum_f64_tail((double)(v * v));
    if ((tid & 63) == 63) red[wave] = part;
    __syncthreads();
    if (live) {
        const int w0 = is_q ? WPV : 0;
        double sum = red[w0];
        if (WPV == 2) sum += red[w0 + 1];
        const float scale = 1.0f / fmaxf(sqrtf((float)sum), eps);
        kq[(is_q ? DK : 0) + i] = v * scale;
    }
    __syncthreads();
}

IT_DEV void gdn_gates(float a, float ssm_a, float b, const uint64_t* etab, const double (*ltab)[2], float* g, float* beta) {
    float softplus = a > 20.0f ? a : it_logf_by(1.0f + it_expf_by(a, etab), ltab);
    *g = it_expf_by(softplus * ssm_a, etab);
    *beta = 1.0f / (1.0f + it_expf_by(-b, etab));
}
// the same on the transcendental unit, for the kernel that reorders its sums anyway
IT_DEV void gdn_gates_fast(const GdnCoreP& p, int h, float* g, float* beta) {
    float a = p.alpha[h] + p.dt_bias[h];
    float softplus = a > 20.0f ? a : fx_logf(1.0f + fx_expf(a));
    *g = fx_expf(softplus * p.ssm_a[h]);
    *beta = fx_sigmoid(p.beta[h]);
}

// Exact form: one lane owns one value row, the three sweeps run in the CPU path's order: chains of DK additions, eight cycles each.
// What is in front of them is asked for at once, and the tables of the gates' exponentials and logarithm sit in LDS (four
// lookups in constant memory, one behind the other, cost as much as a sweep): heads of 64 5.1 -> 4.1 us, of 128 8.4 -> 7.4.
template <int DK>
__global__ __launch_bounds__(64) void gdn_rows_exact_k(GdnCoreP p) {
    __shared__ __align__(16) float kq[2 * DK];
    __shared__ uint64_t etab[32];
    __shared__ double ltab[16][2];
    constexpr int PER = DK / 64;                 // of the key's and of the query's values a lane
    const int lane = threadIdx.x;
    const int dv = DK;
    const int bph = dv / 64;
    const int h = blockIdx.x / bph, jb = blockIdx.x % bph, kh = h % p.n_k_heads;
    const int key_dim = p.n_k_heads * DK;
    float kv[2][PER];
#pragma unroll
    for (int i = 0; i < PER; i++) {
        kv[0][i] = p.conv[key_dim + kh * DK + lane + 64 * i];
        kv[1][i] = p.conv[kh * DK + lane + 64 * i];
    }
    if (lane < 32) etab[lane] = IT_EXP2F_TAB[lane];
    if (lane < 16) {
        ltab[lane][0] = IT_LOGF_TAB[lane][0];
        ltab[lane][1] = IT_LOGF_TAB[lane][1];
    }
    const float a = p.alpha[h] + p.dt_bias[h], ssm_a = p.ssm_a[h], b = p.beta[h];
    const int j = jb * 64 + lane;
    const float v = p.conv[2 * key_dim + h * dv + j];
    float* S = p.state + ((int64_t)h * dv + j) * DK;
    float row[DK];
    const float4* S4 = (const float4*)S;
#pragma unroll
    for (int i = 0; i < DK / 4; i++) {
        float4 t = S4[i];
        row[4 * i] = t.x; row[4 * i + 1] = t.y; row[4 * i + 2] = t.z; row[4 * i + 3] = t.w;
    }
    wave_lds_sync();
    // l2-normalised k (first half of kq) and q (second half) (naive.rs:254-273)
#pragma unroll
    for (int which = 0; which < 2; which++) {
        double part = 0.0;
#pragma unroll
        for (int i = 0; i < PER; i++) part += (double)(kv[which][i] * kv[which][i]);
        part = wave_sum_f64_tail(part);
        const unsigned long long u = __builtin_bit_cast(unsigned long long, part);
        const unsigned lo = __builtin_amdgcn_readlane((int)(u & 0xffffffffull), 63), hi = __builtin_amdgcn_readlane((int)(u >> 32), 63);
        double sum = __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
        float total = (float)sum;
        if (p.exact && !mean_is_certain(sum, DK, 1, &total)) {
            sum = 0.0;
            for (int i = 0; i < DK; i++) {
                const float x = __shfl(kv[which][i / 64], i & 63, 64);
                sum += (double)(x * x);
            }
            total = (float)sum;
        }
        const float scale = 1.0f / fmaxf(sqrtf(total), p.eps);
#pragma unroll
        for (int i = 0; i < PER; i++) kq[which * DK + lane + 64 * i] = kv[which][i] * scale;
    }
    float g, beta;
    gdn_gates(a, ssm_a, b, etab, ltab, &g, &beta);
    wave_lds_sync();
    const float4* k4 = (const float4*)kq;
    const float4* q4 = (const float4*)(kq + DK);
    float pred = 0.0f;
#pragma unroll
    for (int i = 0; i < DK; i += 4) {
        float4 kk = k4[i / 4];
        row[i] *= g;     pred += row[i] * kk.x;
        row[i + 1] *= g; pred += row[i + 1] * kk.y;
        row[i + 2] *= g; pred += row[i + 2] * kk.z;
        row[i + 3] *= g; pred += row[i + 3] * kk.w;
    }
    float delta = beta * (v - pred);
    float o = 0.0f;
#pragma unroll
    for (int i = 0; i < DK; i += 4) {
        float4 kk = k4[i / 4], qq = q4[i / 4];
        row[i] += kk.x * delta;     o += row[i] * (qq.x * p.q_scale);
        row[i + 1] += kk.y * delta; o += row[i + 1] * (qq.y * p.q_scale);
        row[i + 2] += kk.z * delta; o += row[i + 2] * (qq.z * p.q_scale);
        row[i + 3] += kk.w * delta; o += row[i + 3] * (qq.w * p.q_scale);
    }
    float4* W4 = (float4*)S;
#pragma unroll
    for (int i = 0; i < DK / 4; i++) W4[i] = make_float4(row[4 * i], row[4 * i + 1], row[4 * i + 2], row[4 * i + 3]);
    p.core[h * dv + j] = o;
}

// Fast form: LPR lanes share a row (each a contiguous DK/LPR slice, so a row is one 512-byte coalesced read), partial
// dots meet through DPP moves.  Reordered sums: 1e-3 class.  LPR = 8 gives 32 rows per block, LPR = 16 gives 16: the
// launcher takes the one that puts a block on every CU (32 value heads of 128 rows: 256 blocks with LPR = 16).
template <int DK, int LPR>
__global__ __launch_bounds__(256) void gdn_rows_fast_k(GdnCoreP p) {
    constexpr int SEG = DK / LPR;
    constexpr int ROWS = 256 / LPR;
    __shared__ __align__(16) float kq[2 * DK];
    __shared__ double red[5];
    const int tid = threadIdx.x, seg = tid % LPR;
    const int dv = DK;
    const int bph = dv / ROWS;
    const int h = blockIdx.x / bph, jb = blockIdx.x % bph, kh = h % p.n_k_heads;
    const int key_dim = p.n_k_heads * DK;
    // key / query element first, then the state rows: both are in flight while k and q are normalized
    const float kqv = tid < 2 * DK ? p.conv[(tid >= DK ? 0 : key_dim) + kh * DK + (tid >= DK ? tid - DK : tid)] : 0.0f;
    const int j = jb * ROWS + tid / LPR;
    float* S = p.state + ((int64_t)h * dv + j) * DK + seg * SEG;
    float4 st[SEG / 4];
#pragma unroll
    for (int i = 0; i < SEG / 4; i++) st[i] = ((const float4*)S)[i];
    l2_kq_fast<DK>(kqv, p.eps, kq, red);
    float row[SEG];
#pragma unroll
    for (int i = 0; i < SEG / 4; i++) {
        row[4 * i] = st[i].x; row[4 * i + 1] = st[i].y; row[4 * i + 2] = st[i].z; row[4 * i + 3] = st[i].w;
    }
    float g, beta;
    gdn_gates_fast(p, h, &g, &beta);
    float v = p.conv[2 * key_dim + h * dv + j];
    const float* kk = kq + seg * SEG;
    const float* qq = kq + DK + seg * SEG;
    float pred = 0.0f;
#pragma unroll
    for (int i = 0; i < SEG; i++) {
        row[i] *= g;
        pred += row[i] * kk[i];
    }
    pred = group_sum<LPR>(pred);
    float delta = beta * (v - pred);
    float o = 0.0f;
#pragma unroll
    for (int i = 0; i < SEG; i++) {
        row[i] += kk[i] * delta;
        o += row[i] * (qq[i] * p.q_scale);
    }
    o = group_sum<LPR>(o);
#pragma unroll
    for (int i = 0; i < SEG / 4; i++)
        ((float4*)S)[i] = make_float4(row[4 * i], row[4 * i + 1], row[4 * i + 2], row[4 * i + 3]);
    if (seg == 0) p.core[h * dv + j] = o;
}

void gdn_core(const GdnCoreP& p, int dk, hipStream_t s) {
    if (p.exact) {
        int blocks = p.n_v_heads * (dk / 64);
        if (dk == 64) hipLaunchKernelGGL(gdn_rows_exact_k<64>, dim3(blocks), dim3(64), 0, s, p);
        else if (dk == 128) hipLaunchKernelGGL(gdn_rows_exact_k<128>, dim3(blocks), dim3(64), 0, s, p);
    } else {
        // sixteen lanes a row while that still leaves at most a block per CU (256 on this chip), eight otherwise
        const bool wide = p.n_v_heads * (dk / 16) <= 256;
        const int blocks = p.n_v_heads * (dk / (wide ? 16 : 32));
        if (dk == 64 && wide) hipLaunchKernelGGL((gdn_rows_fast_k<64, 16>), dim3(blocks), dim3(256), 0, s, p);
        else if (dk == 64) hipLaunchKernelGGL((gdn_rows_fast_k<64, 8>), dim3(blocks), dim3(256), 0, s, p);
        else if (dk == 128 && wide) hipLaunchKernelGGL((gdn_rows_fast_k<128, 16>), dim3(blocks), dim3(256), 0, s, p);
        else if (dk == 128) hipLaunchKernelGGL((gdn_rows_fast_k<128, 8>), dim3(blocks), dim3(256), 0, s, p);
    }
}

// ------------------------------------------------------------------ moe_glu_fused
// grid (row blocks, n_used + 1): y < n_used is routed pick y, y == n_used the shared expert.
// What bounds it and how it is laid out: as fused_gemv_k (the activation's quads in registers up to the quants, NQ a thread; 0: too many to hold).
// ROUTE: a router of few rows in front, its norm, rows and picks formed by every block.  As a launch of its own it took 1.6 us
// between two launches, 1 us for the activation's trip, 1.2 to norm, quants and dots, and 2.8 for the logits' way out of the
// block's registers, back and the picks; repeated in each block it takes no more time than in one, and the logits stay in LDS
// (four layers of 512 with 16 experts, a prompt of 32 and 64 tokens: 9.11 -> 8.02 ms).
template <int NQ, bool ROUTE>
__global__ __launch_bounds__(256) void moe_glu_fused_k(MoeGluP p) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ uint64_t etab[32];
    const int n_in = p.n_in, nb = n_in >> 5;
    float* xs = (float*)smem;
    int8_t* xq = (int8_t*)(xs + ((nb + 3) & ~3));
    float* terms_all = (float*)(xq + n_in);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int y = blockIdx.y;
    const bool shared = y == p.n_used;
    int64_t e = ROUTE || shared ? 0 : p.route_ids[y];
    auto quad = [&](int j) __attribute__((always_inline)) {
        const int i = 4 * (tid + 256 * j);
        return i < n_in ? load4(p.x + i) : make_float4(0.f, 0.f, 0.f, 0.f);
    };
    float4 xv[NQ ? NQ : 1];
#pragma unroll
    for (int j = 0; j < NQ; j++) xv[j] = quad(j);
    if (tid < 32) etab[tid] = IT_EXP2F_TAB[tid];
    auto put = [&](int j, float4 v) __attribute__((always_inline)) {
        const int i = 4 * (tid + 256 * j);
        uint32_t packed;
        float d;
        quantize_quad(v, &packed, &d);
        if (i < n_in) {
            *(uint32_t*)(xq + i) = packed;
            if ((tid & 7) == 0) xs[i >> 5] = d;
        }
    };
    if constexpr (ROUTE) {
        static_assert(NQ == 1, "a quad a thread");
        __shared__ double red[4];
        __shared__ int ids[64];
        __shared__ float wts[64], logits[64];
        const int i = 4 * tid, rows = p.n_expert + 1, items = rows * nb, ts = nb + 4;
        const bool first = blockIdx.x == 0 && y == 0;
        const float4 wv = i < n_in ? load4(p.norm_w + i) : make_float4(0.f, 0.f, 0.f, 0.f);
        // the rows' 32-value units over the threads: the router's, then the shared gate's
        const float inv = inv_of(nb);
        uint4 wa[ROUTE_ITEMS], wb[ROUTE_ITEMS];
        uint16_t sc[ROUTE_ITEMS];
#pragma unroll
        for (int k = 0; k < ROUTE_ITEMS; k++) {
            const int it = tid + 256 * k;
            if (256 * k >= items) break;
            if (it >= items) continue;
            const bool gate = it >= items - nb;
            const int at = gate ? it - (items - nb) : it;
            const uint4* q = (const uint4*)((gate ? p.sg_q : p.rt_q) + (int64_t)at * 32);
            wa[k] = q[0];
            wb[k] = q[1];
            sc[k] = ((const uint16_t*)(gate ? p.sg_s : p.rt_s))[at];
        }
        float* xf = terms_all;                   // for the serial sum, should it be needed
        if (i < n_in) *(float4*)(xf + i) = xv[0];
        double part = (double)(xv[0].x * xv[0].x);
        part += (double)(xv[0].y * xv[0].y);
        part += (double)(xv[0].z * xv[0].z);
        part += (double)(xv[0].w * xv[0].w);
        part = wave_sum_f64_tail(part);
        if (lane == 63) red[wave] = part;
        __syncthreads();
        float mean;
        if (!mean_is_certain(red[0] + red[1] + red[2] + red[3], n_in, n_in, &mean)) {   // (the same answer in every thread)
            double sum = 0.0;
            for (int n = 0; n < n_in; n++) sum += (double)(xf[n] * xf[n]);
            mean = (float)over(sum, n_in);
        }
        const float scale = 1.0f / sqrtf(mean + p.eps);
        xv[0].x = xv[0].x * scale * wv.x;
        xv[0].y = xv[0].y * scale * wv.y;
        xv[0].z = xv[0].z * scale * wv.z;
        xv[0].w = xv[0].w * scale * wv.w;
        if (first && i < n_in) {
            store4(p.normed + i, xv[0]);
            store4(p.normed2 + i, xv[0]);
        }
        put(0, xv[0]);
        __syncthreads();
        if (!shared) {
#pragma unroll
            for (int k = 0; k < ROUTE_ITEMS; k++) {
                const int it = tid + 256 * k;
                if (256 * k >= items) break;
                if (it >= items) continue;
                const int r = row_of(it, inv), u = it - r * nb;
                const uint4* ap = (const uint4*)(xq + u * 32);
                terms_all[r * ts + u] = unit_q8_0(wa[k], wb[k], sc[k], ap[0], ap[1], xs[u]);
            }
            __syncthreads();
            if (wave == 0) {
                if (lane < rows) {
                    const float dot = fold_terms(terms_all + lane * ts, nb);
                    logits[lane] = dot;
                    if (first) *(lane < p.n_expert ? p.logits_out + lane : p.sg_out) = dot;
                }
                wave_lds_sync();
                wave_route(logits, p.n_expert, p.n_used, ids, wts, lane, etab);
                if (first && lane < p.n_used) {
                    p.route_ids_out[lane] = ids[lane];
                    p.route_w_out[lane] = wts[lane];
                }
            }
            __syncthreads();
            e = ids[y];
        }
    }
    const int fmt = shared ? p.sh_fmt : p.fmt;
    const uint8_t* gq = shared ? p.sh_gq : p.gq + e * p.q_stride;
    const uint8_t* gs = shared ? p.sh_gs : p.gs + e * p.s_stride;
    const uint8_t* uq = shared ? p.sh_uq : p.uq + e * p.q_stride;
    const uint8_t* us = shared ? p.sh_us : p.us + e * p.s_stride;
    const int n_out = shared ? p.sh_n_out : p.n_out;
    float* out = shared ? p.sh_out : p.out + (int64_t)y * p.n_out;

    const int R = p.rows_per_wave;
    const int tstride = nb * 2 + 4;
    float* tg = terms_all + (size_t)wave * 2 * R * tstride;
    float* tu = tg + (size_t)R * tstride;
    const int T = fmt == W_NVFP4 ? nb * 2 : nb;
    const int groups = (n_out + R - 1) / R;
    // first group's gate and up rows start moving before the activation is quantized
    const int g0 = blockIdx.x * 4 + wave;
    const bool has0 = g0 < groups;
    const int row00 = g0 * R, nrows0 = has0 ? min(R, n_out - row00) : 0;
    RowRegs<4> rg, ru;
    if (has0) {
        if (fmt == W_NVFP4) {
            load_items<W_NVFP4, 4>(rg, gq, gs, n_in, row00, nrows0, lane);
            load_items<W_NVFP4, 4>(ru, uq, us, n_in, row00, nrows0, lane);
        } else {
            load_items<W_Q8_0, 4>(rg, gq, gs, n_in, row00, nrows0, lane);
            load_items<W_Q8_0, 4>(ru, uq, us, n_in, row00, nrows0, lane);
        }
    }
    // (a scale of 1, where there is no scale tensor, leaves the bits as they are)
    const float gsc = shared ? p.sh_gscale : p.gscale2 ? p.gscale2[e] : 1.0f, usc = shared ? p.sh_uscale : p.uscale2 ? p.uscale2[e] : 1.0f;
    if constexpr (!ROUTE) {
#pragma unroll
        for (int j = 0; j < NQ; j++) put(j, xv[j]);
        if (NQ == 0)
            for (int j = 0; 1024 * j < n_in; j++) put(j, quad(j));
        __syncthreads();
    }
    for (int g = g0; g < groups; g += gridDim.x * 4) {
        const int row0 = g * R, nrows = min(R, n_out - row0);
        if (g != g0) {
            if (fmt == W_NVFP4) {
                load_items<W_NVFP4, 4>(rg, gq, gs, n_in, row0, nrows, lane);
                load_items<W_NVFP4, 4>(ru, uq, us, n_in, row0, nrows, lane);
            } else {
                load_items<W_Q8_0, 4>(rg, gq, gs, n_in, row0, nrows, lane);
                load_items<W_Q8_0, 4>(ru, uq, us, n_in, row0, nrows, lane);
            }
        }
        if (fmt == W_NVFP4) {
            compute_items<W_NVFP4, 4>(rg, n_in, nrows, xq, xs, tg, tstride, lane);
            compute_items<W_NVFP4, 4>(ru, n_in, nrows, xq, xs, tu, tstride, lane);
        } else {
            compute_items<W_Q8_0, 4>(rg, n_in, nrows, xq, xs, tg, tstride, lane);
            compute_items<W_Q8_0, 4>(ru, n_in, nrows, xq, xs, tu, tstride, lane);
        }
        wave_lds_sync();
        // lanes 0 .. 31 fold gate rows, 32 .. 63 up rows: the two chains side by side
        const int half = lane >> 5, r = lane & 31;
        float acc = 0.0f;
        if (r < nrows) acc = fold_terms((half ? tu : tg) + r * tstride, T);
        acc *= half ? usc : gsc;
        const float up = __shfl_xor(acc, 32, 64);
        if (lane < nrows) out[row0 + lane] = it_silu_by(acc, etab) * up;
        wave_lds_sync();
    }
}

// rows of a wave, blocks of a pick and the LDS of a block
struct GluShape {
    int rows, blocks;
    size_t lds;
};
static GluShape glu_shape(const MoeGluP& p) {
    const int nb = p.n_in / 32;
    int R = 4;
    while (R > 1 && R * nb > 256) R /= 2;
    auto lds_for = [&](int r) {
        return (size_t)((nb + 3) & ~3) * 4 + p.n_in + (size_t)4 * 2 * r * (nb * 2 + 4) * 4;
    };
    while (R > 1 && lds_for(R) > 60 * 1024) R /= 2;
    const int n_out = std::max(p.n_out, p.sh_n_out);
    // (a router in front: its rows' terms, and before them the activation, in the terms' place)
    const size_t route = p.norm_w ? (size_t)((nb + 3) & ~3) * 4 + p.n_in + std::max((size_t)p.n_in, (size_t)(p.n_expert + 1) * (nb + 4)) * 4 : 0;
    return {R, std::max(1, (n_out + 4 * R - 1) / (4 * R)), std::max(lds_for(R), route)};   // one row group per wave
}

void moe_glu_fused(MoeGluP p, hipStream_t s) {
    if (moe_glu_fast(p, s)) return;
    const GluShape sh = glu_shape(p);
    p.rows_per_wave = sh.rows;
    const dim3 grid(sh.blocks, p.n_used + 1);
    if (p.norm_w) hipLaunchKernelGGL((moe_glu_fused_k<1, true>), grid, dim3(256), sh.lds, s, p);
    else if (p.n_in <= 1024) hipLaunchKernelGGL((moe_glu_fused_k<1, false>), grid, dim3(256), sh.lds, s, p);
    else if (p.n_in <= 2048) hipLaunchKernelGGL((moe_glu_fused_k<2, false>), grid, dim3(256), sh.lds, s, p);
    else if (p.n_in <= 4096) hipLaunchKernelGGL((moe_glu_fused_k<4, false>), grid, dim3(256), sh.lds, s, p);
    else hipLaunchKernelGGL((moe_glu_fused_k<0, false>), grid, dim3(256), sh.lds, s, p);
}

// Taken while a thread holds the router's units (four: rows * n_in / 32 <= 1,024) beside one quad of the activation, a wave
// folds the rows side by side, and the blocks, which all repeat it, have a CU each.
bool moe_route_glu(const FusedGemvP& a, MoeGluP* g) {
    const int nb = g->n_in / 32, rows = g->n_expert + 1;
    if (!a.exact || !g->exact || a.mode != 1 || a.n_mats != 2 || a.n_in != g->n_in || g->n_in > 1024 || g->n_in % 32 || g->n_tok > 1) return false;
    for (int k = 0; k < 2; k++)
        if (a.m[k].fmt != W_Q8_0 || a.m[k].epi != 0 || (reinterpret_cast<uintptr_t>(a.m[k].q) & 15)) return false;
    if (a.m[0].n_out != g->n_expert || a.m[1].n_out != 1 || rows > 64 || rows * nb > 256 * ROUTE_ITEMS || g->n_used > 64) return false;
    if (a.x == a.x_copy || a.x == a.x_copy2) return false;   // (blocks read it while one writes)
    MoeGluP p = *g;
    p.x = a.x;
    p.norm_w = a.norm_w;
    p.eps = a.eps;
    p.rt_q = a.m[0].q;
    p.rt_s = a.m[0].s;
    p.sg_q = a.m[1].q;
    p.sg_s = a.m[1].s;
    p.normed = a.x_copy;
    p.normed2 = a.x_copy2;
    p.logits_out = a.m[0].out;
    p.sg_out = a.m[1].out;
    p.route_ids_out = a.route_ids;
    p.route_w_out = a.route_w;
    const GluShape sh = glu_shape(p);
    if (sh.blocks * (p.n_used + 1) > 256 || sh.lds > 64 * 1024) return false;
    *g = p;
    return true;
}

// ------------------------------------------------------------------ moe_down_fused
// x[j] += sum_e w_e * (down_e[j] . g_e * scale2_e) + (shared_down[j] . g_sh) * sigmoid(logit)
// (src/ops/mod.rs:1134-1171 then add_assign), experts ascending, shared last.
// What bounds it and how it is laid out: as fused_gemv_k.  What a row's end needs (the picks' scales and weights, the gate's
// logit, the residual stream) is asked for at the start.
constexpr int DOWN_LDS_MAX = 159 * 1024, DOWN_ITEMS = 8, DOWN_QUADS = 6;   // (quads: of the intermediates, in a thread's registers; longer ones are staged in LDS)
__global__ __launch_bounds__(256) void moe_down_fused_k(MoeDownP p) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ uint64_t etab[32];
    const int n_in = p.n_in, nb = n_in >> 5;       // expert down: n_in = expert_ff
    const int sh_in = p.sh_n_in, sh_nb = sh_in >> 5;
    const int NU = p.n_used;
    // LDS: per pick quantized activation, then the shared one
    float* xs = (float*)smem;                                     // NU*nb + sh_nb scales
    int8_t* xq = (int8_t*)(xs + ((NU * nb + sh_nb + 3) & ~3));    // NU*n_in + sh_in quants
    float* terms_all = (float*)(xq + ((NU * n_in + sh_in + 15) & ~15));
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int my_id = p.route_ids[lane < NU ? lane : 0];   // every pick in one load
    const float my_w = p.route_w[lane < NU ? lane : 0];
    const int total = NU * n_in + sh_in;                   // the intermediates: the picks' and the shared one's, 32-aligned
    const bool by_regs = total <= 4 * 256 * DOWN_QUADS;
    float4 xv[DOWN_QUADS];
    if (by_regs) {
#pragma unroll
        for (int j = 0; j < DOWN_QUADS; j++) {
            const int i = 4 * (tid + 256 * j);
            xv[j] = i < NU * n_in ? load4(p.g_all + i) : i < total ? load4(p.g_shared + (i - NU * n_in)) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    }
    const float logit = p.logit[0];
    if (tid < 32) etab[tid] = IT_EXP2F_TAB[tid];
    it_count_expert_reads(p.route_ids, NU, p.counts_gate, p.counts_up, p.counts_down, p.tally);
    const int R = p.rows_per_wave;
    const int T = p.fmt == W_NVFP4 ? nb * 2 : nb;
    const int shT = p.sh_fmt == W_NVFP4 ? sh_nb * 2 : sh_nb;
    const int Tmax = (T > shT ? T : shT);
    const int tstride = Tmax + 4;
    // terms[(y * R + r) * tstride + k]
    float* terms = terms_all + (size_t)wave * (NU + 1) * R * tstride;
    const int groups = (p.n_out + R - 1) / R;
    // A wave's (pick, row, 32-element unit) items are dealt out over its lanes without a gap, 64 * DOWN_ITEMS of them (all of
    // a group's, for what the launcher sizes it for) in flight at once.
    RowRegs<DOWN_ITEMS> rr;
    RowRegs<1> rsh;
    auto load_all = [&](int row0, int nrows, int i0) __attribute__((always_inline)) {
        const int per = nrows * nb;
        const float inv_per = inv_of(per), inv_nb = inv_of(nb);
#pragma unroll
        for (int k = 0; k < DOWN_ITEMS; k++) {
            if (i0 + k * 64 >= NU * per) break;
            const int it = min(i0 + k * 64 + lane, NU * per - 1), y = row_of(it, inv_per), ru = it - y * per, r = row_of(ru, inv_nb), u = ru - r * nb;
            const int64_t e = __shfl(my_id, y, 64);
            const int64_t row = row0 + r;
            const uint8_t *q = p.q + e * p.q_stride, *sc = p.s + e * p.s_stride;
            if (p.fmt == W_NVFP4) {
                rr.wa[k] = *(const uint4*)(q + row * (n_in >> 1) + u * 16);
            } else {
                const uint4* wp = (const uint4*)(q + row * n_in + u * 32);
                rr.wa[k] = wp[0];
                rr.wb[k] = wp[1];
            }
            rr.sc[k] = ((const uint16_t*)sc)[row * nb + u];
        }
    };
    auto load_shared = [&](int row0, int nrows) __attribute__((always_inline)) {
        if (p.sh_fmt == W_NVFP4) load_items<W_NVFP4, 1>(rsh, p.sh_q, p.sh_s, sh_in, row0, nrows, lane);
        else load_items<W_Q8_0, 1>(rsh, p.sh_q, p.sh_s, sh_in, row0, nrows, lane);
    };
    const int g0 = blockIdx.x * 4 + wave;
    // lane (y, r) of a group: its pick's second scale and weight; lane r: the row's value so far
    float sc2 = 1.0f, x_old = 0.0f;
    auto ask_end = [&](int row0, int nrows) __attribute__((always_inline)) {
        const int y = row_of(lane, inv_of(nrows));
        const int id = __shfl(my_id, min(y, NU - 1), 64);
        sc2 = y >= NU ? p.sh_dscale : p.scale2 ? p.scale2[id] : 1.0f;
        x_old = lane < nrows ? p.x[row0 + lane] : 0.0f;
    };
    if (g0 < groups) {
        const int nrows = min(R, p.n_out - g0 * R);
        load_all(g0 * R, nrows, 0);
        load_shared(g0 * R, nrows);
        ask_end(g0 * R, nrows);
    }
    if (by_regs) {
#pragma unroll
        for (int j = 0; j < DOWN_QUADS; j++) {
            if (1024 * j >= total) break;
            const int i = 4 * (tid + 256 * j);
            uint32_t packed;
            float d;
            quantize_quad(xv[j], &packed, &d);
            if (i < total) {
                *(uint32_t*)(xq + i) = packed;
                if ((tid & 7) == 0) xs[i >> 5] = d;
            }
        }
    } else {
        // stage all NU + 1 intermediates as f32 (the term region is free until the main loop)
        float* all = terms_all;
        for (int i = tid; i < total; i += 256) all[i] = i < NU * n_in ? p.g_all[i] : p.g_shared[i - NU * n_in];
        __syncthreads();
        // one Q8_0 block per 8 lanes; picks and the shared vector are back to back and 32-aligned
        lds_quantize_q8_0(all, total, xs, xq);
    }
    __syncthreads();
    const float gate = it_sigmoid_by(logit, etab);
    for (int g = g0; g < groups; g += gridDim.x * 4) {
        const int row0 = g * R, nrows = min(R, p.n_out - row0);
        if (g != g0) {
            load_shared(row0, nrows);
            ask_end(row0, nrows);
        }
        const int per = nrows * nb;
        const float inv_per = inv_of(per), inv_nb = inv_of(nb), inv_rows = inv_of(nrows);
        for (int i0 = 0; i0 < NU * per; i0 += 64 * DOWN_ITEMS) {
            if (g != g0 || i0) load_all(row0, nrows, i0);
#pragma unroll
            for (int k = 0; k < DOWN_ITEMS; k++) {
                if (i0 + k * 64 >= NU * per) break;
                const int it = i0 + k * 64 + lane, y = row_of(it, inv_per), ru = it - y * per, r = row_of(ru, inv_nb), u = ru - r * nb;
                if (it >= NU * per) continue;
                const uint4* ap = (const uint4*)(xq + y * n_in + u * 32);
                const uint4 a0 = ap[0], a1 = ap[1];
                const float dx = xs[y * nb + u];
                float* t = terms + ((size_t)y * R + r) * tstride;
                if (p.fmt == W_Q8_0) {
                    t[u] = unit_q8_0(rr.wa[k], rr.wb[k], (uint16_t)rr.sc[k], a0, a1, dx);
                } else {
                    float tA, tB;
                    unit_nvfp4(rr.wa[k], rr.sc[k], a0, a1, dx, &tA, &tB);
                    t[2 * u] = tA;
                    t[2 * u + 1] = tB;
                }
            }
        }
        {
            float* t = terms + (size_t)NU * R * tstride;
            if (p.sh_fmt == W_NVFP4) compute_items<W_NVFP4, 1>(rsh, sh_in, nrows, xq + NU * n_in, xs + NU * nb, t, tstride, lane);
            else compute_items<W_Q8_0, 1>(rsh, sh_in, nrows, xq + NU * n_in, xs + NU * nb, t, tstride, lane);
        }
        wave_lds_sync();
        // lane = (y, r): fold its dot; lane r adds them up, the picks in order, the shared expert last
        float dot = 0.0f;
        const int pairs = (NU + 1) * nrows;
        const int y = row_of(lane, inv_rows), r = lane - y * nrows;
        if (lane < pairs) dot = fold_terms(terms + ((size_t)y * R + r) * tstride, y < NU ? T : shT) * sc2;
        const float w = __shfl(my_w, min(y, NU - 1), 64);
        dot = y < NU ? w * dot : dot * gate;
        float v = 0.0f;
#pragma unroll 4
        for (int k = 0; k <= NU; k++) v += __shfl(dot, min(k * nrows + lane, 63), 64);
        if (lane < nrows) p.x[row0 + lane] = x_old + v;
        wave_lds_sync();
    }
}

// LDS of a block: the picks' and the shared intermediate's scales and quants, and the terms of r rows a wave (f32 staging shares their place)
static size_t down_lds(const MoeDownP& p, int r) {
    const int nb = p.n_in / 32, sh_nb = p.sh_n_in / 32;
    const int T = std::max(p.fmt == W_NVFP4 ? nb * 2 : nb, p.sh_fmt == W_NVFP4 ? sh_nb * 2 : sh_nb);
    const size_t total = (size_t)p.n_used * p.n_in + p.sh_n_in;
    return (size_t)((p.n_used * nb + sh_nb + 3) & ~3) * 4 + ((total + 15) & ~(size_t)15) + std::max((size_t)4 * (p.n_used + 1) * r * (T + 4) * 4, total * 4);
}

void moe_down_fused(MoeDownP p, hipStream_t s) {
    if (!p.exact && moe_down_fast(p, s)) return;
    const int nb = p.n_in / 32, sh_nb = p.sh_n_in / 32;
    // a row group per wave over the whole chip (256 blocks of four waves), and what the kernel's registers hold
    int R = 4;
    while (R > 1 && ((p.n_used + 1) * R > 64 || R * sh_nb > 64 || p.n_used * R * nb > 64 * DOWN_ITEMS || (p.n_out + R - 1) / R < 1024)) R /= 2;
    while (R > 1 && down_lds(p, R) > 60 * 1024) R /= 2;
    p.rows_per_wave = R;
    int groups = (p.n_out + R - 1) / R;
    int blocks = (groups + 3) / 4;
    if (blocks > 512) blocks = 512;
    (void)lds_allowed<&moe_down_fused_k>(DOWN_LDS_MAX);   // (refused: the launch reports it)
    hipLaunchKernelGGL(moe_down_fused_k, dim3(blocks), dim3(256), down_lds(p, R), s, p);
}

// The kernels that keep the CPU path's order take 256 units of a gate / up row and 64 of the shared down row at once, and
// intermediates that fit LDS.  In fast mode the picks are made by the fast gate / up kernel, so there is no other.
bool moe_fused_takes(const MoeGluP& g, const MoeDownP& d) {
    if (g.exact ? g.n_in > 4 * 64 * 32 : !moe_glu_fast(g, nullptr, true)) return false;
    return (!d.exact && moe_down_fast(d, nullptr, true)) || (d.sh_n_in <= 64 * 32 && down_lds(d, 1) <= DOWN_LDS_MAX);
}

// ------------------------------------------------------------------ attention prep
// One block per head: query heads take q out of the interleaved [q | gate] projection,
// rms_norm_heads, rope; key heads the same and write f16 into the K slab at `pos`;
// value heads write f16 into the V slab.
__global__ __launch_bounds__(64) void attn_prep_k(AttnPrepP p) {
    extern __shared__ float hbuf[];
    __shared__ double red[2];
    const int hd = p.head_dim, tid = threadIdx.x;
    const int pos = *p.pos_dyn;
    int b = blockIdx.x;
    if (b >= p.n_head + p.n_head_kv) {  // value head
        const int h = b - p.n_head - p.n_head_kv;
        uint16_t* dst = p.v_slab + (int64_t)pos * p.kv_dim + h * hd;
        for (int i = tid; i < hd; i += 64) dst[i] = it_f32_to_f16(p.v[h * hd + i]);
        return;
    }
    const bool is_q = b < p.n_head;
    const int h = is_q ? b : b - p.n_head;
    const float* src = is_q ? p.qg + (int64_t)h * 2 * hd : p.k + (int64_t)h * hd;
    const float* w = is_q ? p.q_norm : p.k_norm;
    for (int i = tid; i < hd; i += 64) hbuf[i] = src[i];
    __syncthreads();
    float scale = 1.0f / sqrtf(block_meansq<64>(hbuf, hd, hd, p.exact, red) + p.eps);
    __syncthreads();
    for (int i = tid; i < hd; i += 64) hbuf[i] = hbuf[i] * scale * w[i];
    __syncthreads();
    const int half = p.n_rot / 2;
    for (int i = tid; i < half; i += 64) {
        float2 cs = p.rope[(int64_t)pos * half + i];
        float x0 = hbuf[i], x1 = hbuf[i + half];
        hbuf[i] = x0 * cs.x - x1 * cs.y;
        hbuf[i + half] = x0 * cs.y + x1 * cs.x;
    }
    __syncthreads();
    if (is_q) {
        for (int i = tid; i < hd; i += 64) p.q[h * hd + i] = hbuf[i];
    } else {
        uint16_t* dst = p.k_slab + (int64_t)pos * p.kv_dim + h * hd;
        for (int i = tid; i < hd; i += 64) dst[i] = it_f32_to_f16(hbuf[i]);
    }
}

void attn_prep(const AttnPrepP& p, hipStream_t s) {
    hipLaunchKernelGGL(attn_prep_k, dim3(p.n_head + 2 * p.n_head_kv), dim3(64), p.head_dim * sizeof(float), s, p);
}

}  // namespace itk
