// GQA attention over the f16 KV slabs.
//
// attend_exact keeps the reference CPU path's order (/root/reference
// src/ops/naive.rs:420-466): score = (serial dot) * scale; softmax with a serial
// sum; the weighted V sum walks positions outermost.  Bit-identical to the CPU.
//
// attend_split is split-K flash decoding: each block owns one kv head (all of its
// query heads share the K/V stream) and one range of positions, keeps an
// online-softmax partial (acc, m, l), and a second kernel merges the partials.
// Up to 16 queries take the f16 matrix-core kernel (k_attn_decode.hip), larger
// batches that the one-pass prefill kernel does not take a position-per-thread
// kernel over 128-position chunks.  Reordered sums: compared against the exact
// path at 1e-3.
#include <algorithm>
#include "it_device.h"
#include "it_dot.h"
#include "it_reduce.h"
#include "kernels.h"
#include "kernels_fused.h"

namespace itk {

// ------------------------------------------------------------------ exact
// One block per (query, head).  Scores and weights sit in LDS up to EXACT_LDS positions (beyond, in `scratch`).  What has an
// order is a chain: a position's dot in its thread, the weights' sum in one lane, a dim's weighted sum in its thread, each
// with its loads several steps ahead.  333 positions, 16 heads of 256: 28 us (115 with every read waited for
// and the weight divided anew for every dim).
// PREP (one query): the block forms its query head and the new position's key and value from the projections, a wave each, and
// keeps those in LDS; the first head of a KV head leaves them in the slabs, which no block reads at that position.  As a launch
// in front (attn_prep) that took 4.6 us, 2.5 of them its start and the projections' trip.  A token of four layers of 512 values,
// 117.4 -> 115.4 us.
constexpr int EXACT_LDS = 4096;
// head_norm and rotation of one head of `hd` values by one wave, in place in LDS, as attn_prep_k.  The first 256 values' weights
// and rotations are asked for with the values (a trip to L2 each otherwise).
IT_DEV void wave_norm_rope(float* h, const float* __restrict__ src, const float* __restrict__ w, int hd, const AttnPrepP& p, int pos, int lane) {
    constexpr int AHEAD = 4;
    const int half = p.n_rot / 2;
    const float2* const rope = p.rope + (int64_t)pos * half;
    float x[AHEAD], wx[AHEAD];
    float2 cs[AHEAD / 2];
#pragma unroll
    for (int k = 0; k < AHEAD; k++) {
        const int i = lane + 64 * k;
        x[k] = i < hd ? src[i] : 0.0f;
        wx[k] = i < hd ? w[i] : 0.0f;
        if (k < AHEAD / 2) cs[k] = i < half ? rope[i] : make_float2(1.0f, 0.0f);
    }
    double part = 0.0;
#pragma unroll
    for (int k = 0; k < AHEAD; k++) {
        if (lane + 64 * k < hd) h[lane + 64 * k] = x[k];
        part += (double)(x[k] * x[k]);
    }
    for (int i = lane + 64 * AHEAD; i < hd; i += 64) {
        const float v = src[i];
        h[i] = v;
        part += (double)(v * v);
    }
    const double sum = __shfl(wave_sum_f64_tail(part), 63, 64);
    wave_lds_sync();
    float mean;
    if (!mean_is_certain(sum, hd, hd, &mean)) {   // (the same answer in every lane)
        double serial = 0.0;
        for (int i = 0; i < hd; i++) serial += (double)(h[i] * h[i]);
        mean = (float)over(serial, hd);
    }
    const float scale = 1.0f / sqrtf(mean + p.eps);
    wave_lds_sync();
#pragma unroll
    for (int k = 0; k < AHEAD; k++)
        if (lane + 64 * k < hd) h[lane + 64 * k] = x[k] * scale * wx[k];
    for (int i = lane + 64 * AHEAD; i < hd; i += 64) h[i] = h[i] * scale * w[i];
    wave_lds_sync();
    auto turn = [&](int i, float2 r) __attribute__((always_inline)) {
        const float x0 = h[i], x1 = h[i + half];
        h[i] = x0 * r.x - x1 * r.y;
        h[i + half] = x0 * r.y + x1 * r.x;
    };
#pragma unroll
    for (int k = 0; k < AHEAD / 2; k++)
        if (lane + 64 * k < half) turn(lane + 64 * k, cs[k]);
    for (int i = lane + 32 * AHEAD; i < half; i += 64) turn(i, rope[i]);
    wave_lds_sync();
}
template <bool PREP>
__global__ __launch_bounds__(1024) void attend_exact_k(AttnArgs a, AttnPrepP pr, float* __restrict__ scratch, float* __restrict__ out,
                                                      const float* __restrict__ gate, int gate_stride, int lds_pos) {
    extern __shared__ __align__(16) float qs[];  // head_dim, then the first lds_pos scores (a multiple of 4 each), then PREP's key and value
    __shared__ float red[17];
    __shared__ uint64_t etab[32];   // (a lookup in constant memory is a trip to L2)
    const int hd = a.head_dim, tid = threadIdx.x, nt = blockDim.x;
    if (tid < 32) etab[tid] = IT_EXP2F_TAB[tid];
    const int n_pos_last = a.n_pos_dyn ? *a.n_pos_dyn : a.n_pos;
    const int t = blockIdx.x / a.n_head, h = blockIdx.x % a.n_head;
    const int group = a.n_head / a.n_head_kv;
    const int h_kv = h / group;
    const int n_pos = n_pos_last - a.n_q + 1 + t, n_lds = min(n_pos, lds_pos);
    const int off = h_kv * hd;
    const float* q = a.q + ((int64_t)t * a.n_head + h) * hd;
    float* near = qs + ((hd + 3) & ~3);
    float* far = scratch + (int64_t)blockIdx.x * n_pos_last;
    auto score = [&](int s) -> float& { return s < lds_pos ? near[s] : far[s]; };
    const int n_slab = PREP ? n_pos - 1 : n_pos;   // positions read from the slabs
    float* const fresh = near + lds_pos;           // the new position's key, then its value
    if constexpr (PREP) {
        const int wave = tid >> 6, lane = tid & 63, pos = n_pos - 1;
        const bool leaves = h % group == 0;
        if (wave == 0) {
            wave_norm_rope(qs, pr.qg + (int64_t)h * 2 * hd, pr.q_norm, hd, pr, pos, lane);
            for (int i = lane; i < hd; i += 64) pr.q[(int64_t)h * hd + i] = qs[i];
        } else if (wave == 1) {
            wave_norm_rope(fresh, pr.k + off, pr.k_norm, hd, pr, pos, lane);
            for (int i = lane; i < hd; i += 64) {
                const uint16_t v = it_f32_to_f16(fresh[i]);
                fresh[i] = it_f16_to_f32(v);
                if (leaves) pr.k_slab[(int64_t)pos * a.kv_dim + off + i] = v;
            }
        } else if (wave == 2) {
            for (int i = lane; i < hd; i += 64) {
                const uint16_t v = it_f32_to_f16(pr.v[off + i]);
                fresh[hd + i] = it_f16_to_f32(v);
                if (leaves) pr.v_slab[(int64_t)pos * a.kv_dim + off + i] = v;
            }
        }
    } else {
        for (int i = tid; i < hd; i += nt) qs[i] = q[i];
    }
    __syncthreads();
    float m = -INFINITY;
    if (PREP && tid == nt - 1) {                   // (of the wave with the fewest positions of its own)
        float dot = 0.0f;
#pragma unroll 8
        for (int i = 0; i < hd; i++) dot += qs[i] * fresh[i];
        m = dot * a.scale;
        score(n_slab) = m;
    }
    for (int s = tid; s < n_slab; s += nt) {
        const uint16_t* key = a.k + (int64_t)s * a.kv_dim + off;
        float dot = 0.0f;
        auto add8 = [&](int i, uint4 kk) {
            const uint32_t w[4] = {kk.x, kk.y, kk.z, kk.w};
#pragma unroll
            for (int c = 0; c < 4; c++) {
                dot += qs[i + 2 * c] * it_f16_to_f32((uint16_t)(w[c] & 0xffff));
                dot += qs[i + 2 * c + 1] * it_f16_to_f32((uint16_t)(w[c] >> 16));
            }
        };
        int i = 0;
        if (hd >= 64) {   // 64 dims at a time, the next 64 on their way
            uint4 nx[8];
#pragma unroll
            for (int p = 0; p < 8; p++) nx[p] = *(const uint4*)(key + 8 * p);
            for (; i + 64 <= hd; i += 64) {
                uint4 cur[8];
#pragma unroll
                for (int p = 0; p < 8; p++) cur[p] = nx[p];
                const int n = i + 128 <= hd ? i + 64 : i;
#pragma unroll
                for (int p = 0; p < 8; p++) nx[p] = *(const uint4*)(key + n + 8 * p);
#pragma unroll
                for (int p = 0; p < 8; p++) add8(i + 8 * p, cur[p]);
            }
        }
        for (; i < hd; i += 8) add8(i, *(const uint4*)(key + i));
        const float v = dot * a.scale;
        score(s) = v;
        m = fmaxf(m, v);
    }
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_down(m, o, 64));
    if ((tid & 63) == 0) red[tid >> 6] = m;
    __syncthreads();
    m = red[0];
    for (int w = 1; w < nt / 64; w++) m = fmaxf(m, red[w]);
    for (int s = tid; s < n_pos; s += nt) score(s) = it_expf_by(score(s) - m, etab);
    __threadfence_block();
    __syncthreads();
    if (tid < 64) {   // (every lane: reads of one address by all cost less than by one lane)
        float sum = fold_terms(near, n_lds);
#pragma unroll 16
        for (int s = lds_pos; s < n_pos; s++) sum += far[s];
        red[16] = sum;
    }
    __syncthreads();
    const float sum = red[16];
    for (int s = tid; s < n_pos; s += nt) score(s) = score(s) / sum;
    __threadfence_block();
    __syncthreads();
    for (int i = tid; i < hd; i += nt) {
        const uint16_t* v = a.v + off + i;
        float acc = 0.0f;
        int s = 0;
        const int n_near = min(n_slab, lds_pos);
        constexpr int AHEAD = 32;   // positions whose values are on their way while as many are added
        uint16_t x0[AHEAD], x1[AHEAD];
        auto ask = [&](uint16_t (&x)[AHEAD], int from) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < AHEAD; c++) x[c] = v[(int64_t)min(from + c, n_slab - 1) * a.kv_dim];
        };
        auto add = [&](const uint16_t (&x)[AHEAD], int from) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < AHEAD; c++) acc += near[from + c] * it_f16_to_f32(x[c]);
        };
        if (n_near >= AHEAD) ask(x0, 0);
        for (; s + 2 * AHEAD <= n_near; s += 2 * AHEAD) {
            ask(x1, s + AHEAD);
            add(x0, s);
            ask(x0, s + 2 * AHEAD);
            add(x1, s + AHEAD);
        }
        if (s + AHEAD <= n_near) {
            add(x0, s);
            s += AHEAD;
        }
        for (; s < n_near; s++) acc += near[s] * it_f16_to_f32(v[(int64_t)s * a.kv_dim]);
#pragma unroll 8
        for (s = lds_pos; s < n_slab; s++) acc += far[s] * it_f16_to_f32(v[(int64_t)s * a.kv_dim]);
        if (PREP) acc += score(n_slab) * fresh[hd + i];
        if (gate) acc *= it_sigmoid(gate[(int64_t)h * gate_stride + i]);   // (n_q == 1: sigmoid_mul of the gated block)
        out[((int64_t)t * a.n_head + h) * hd + i] = acc;
    }
}

void attend_exact(const AttnArgs& a, float* scratch, float* out, hipStream_t s, const float* gate, int gate_stride, const AttnPrepP* prep) {
    if (a.n_q <= 0) return;
    const int lds_pos = std::min((a.n_pos + 3) & ~3, EXACT_LDS);
    // few blocks: a thread per position while the score phase has that many; many: blocks that share a CU
    const int threads = a.n_q * a.n_head < 512 && a.n_pos > 256 ? 1024 : 256;
    const size_t lds = ((size_t)((a.head_dim + 3) & ~3) + lds_pos + (prep ? 2 * a.head_dim : 0)) * sizeof(float);
    const dim3 grid(a.n_q * a.n_head), block(threads);
    if (prep) hipLaunchKernelGGL(attend_exact_k<true>, grid, block, lds, s, a, *prep, scratch, out, gate, gate_stride, lds_pos);
    else hipLaunchKernelGGL(attend_exact_k<false>, grid, block, lds, s, a, AttnPrepP{}, scratch, out, gate, gate_stride, lds_pos);
}

// ------------------------------------------------------------------ split-K
constexpr int CHUNK = 128;


// partial layout per (t, head, split): [hd acc][m][l]
template <int G>
__global__ __launch_bounds__(256) void attend_split_k(AttnArgs a, int n_split, float* __restrict__ part) {
    extern __shared__ float lds[];
    const int hd = a.head_dim;
    float* qs = lds;                 // [G][hd]
    float* sc = lds + G * hd;        // [CHUNK][G]
    __shared__ float mrow[G], lrow[G];
    const int n_pos_last = a.n_pos_dyn ? *a.n_pos_dyn : a.n_pos;
    const int t = blockIdx.x / a.n_head_kv, h_kv = blockIdx.x % a.n_head_kv;
    const int split = blockIdx.y;
    const int n_pos = n_pos_last - a.n_q + 1 + t;
    const int s0 = split * CHUNK;
    const int len = min(CHUNK, n_pos - s0);
    const int off = h_kv * hd;
    const int h0 = h_kv * G;
    float* my_part = part + (((int64_t)t * a.n_head + h0) * n_split + split) * (hd + 2);
    const int64_t part_head_stride = (int64_t)n_split * (hd + 2);
    if (len <= 0) {
        // empty chunk: m = -inf, l = 0 marks it for the merge
        if (threadIdx.x < G) {
            float* p = my_part + threadIdx.x * part_head_stride;
            p[hd] = -INFINITY;
            p[hd + 1] = 0.0f;
        }
        return;
    }
    for (int i = threadIdx.x; i < G * hd; i += 256) qs[i] = a.q[((int64_t)t * a.n_head + h0) * hd + i];
    __syncthreads();
    // scores: thread = (position, half of the group)
    {
        const int s = threadIdx.x % CHUNK, half = threadIdx.x / CHUNK;  // 256 threads = 128 x 2
        constexpr int GH = (G + 1) / 2;
        const int g0 = half * GH;
        if (s < len) {
            float acc[GH];
#pragma unroll
            for (int g = 0; g < GH; g++) acc[g] = 0.0f;
            const uint16_t* key = a.k + (int64_t)(s0 + s) * a.kv_dim + off;
            for (int i = 0; i < hd; i += 8) {
                uint4 kk = *(const uint4*)(key + i);
                float kf[8];
                kf[0] = it_f16_to_f32((uint16_t)(kk.x & 0xffff)); kf[1] = it_f16_to_f32((uint16_t)(kk.x >> 16));
                kf[2] = it_f16_to_f32((uint16_t)(kk.y & 0xffff)); kf[3] = it_f16_to_f32((uint16_t)(kk.y >> 16));
                kf[4] = it_f16_to_f32((uint16_t)(kk.z & 0xffff)); kf[5] = it_f16_to_f32((uint16_t)(kk.z >> 16));
                kf[6] = it_f16_to_f32((uint16_t)(kk.w & 0xffff)); kf[7] = it_f16_to_f32((uint16_t)(kk.w >> 16));
#pragma unroll
                for (int g = 0; g < GH; g++) {
                    if (g0 + g < G) {
                        const float4 q0 = *(const float4*)(qs + (g0 + g) * hd + i);
                        const float4 q1 = *(const float4*)(qs + (g0 + g) * hd + i + 4);
                        acc[g] += q0.x * kf[0] + q0.y * kf[1] + q0.z * kf[2] + q0.w * kf[3] + q1.x * kf[4] +
                                  q1.y * kf[5] + q1.z * kf[6] + q1.w * kf[7];
                    }
                }
            }
#pragma unroll
            for (int g = 0; g < GH; g++)
                if (g0 + g < G) sc[s * G + g0 + g] = acc[g] * a.scale;
        }
    }
    __syncthreads();
    // per-head max and exp-sum over the chunk: wave w takes heads w, w+4, ...
    {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        for (int g = wave; g < G; g += 4) {
            float m = -INFINITY;
            for (int s = lane; s < len; s += 64) m = fmaxf(m, sc[s * G + g]);
            for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
            float l = 0.0f;
            for (int s = lane; s < len; s += 64) {
                float p = __expf(sc[s * G + g] - m);
                sc[s * G + g] = p;
                l += p;
            }
            for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o, 64);
            if (lane == 0) {
                mrow[g] = m;
                lrow[g] = l;
            }
        }
    }
    __syncthreads();
    // weighted values: thread = output dimension
    for (int i = threadIdx.x; i < hd; i += 256) {
        float acc[G];
#pragma unroll
        for (int g = 0; g < G; g++) acc[g] = 0.0f;
        const uint16_t* val = a.v + (int64_t)s0 * a.kv_dim + off + i;
        for (int s = 0; s < len; s++) {
            float v = it_f16_to_f32(val[(int64_t)s * a.kv_dim]);
#pragma unroll
            for (int g = 0; g < G; g++) acc[g] += sc[s * G + g] * v;
        }
#pragma unroll
        for (int g = 0; g < G; g++) my_part[g * part_head_stride + i] = acc[g];
    }
    if (threadIdx.x < G) {
        float* p = my_part + threadIdx.x * part_head_stride;
        p[hd] = mrow[threadIdx.x];
        p[hd + 1] = lrow[threadIdx.x];
    }
}

// gate (optional): out *= sigmoid(gate[head * gate_stride + i]) — the attention block's output gate.
// One block per (query, head).  Only the splits that hold positions are visited (n_live of them);
// their weights exp(m_s - m) are formed once, in LDS.
__global__ __launch_bounds__(1024) void attend_merge_k(const float* __restrict__ part, int n_split, int hd,
                                                       float* __restrict__ out, const float* __restrict__ gate,
                                                       int gate_stride, int n_q, int n_head, int chunk, int n_pos_arg,
                                                       const int* n_pos_dyn) {
    // blockDim = 4 * hd: four groups of hd threads, group g sums the splits s = g (mod 4)
    extern __shared__ float wsplit[];  // [n_split] then [4][hd]
    __shared__ float redm[16], redl[16];
    float* accs = wsplit + n_split;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = (blockDim.x + 63) >> 6;
    const int t = blockIdx.x / n_head;
    const int n_pos = (n_pos_dyn ? *n_pos_dyn : n_pos_arg) - n_q + 1 + t;
    int n_live = (n_pos + chunk - 1) / chunk;
    if (n_live > n_split) n_live = n_split;
    const float* p = part + (int64_t)blockIdx.x * n_split * (hd + 2);
    float m = -INFINITY;
    for (int s = tid; s < n_live; s += blockDim.x) m = fmaxf(m, p[(int64_t)s * (hd + 2) + hd]);
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    if (lane == 0) redm[wave] = m;
    __syncthreads();
    m = redm[0];
    for (int w = 1; w < nw; w++) m = fmaxf(m, redm[w]);
    float l = 0.0f;
    for (int s = tid; s < n_live; s += blockDim.x) {
        const float ms = p[(int64_t)s * (hd + 2) + hd];
        const float w = ms != -INFINITY ? __expf(ms - m) : 0.0f;
        wsplit[s] = w;
        l += p[(int64_t)s * (hd + 2) + hd + 1] * w;
    }
    for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o, 64);
    if (lane == 0) redl[wave] = l;
    __syncthreads();
    l = 0.0f;
    for (int w = 0; w < nw; w++) l += redl[w];
    const int g = tid / hd, i = tid - g * hd;
    float a0 = 0.0f, a1 = 0.0f;
    int s = g;
    for (; s + 4 < n_live; s += 8) {
        a0 += p[(int64_t)s * (hd + 2) + i] * wsplit[s];
        a1 += p[(int64_t)(s + 4) * (hd + 2) + i] * wsplit[s + 4];
    }
    if (s < n_live) a0 += p[(int64_t)s * (hd + 2) + i] * wsplit[s];
    accs[g * hd + i] = a0 + a1;
    __syncthreads();
    if (g == 0) {
        float r = ((accs[i] + accs[hd + i]) + (accs[2 * hd + i] + accs[3 * hd + i])) / l;
        if (gate) r *= fx_sigmoid(gate[(int64_t)blockIdx.x * gate_stride + i]);
        out[(int64_t)blockIdx.x * hd + i] = r;
    }
}

bool attend_split(const AttnArgs& a, int n_split, float* scratch, float* out, hipStream_t s) {
    if (attend_prefill(a, 1, nullptr, out, s)) return true;
    return attend_split_gated(a, n_split, scratch, out, nullptr, 0, s);
}

// Ranges that scratch has to hold partial results of.  Few queries (k_attn_decode.hip): one for every TILE keys, at most
// DECODE_SPLIT_MAX; the launch may use fewer.  Larger batches: a chunk each.
constexpr int TILE = 64, DECODE_SPLIT_MAX = 256;
int attend_split_count(int n_pos_max, int n_q, int head_dim, int group) {
    if (attend_decode_takes(n_q, head_dim, group)) return std::max(1, std::min(DECODE_SPLIT_MAX, (n_pos_max + TILE - 1) / TILE));
    return (n_pos_max + CHUNK - 1) / CHUNK;
}

bool attend_tile_prep_ok(const AttnArgs& a, const TilePrepP& pr) {
    const int G = a.n_head / a.n_head_kv, half = pr.n_rot / 2;
    if (a.n_q != 1 || !attend_decode_takes(1, a.head_dim, G) || !a.n_pos_dyn) return false;
    const int lph = a.head_dim / 4, hpp = 64 / lph;
    if (G % hpp && G > hpp) return false;
    // the rotated halves must be whole lanes and a power-of-two number of them, inside the head
    if (pr.n_rot <= 0 || half % 4 || ((half / 4) & (half / 4 - 1)) || pr.n_rot > a.head_dim) return false;
    return a.kv_dim % 4 == 0;
}

static bool attend_split_impl(const AttnArgs& a, const TilePrepP* prep, int n_split, float* scratch, float* out,
                              const float* gate, int gate_stride, hipStream_t s);

bool attend_split_gated(const AttnArgs& a, int n_split, float* scratch, float* out, const float* gate,
                        int gate_stride, hipStream_t s) {
    return attend_split_impl(a, nullptr, n_split, scratch, out, gate, gate_stride, s);
}

bool attend_split_gated_prep(const AttnArgs& a, const TilePrepP& pr, int n_split, float* scratch, float* out,
                             const float* gate, int gate_stride, hipStream_t s) {
    return attend_split_impl(a, &pr, n_split, scratch, out, gate, gate_stride, s);
}

// false: nothing was launched and `out` is untouched (a group size the kernels do not take, or LDS that could not be had);
// the caller records the error
static bool attend_split_impl(const AttnArgs& a, const TilePrepP* prep, int n_split, float* scratch, float* out,
                              const float* gate, int gate_stride, hipStream_t s) {
    if (a.n_q <= 0) return true;
    const int G = a.n_head / a.n_head_kv;
    if (attend_decode_takes(a.n_q, a.head_dim, G)) return attend_decode(a, prep, n_split, scratch, out, gate, gate_stride, s);
    dim3 grid(a.n_q * a.n_head_kv, n_split), block(256);
    size_t lds = ((size_t)G * a.head_dim + (size_t)CHUNK * G) * sizeof(float);
    switch (G) {
        case 1: hipLaunchKernelGGL(attend_split_k<1>, grid, block, lds, s, a, n_split, scratch); break;
        case 2: hipLaunchKernelGGL(attend_split_k<2>, grid, block, lds, s, a, n_split, scratch); break;
        case 4: hipLaunchKernelGGL(attend_split_k<4>, grid, block, lds, s, a, n_split, scratch); break;
        case 8: hipLaunchKernelGGL(attend_split_k<8>, grid, block, lds, s, a, n_split, scratch); break;
        default: return false;  // the caller takes the exact kernel for other group sizes
    }
    hipLaunchKernelGGL(attend_merge_k, dim3(a.n_q * a.n_head), dim3(4 * a.head_dim),
                       (size_t)(n_split + 4 * a.head_dim) * sizeof(float), s, scratch, n_split, a.head_dim, out, gate,
                       gate_stride, a.n_q, a.n_head, CHUNK, a.n_pos, a.n_pos_dyn);
    return true;
}

}  // namespace itk
