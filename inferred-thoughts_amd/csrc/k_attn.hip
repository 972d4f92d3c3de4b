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
#include "it_launch.h"
#include "it_reduce.h"
#include "kernels.h"
#include "kernels_fused.h"

namespace itk {

// ------------------------------------------------------------------ exact
// One block per (query, head).  Scores and weights sit in LDS up to EXACT_LDS positions (beyond, in `scratch`).  What has an
// order is a chain: a position's dot in its thread, the weights' sum in one lane, a dim's weighted sum in its thread, each
// with its loads several steps ahead.  333 positions, 16 heads of 256: 28 us (115 with every read waited for
// and the weight divided anew for every dim).
constexpr int EXACT_LDS = 4096;
__global__ __launch_bounds__(1024) void attend_exact_k(AttnArgs a, float* __restrict__ scratch, float* __restrict__ out,
                                                      const float* __restrict__ gate, int gate_stride, int lds_pos) {
    extern __shared__ __align__(16) float qs[];  // head_dim, then the first lds_pos scores (a multiple of 4 each)
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
    for (int i = tid; i < hd; i += nt) qs[i] = q[i];
    __syncthreads();
    float m = -INFINITY;
    for (int s = tid; s < n_pos; s += nt) {
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
        constexpr int AHEAD = 32;   // positions whose values are on their way while as many are added
        uint16_t x0[AHEAD], x1[AHEAD];
        auto ask = [&](uint16_t (&x)[AHEAD], int from) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < AHEAD; c++) x[c] = v[(int64_t)min(from + c, n_pos - 1) * a.kv_dim];
        };
        auto add = [&](const uint16_t (&x)[AHEAD], int from) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < AHEAD; c++) acc += near[from + c] * it_f16_to_f32(x[c]);
        };
        if (n_lds >= AHEAD) ask(x0, 0);
        for (; s + 2 * AHEAD <= n_lds; s += 2 * AHEAD) {
            ask(x1, s + AHEAD);
            add(x0, s);
            ask(x0, s + 2 * AHEAD);
            add(x1, s + AHEAD);
        }
        if (s + AHEAD <= n_lds) {
            add(x0, s);
            s += AHEAD;
        }
        for (; s < n_lds; s++) acc += near[s] * it_f16_to_f32(v[(int64_t)s * a.kv_dim]);
#pragma unroll 8
        for (s = lds_pos; s < n_pos; s++) acc += far[s] * it_f16_to_f32(v[(int64_t)s * a.kv_dim]);
        if (gate) acc *= it_sigmoid(gate[(int64_t)h * gate_stride + i]);   // (n_q == 1: sigmoid_mul of the gated block)
        out[((int64_t)t * a.n_head + h) * hd + i] = acc;
    }
}

void attend_exact(const AttnArgs& a, float* scratch, float* out, hipStream_t s, const float* gate, int gate_stride) {
    if (a.n_q <= 0) return;
    const int lds_pos = std::min((a.n_pos + 3) & ~3, EXACT_LDS);
    // few blocks: a thread per position while the score phase has that many; many: blocks that share a CU
    const int threads = a.n_q * a.n_head < 512 && a.n_pos > 256 ? 1024 : 256;
    hipLaunchKernelGGL(attend_exact_k, dim3(a.n_q * a.n_head), dim3(threads), ((size_t)((a.head_dim + 3) & ~3) + lds_pos) * sizeof(float), s, a,
                       scratch, out, gate, gate_stride, lds_pos);
}

// ------------------------------------------------------------------ exact, one query
// A recorded token's: a block per head and 64 dims of its result forms the query and the new position's key and value from the
// projections, a wave each, and keeps the new rows in LDS; the first block of a KV head leaves them in the slabs, which no block reads
// at that position.  (A launch in front took 4.6 us for that, 2.5 of them its start and the projections' trip.)
// The chains are attend_exact_k's; what bounded them there were 16-byte reads of rows a KV stride apart, a line a lane, values two
// bytes at a time, and what one CU is served (174 KB of keys in 3 us, as much of values in 6).  So a wave brings 64 keys' rows 64 dims
// at a time, whole lines, through a piece of LDS of its own (rows 144 bytes apart: no bank conflicts), the next piece in registers
// meanwhile; a block brings its 64 dims of 512 values while the weights are formed, all threads form the products, and one wave adds
// them up.  340 positions, 16 heads of 256: 27.3 -> 15.1 us (22.5 with all dims in a block); a token of four layers of 512 values,
// 33 to 290 positions, 8 heads of 64: 115.7 -> 112.0 us.  Longer contexts, where a head's blocks repeat its scores and the weights lie in
// memory from 4,096 on: an attention block with 16 heads of 256 over 2,000 / 4,000 / 8,000 / 32,000 positions 131, 237, 537, 2,373 us in the two
// launches, 67, 105, 203, 804 so; 8 heads of 64 92, 157, 308, 1,720 and 54, 75, 144, 590.
constexpr int ONE_DIMS = 64, ONE_T = 512, ONE_ROW = 144, ONE_V = 8;      // threads; bytes of a key's piece in LDS; 16-byte pieces of values a thread brings
constexpr int ONE_VALUES = ONE_T * ONE_V * 16, ONE_STAGE = 2 * ONE_VALUES;   // (as f32 products)
static_assert(ONE_T * ONE_ROW <= ONE_STAGE, "the keys' pieces lie where the values go later");
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
// a lane's value, in a scalar register; and its product with a half of `h`, rounded once as a product of f32 is (what is added to
// nothing is never -0: a sum that starts at 0 cannot tell the sign of a zero)
IT_DEV float lane_value(float v, int lane) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane)); }
template <bool HIGH, bool SCALAR>   // SCALAR: `s` is the same in every lane
IT_DEV float times_half(float s, uint32_t h) {
    float r;
    if constexpr (SCALAR) {
        if constexpr (HIGH) asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "=v"(r) : "s"(s), "v"(h));
        else asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel_hi:[0,1,0]" : "=v"(r) : "s"(s), "v"(h));
    } else {
        if constexpr (HIGH) asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "=v"(r) : "v"(s), "v"(h));
        else asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel_hi:[0,1,0]" : "=v"(r) : "v"(s), "v"(h));
    }
    return r;
}
template <int HD>
__global__ __launch_bounds__(ONE_T) void attend_exact_one_k(AttnArgs a, AttnPrepP pr, float* __restrict__ scratch, float* __restrict__ out,
                                                            const float* __restrict__ gate, int gate_stride, int lds_pos) {
    extern __shared__ __align__(16) uint8_t one_smem[];   // ONE_STAGE bytes, then the query, the new key and value, and lds_pos scores
    __shared__ float red[ONE_T / 64 + 1];
    __shared__ uint64_t etab[32];
    constexpr int hd = HD, NP = HD / 64;             // pieces of a key
    constexpr int pv = ONE_DIMS / 8, rows = ONE_VALUES / 2 / ONE_DIMS;   // 16-byte pieces of a row of values, rows brought at a time
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint8_t* const lds = one_smem;
    float* const qs = (float*)(lds + ONE_STAGE);
    float* const fresh = qs + hd;                    // key, value
    float* const near = fresh + 2 * hd;
    const int n_pos = *a.n_pos_dyn, pos = n_pos - 1, n_lds = min(n_pos, lds_pos);   // positions 0 .. pos - 1 are read from the slabs
    const int h = blockIdx.x, group = a.n_head / a.n_head_kv, off = h / group * hd, d0 = ONE_DIMS * blockIdx.y;   // the block's dims of the result
    float* const far = scratch + (int64_t)(blockIdx.y * gridDim.x + h) * n_pos;
    // (LDS and memory by separate instructions: through a pointer to either, a read waits for all that is on its way)
    auto put = [&](int s, float v) __attribute__((always_inline)) {
        if (s < lds_pos) near[s] = v;
        asm volatile("");
        if (s >= lds_pos) far[s] = v;
    };
    if (tid < 32) etab[tid] = IT_EXP2F_TAB[tid];

    // ---- scores: step `it` of a wave is piece it % NP of positions 64 wave + 512 (it / NP) ..
    const int steps = pos > 64 * wave ? (pos - 64 * wave + ONE_T - 1) / ONE_T * NP : 0;
    uint8_t* const piece = lds + wave * 64 * ONE_ROW;
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));   // (arrays of uint4 were left in memory)
    u4 kk[8] = {};
    auto ask_k = [&](int base, int p) __attribute__((always_inline)) {
        const uint16_t* const from = a.k + off + 64 * p + 8 * (lane & 7);
#pragma unroll
        for (int j = 0; j < 8; j++) kk[j] = *(const u4*)(from + (int64_t)min(base + 8 * j + (lane >> 3), pos - 1) * a.kv_dim);
    };
    if (steps) ask_k(64 * wave, 0);
    {
        const bool first = d0 == 0, leaves = first && h % group == 0;
        if (wave == 0) {
            wave_norm_rope(qs, pr.qg + (int64_t)h * 2 * hd, pr.q_norm, hd, pr, pos, lane);
            if (first)
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
    }
    __syncthreads();
    float m = -INFINITY;
    if (tid == ONE_T - 1) {                          // (of the wave with the fewest positions of its own)
        float dot = 0.0f;
#pragma unroll 8
        for (int i = 0; i < hd; i++) dot += qs[i] * fresh[i];
        m = dot * a.scale;
        put(pos, m);
    }
    // products are formed eight ahead of their addition, and the scalar they take two ahead of them (each waits some eight cycles
    // for the one before it; the zeros in front add nothing)
    float dot = 0.0f, due[8] = {};
    for (int it = 0, base = 64 * wave, p = 0; it < steps; it++) {
#pragma unroll
        for (int j = 0; j < 8; j++) *(u4*)(piece + (8 * j + (lane >> 3)) * ONE_ROW + 16 * (lane & 7)) = kk[j];
        wave_lds_sync();
        const float q = qs[64 * p + lane];
        const int s = base + lane;
        const bool whole = ++p == NP;
        if (whole) {
            p = 0;
            base += ONE_T;
        }
        if (it + 1 < steps) ask_k(base, p);
        const uint8_t* const row = piece + lane * ONE_ROW;
        u4 x[8];
#pragma unroll
        for (int j = 0; j < 8; j++) x[j] = *(const u4*)(row + 16 * j);
        float s0 = lane_value(q, 0), s1 = lane_value(q, 1);
#pragma unroll
        for (int e = 0; e < 64; e++) {
            const float s2 = lane_value(q, min(e + 2, 63));
            dot += due[e % 8];
            const uint32_t pair = x[e / 8][e / 2 % 4];
            due[e % 8] = e & 1 ? times_half<true, true>(s0, pair) : times_half<false, true>(s0, pair);
            s0 = s1;
            s1 = s2;
            __builtin_amdgcn_sched_barrier(0);
        }
        wave_lds_sync();
        if (whole) {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                dot += due[e];
                due[e] = 0.0f;
            }
            const float v = dot * a.scale;
            dot = 0.0f;
            if (s < pos) {
                put(s, v);
                m = fmaxf(m, v);
            }
        }
    }
    // ---- the first values, while the weights are formed
    u4 vv[ONE_V] = {};
    auto ask_v = [&](int row0) __attribute__((always_inline)) {
        const uint16_t* const from = a.v + off + d0 + 8 * (tid % pv);
#pragma unroll
        for (int j = 0; j < ONE_V; j++) {
            if (row0 + ONE_T / pv * j >= pos) break;
            vv[j] = *(const u4*)(from + (int64_t)min(row0 + tid / pv + ONE_T / pv * j, pos - 1) * a.kv_dim);
        }
    };
    if (pos) ask_v(0);
    m = group_max<64>(m);
    if (lane == 0) red[wave] = m;
    __syncthreads();
    m = red[0];
#pragma unroll
    for (int w = 1; w < ONE_T / 64; w++) m = fmaxf(m, red[w]);
    for (int s = tid; s < n_lds; s += ONE_T) near[s] = it_expf_by(near[s] - m, etab);
    for (int s = lds_pos + tid; s < n_pos; s += ONE_T) far[s] = it_expf_by(far[s] - m, etab);
    __threadfence_block();
    __syncthreads();
    if (wave == 0) {   // (every lane: reads of one address by all cost less than by one lane)
        float sum = fold_terms(near, n_lds);
#pragma unroll 16
        for (int s = lds_pos; s < n_pos; s++) sum += far[s];
        red[ONE_T / 64] = sum;
    }
    __syncthreads();
    const float sum = red[ONE_T / 64];
    for (int s = tid; s < n_lds; s += ONE_T) near[s] = near[s] / sum;
    for (int s = lds_pos + tid; s < n_pos; s += ONE_T) far[s] = far[s] / sum;
    __threadfence_block();

    // ---- the weighted sum: every thread forms the products of what it has brought, the first wave adds them up, a dim a lane.
    // Products lie [dim][row]; which four rows lie where is turned by the dim, so that eight rows of eight dims (written at once) and
    // four rows of sixteen dims (read at once) hit different banks.
    float* const prod = (float*)lds;
    auto turn = [](int d) __attribute__((always_inline)) { return 2 * (((d >> 3) ^ d) & 7) | ((d >> 3) & 1); };
    float acc = 0.0f;
    for (int row0 = 0; row0 < pos; row0 += rows) {
        __syncthreads();                             // (the weights are there; the products before have been read)
        float w[ONE_V];
        static_assert(EXACT_LDS % rows == 0, "all of a piece's weights in LDS, or none");
        if (row0 < lds_pos) {
#pragma unroll
            for (int j = 0; j < ONE_V; j++) w[j] = near[min(row0 + tid / pv + ONE_T / pv * j, pos)];
        } else {
#pragma unroll
            for (int j = 0; j < ONE_V; j++) w[j] = far[min(row0 + tid / pv + ONE_T / pv * j, pos)];
        }
#pragma unroll
        for (int j = 0; j < ONE_V; j++) {
            const int r = tid / pv + ONE_T / pv * j, s = row0 + r;
            if (row0 + ONE_T / pv * j >= pos) break;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int d = 8 * (tid % pv) + e;
                const uint32_t pair = vv[j][e / 2];
                const float x = e & 1 ? times_half<true, false>(w[j], pair) : times_half<false, false>(w[j], pair);
                prod[d * rows + 4 * ((r >> 2) ^ turn(d)) + (r & 3)] = s < pos ? x : 0.0f;   // (0 adds nothing)
            }
        }
        if (row0 + rows < pos) ask_v(row0 + rows);
        __syncthreads();
        if (wave) continue;
        constexpr int AHEAD = 8;                     // times four rows, on their way while as many are added
        const float4* const p = (const float4*)(prod + lane * rows);
        const int n4 = (min(rows, pos - row0) + 4 * AHEAD - 1) / (4 * AHEAD) * AHEAD, t = turn(lane);
        float4 x0[AHEAD], x1[AHEAD];
        auto get = [&](float4 (&x)[AHEAD], int r4) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < AHEAD; c++) x[c] = p[min(r4 + c, rows / 4 - 1) ^ t];
        };
        auto add = [&](const float4 (&x)[AHEAD]) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < AHEAD; c++) {
                acc += x[c].x;
                acc += x[c].y;
                acc += x[c].z;
                acc += x[c].w;
            }
        };
        get(x0, 0);
        int r4 = 0;
        for (; r4 + 2 * AHEAD <= n4; r4 += 2 * AHEAD) {
            get(x1, r4 + AHEAD);
            add(x0);
            get(x0, r4 + 2 * AHEAD);
            add(x1);
        }
        if (r4 < n4) add(x0);
    }
    if (!pos) __syncthreads();                       // (the new position's weight)
    if (tid < ONE_DIMS) {
        acc += (pos < lds_pos ? near[pos] : far[pos]) * fresh[hd + d0 + tid];
        if (gate) acc *= it_sigmoid(gate[(int64_t)h * gate_stride + d0 + tid]);   // (sigmoid_mul of the gated block)
        out[(int64_t)h * hd + d0 + tid] = acc;
    }
}

template <int HD>
static bool one_launch(const AttnArgs& a, const AttnPrepP& prep, float* scratch, float* out, const float* gate, int gate_stride, hipStream_t s, bool dry_run) {
    auto lds = [](int lds_pos) { return ONE_STAGE + (size_t)(3 * HD + lds_pos) * sizeof(float); };
    const int lds_pos = std::min((a.n_pos + 3) & ~3, EXACT_LDS);
    if (!lds_allowed<&attend_exact_one_k<HD>>(lds(EXACT_LDS))) return false;
    if (!dry_run) hipLaunchKernelGGL(attend_exact_one_k<HD>, dim3(a.n_head, HD / ONE_DIMS), dim3(ONE_T), lds(lds_pos), s, a, prep, scratch, out, gate, gate_stride, lds_pos);
    return true;
}
int attend_exact_one_rows(int head_dim) { return head_dim == 64 || head_dim == 128 || head_dim == 256 ? head_dim / ONE_DIMS : 1; }
bool attend_exact_one(const AttnArgs& a, const AttnPrepP& prep, float* scratch, float* out, const float* gate, int gate_stride, hipStream_t s, bool dry_run) {
    if (a.n_q != 1 || !a.n_pos_dyn || a.kv_dim % 8 || ((uintptr_t)a.k & 15) || ((uintptr_t)a.v & 15)) return false;
    // a head's blocks read the projections, write their dims of the result and, one of them, the query, each at its own time
    if (out == prep.q || out == prep.k || out == prep.v) return false;
    if (a.head_dim == 64) return one_launch<64>(a, prep, scratch, out, gate, gate_stride, s, dry_run);
    if (a.head_dim == 128) return one_launch<128>(a, prep, scratch, out, gate, gate_stride, s, dry_run);
    return a.head_dim == 256 && one_launch<256>(a, prep, scratch, out, gate, gate_stride, s, dry_run);
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
