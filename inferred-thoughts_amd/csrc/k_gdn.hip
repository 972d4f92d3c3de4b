// Gated delta rule (GatedDeltaNet's recurrent core).
//
// Follows /root/reference src/ops/naive.rs:86-135 per token and :339-350 over the
// batch; head grouping is modulo (src/ops/mod.rs:404-413).  State is
// [value head][value row][key] f32, key contiguous.
//
// Exact mode: four lanes own one value row, a quarter of its dk floats each, in registers for the whole batch.  Decay,
// correction and products are the lane's own; a sum over the row runs through the four in turn, each adding its quarter to
// what the one before it hands over, so that every addition is the reference's, in its order.
#include "it_device.h"
#include "it_dot.h"
#include "it_reduce.h"
#include "kernels.h"

namespace itk {

// A block is 16 rows of one head (256 blocks for 32 heads of 128).  Tokens go in chunks of 16: a chunk's k, q
// (scaled), v and gates are staged in LDS, the next chunk's loads in flight meanwhile.  Bound by the instructions between a token's
// state and the next one's, a chain of dk dependent additions among them (one lane per row, with every token's loads waited for, took
// 4.1 us a token of 128).  The read-out's chain is not between them: a second wave adds its products up, through LDS, while the first
// is at the next token, stages the chunks and stores (333 tokens, 32 heads of 128: 272 us in one wave, 248 so; the request with eight more tokens 3.08 -> 3.06 ms).
constexpr int DX_TCH = 16, DX_ROWS = 16;
IT_DEV float quad_lane(float v, int which) {   // lane `which` of each aligned group of four, to all of it
    const int u = __builtin_bit_cast(int, v);
    const int r = which == 0   ? __builtin_amdgcn_update_dpp(0, u, 0x00, 0xf, 0xf, true)
                  : which == 1 ? __builtin_amdgcn_update_dpp(0, u, 0x55, 0xf, 0xf, true)
                  : which == 2 ? __builtin_amdgcn_update_dpp(0, u, 0xAA, 0xf, 0xf, true)
                               : __builtin_amdgcn_update_dpp(0, u, 0xFF, 0xf, 0xf, true);
    return __builtin_bit_cast(float, r);
}
template <int SEG>
IT_DEV float quad_chain(const float (&p)[SEG]) {
    float acc = 0.0f;
#pragma unroll
    for (int s = 0; s < 4; s++) {
        float a = acc;
#pragma unroll
        for (int e = 0; e < SEG; e++) a += p[e];
        acc = quad_lane(a, s);
    }
    return acc;
}
template <int DK>
__global__ __launch_bounds__(128) void delta_rule_k(DeltaArgs d, float* __restrict__ state, float* __restrict__ out, float q_scale) {
    constexpr int SEG = DK / 4, SS = SEG + 4;             // + 4: the four quarters' 16-byte reads fall on different banks
    constexpr int L4 = DX_TCH * DK / 4 / 64;              // float4 of k (and of q) per lane and chunk
    __shared__ __align__(16) float kb[2][DX_TCH][4 * SS], qb[2][DX_TCH][4 * SS];
    __shared__ float vb[2][DX_TCH][DX_ROWS], gb[2][DX_TCH][2];
    constexpr int PS = DX_ROWS * SS + 16;                 // (rows' and quarters' 16-byte accesses: other banks, written and read)
    __shared__ __align__(16) float pb[2][4 * PS];         // a token's read-out products, quarter by quarter
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane >> 2, seg = lane & 3;
    const int dv = d.head_v_dim;
    const int bph = (dv + DX_ROWS - 1) / DX_ROWS;
    const int h = blockIdx.x / bph, jb = blockIdx.x % bph;
    const int kh = h % d.n_k_heads;
    const int j = jb * DX_ROWS + r, jc = min(j, dv - 1);   // rows past the head repeat its last one and are not stored
    float* S = state + ((int64_t)h * dv + jc) * DK + seg * SEG;
    const int kper = d.n_k_heads * DK, vper = d.n_v_heads * dv, n = d.n_tokens;

    float row[SEG];
#pragma unroll
    for (int i = 0; i < SEG / 4; i++) {
        const float4 t = ((const float4*)S)[i];
        row[4 * i] = t.x; row[4 * i + 1] = t.y; row[4 * i + 2] = t.z; row[4 * i + 3] = t.w;
    }
    typedef float f4 __attribute__((ext_vector_type(4)));   // (arrays of float4 were left in memory)
    f4 rk[L4] = {}, rq[L4] = {};
    float rv[DX_TCH * DX_ROWS / 64] = {}, ra = 0.0f, rb = 0.0f;
    auto load = [&](int t0) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < L4; p++) {
            const int idx = p * 64 + lane, t = min(t0 + idx / (DK / 4), n - 1), c = idx % (DK / 4);
            rk[p] = ((const f4*)(d.k + (int64_t)t * kper + kh * DK))[c];
            rq[p] = ((const f4*)(d.q + (int64_t)t * kper + kh * DK))[c];
        }
#pragma unroll
        for (int p = 0; p < DX_TCH * DX_ROWS / 64; p++) {
            const int idx = p * 64 + lane, t = min(t0 + idx / DX_ROWS, n - 1);
            rv[p] = d.v[(int64_t)t * vper + h * dv + min(jb * DX_ROWS + idx % DX_ROWS, dv - 1)];
        }
        const int t = min(t0 + (lane & (DX_TCH - 1)), n - 1);
        ra = d.alpha[(int64_t)t * d.n_v_heads + h] + d.dt_bias[h];
        rb = d.beta[(int64_t)t * d.n_v_heads + h];
    };
    auto stash = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < L4; p++) {
            const int idx = p * 64 + lane, t = idx / (DK / 4), i = 4 * (idx % (DK / 4));
            const int at = i / SEG * SS + i % SEG;
            *(f4*)&kb[b][t][at] = rk[p];
            *(f4*)&qb[b][t][at] = f4{rq[p].x * q_scale, rq[p].y * q_scale, rq[p].z * q_scale, rq[p].w * q_scale};
        }
#pragma unroll
        for (int p = 0; p < DX_TCH * DX_ROWS / 64; p++) vb[b][(p * 64 + lane) / DX_ROWS][(p * 64 + lane) % DX_ROWS] = rv[p];
        const float softplus = ra > 20.0f ? ra : it_logf(1.0f + it_expf(ra));
        const float g = it_expf(softplus * d.ssm_a[h]), beta = 1.0f / (1.0f + it_expf(-rb));
        if (lane < DX_TCH) {
            gb[b][lane][0] = g;
            gb[b][lane][1] = beta;
        }
    };
    auto meet = [&]() __attribute__((always_inline)) {      // (what is on its way from memory is not waited for)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    if (wave) {
        load(0);
        stash(0);
    }
    meet();
    // the first wave's next token: key, gates, value (asked for a token ahead: a trip to LDS between two tokens otherwise)
    f4 kn[SEG / 4];
    float gn = 0.0f, bn = 0.0f, vn = 0.0f;
    auto ask = [&](int b, int t) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < SEG / 4; i++) kn[i] = *(const f4*)&kb[b][t][seg * SS + 4 * i];
        gn = gb[b][t][0];
        bn = gb[b][t][1];
        vn = vb[b][t][r];
    };
    ask(0, 0);
    for (int t0 = 0, b = 0; t0 < n; t0 += DX_TCH, b ^= 1) {
        const int live = min(DX_TCH, n - t0);
        for (int t = 0; t < live; t++) {
            float* const mine = pb[t & 1];                  // (a chunk that another follows is even)
            if (wave == 0) {
                const float g = gn, beta = bn, v = vn;
                const float4* q4 = (const float4*)&qb[b][t][seg * SS];
                float kk[SEG], p[SEG];
                f4 qx[SEG / 4];
#pragma unroll
                for (int i = 0; i < SEG / 4; i++) {
                    kk[4 * i] = kn[i].x; kk[4 * i + 1] = kn[i].y; kk[4 * i + 2] = kn[i].z; kk[4 * i + 3] = kn[i].w;
                    qx[i] = ((const f4*)q4)[i];
                }
                if (t + 1 < live) ask(b, t + 1);
                else ask(b ^ 1, 0);                         // (the next chunk's is there; behind the last one it is not used)
#pragma unroll
                for (int i = 0; i < SEG; i++) {
                    row[i] *= g;
                    p[i] = row[i] * kk[i];
                }
                const float delta = beta * (v - quad_chain<SEG>(p));
#pragma unroll
                for (int i = 0; i < SEG / 4; i++) {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        row[4 * i + e] += kk[4 * i + e] * delta;
                        p[4 * i + e] = row[4 * i + e] * qx[i][e];
                    }
                    *(float4*)&mine[seg * PS + r * SS + 4 * i] = make_float4(p[4 * i], p[4 * i + 1], p[4 * i + 2], p[4 * i + 3]);
                }
            }
            meet();
            if (wave) {
                float o = 0.0f;
#pragma unroll
                for (int s = 0; s < 4; s++) o = fold_terms_from(o, mine + s * PS + (lane & 15) * SS, SEG);
                if (lane < DX_ROWS && jb * DX_ROWS + lane < dv) out[(int64_t)(t0 + t) * vper + h * dv + jb * DX_ROWS + lane] = o;
                if (t0 + DX_TCH < n) {                      // (a whole chunk)
                    if (t == 0) load(t0 + DX_TCH);
                    if (t == DX_TCH / 2) stash(b ^ 1);
                }
            }
        }
    }
    if (wave) return;
    if (j < dv) {
#pragma unroll
        for (int i = 0; i < SEG / 4; i++) ((float4*)S)[i] = make_float4(row[4 * i], row[4 * i + 1], row[4 * i + 2], row[4 * i + 3]);
    }
}

// ------------------------------------------------------------------ fast form over a batch
// 32 value rows per block, 8 lanes per row (DK / 8 keys each): the row's dots are reduced
// with three lane exchanges, so the sums are not in the CPU path's order (fast mode only).
// The gates of every token of the batch are formed once, up front, in LDS.  The batch is
// walked in chunks of 16 tokens: a chunk's k, q and v are staged into LDS with coalesced
// loads while the previous chunk is being applied, so a token step touches only LDS and
// registers and the only block barrier is the one between chunks.
constexpr int GDN_TCH = 16;

template <int DK>
__global__ __launch_bounds__(256) void delta_rule_fast_k(DeltaArgs d, float* __restrict__ state,
                                                         float* __restrict__ out, float q_scale) {
    constexpr int SEG = DK / 8;
    constexpr int V4 = SEG / 4;
    constexpr int KQ4 = GDN_TCH * DK / 4;          // float4 per chunk of k (and of q)
    constexpr int KQL = (KQ4 + 255) / 256;          // per thread
    extern __shared__ __align__(16) float lds[];
    float* gates = lds;                                               // [n_tokens][2]
    float* kbuf = lds + (((size_t)d.n_tokens * 2 + 3) & ~(size_t)3);  // [2][TCH][DK]
    float* qbuf = kbuf + 2 * GDN_TCH * DK;                            // [2][TCH][DK]
    float* vbuf = qbuf + 2 * GDN_TCH * DK;                            // [2][TCH][32]
    const int tid = threadIdx.x, seg = tid & 7, r = tid >> 3;
    const int dv = d.head_v_dim;
    const int bph = dv / 32;
    const int h = blockIdx.x / bph, jb = blockIdx.x % bph, kh = h % d.n_k_heads;
    const int j = jb * 32 + r;
    const int kper = d.n_k_heads * DK, vper = d.n_v_heads * dv;
    for (int t = tid; t < d.n_tokens; t += 256) {
        const float a = d.alpha[(int64_t)t * d.n_v_heads + h] + d.dt_bias[h];
        const float softplus = a > 20.0f ? a : fx_logf(1.0f + fx_expf(a));
        gates[2 * t] = fx_expf(softplus * d.ssm_a[h]);
        gates[2 * t + 1] = fx_sigmoid(d.beta[(int64_t)t * d.n_v_heads + h]);
    }
    float* S = state + ((int64_t)h * dv + j) * DK + seg * SEG;
    float row[SEG];
#pragma unroll
    for (int i = 0; i < V4; i++) {
        const float4 t4 = ((const float4*)S)[i];
        row[4 * i] = t4.x; row[4 * i + 1] = t4.y; row[4 * i + 2] = t4.z; row[4 * i + 3] = t4.w;
    }
    float4 rk[KQL], rq[KQL];
    float rv[2];
    auto fetch = [&](int t0) {
#pragma unroll
        for (int p = 0; p < KQL; p++) {
            const int idx = tid + p * 256, tt = idx / (DK / 4), c4 = idx % (DK / 4);
            const bool ok = idx < KQ4 && t0 + tt < d.n_tokens;
            rk[p] = ok ? ((const float4*)(d.k + (int64_t)(t0 + tt) * kper + kh * DK))[c4] : make_float4(0.f, 0.f, 0.f, 0.f);
            rq[p] = ok ? ((const float4*)(d.q + (int64_t)(t0 + tt) * kper + kh * DK))[c4] : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const int idx = tid + p * 256, tt = idx >> 5, rr = idx & 31;
            rv[p] = t0 + tt < d.n_tokens ? d.v[(int64_t)(t0 + tt) * vper + h * dv + jb * 32 + rr] : 0.0f;
        }
    };
    auto stash = [&](int buf) {
#pragma unroll
        for (int p = 0; p < KQL; p++) {
            const int idx = tid + p * 256;
            if (idx < KQ4) {
                ((float4*)(kbuf + buf * GDN_TCH * DK))[idx] = rk[p];
                ((float4*)(qbuf + buf * GDN_TCH * DK))[idx] = rq[p];
            }
        }
#pragma unroll
        for (int p = 0; p < 2; p++) vbuf[buf * GDN_TCH * 32 + tid + p * 256] = rv[p];
    };
    fetch(0);
    stash(0);
    __syncthreads();
    for (int t0 = 0, c = 0; t0 < d.n_tokens; t0 += GDN_TCH, c++) {
        const int buf = c & 1;
        if (t0 + GDN_TCH < d.n_tokens) fetch(t0 + GDN_TCH);
        const int nt = min(GDN_TCH, d.n_tokens - t0);
        for (int tt = 0; tt < nt; tt++) {
            const float4* k4 = (const float4*)(kbuf + (buf * GDN_TCH + tt) * DK + seg * SEG);
            const float4* q4 = (const float4*)(qbuf + (buf * GDN_TCH + tt) * DK + seg * SEG);
            float kk[SEG], qq[SEG];
#pragma unroll
            for (int i = 0; i < V4; i++) {
                const float4 a = k4[i], b = q4[i];
                kk[4 * i] = a.x; kk[4 * i + 1] = a.y; kk[4 * i + 2] = a.z; kk[4 * i + 3] = a.w;
                qq[4 * i] = b.x; qq[4 * i + 1] = b.y; qq[4 * i + 2] = b.z; qq[4 * i + 3] = b.w;
            }
            const float v = vbuf[(buf * GDN_TCH + tt) * 32 + r];
            const float g = gates[2 * (t0 + tt)], beta = gates[2 * (t0 + tt) + 1];
            float pred = 0.0f;
#pragma unroll
            for (int i = 0; i < SEG; i++) {
                row[i] *= g;
                pred += row[i] * kk[i];
            }
            pred = sum8_lanes(pred);
            const float delta = beta * (v - pred);
            float o = 0.0f;
#pragma unroll
            for (int i = 0; i < SEG; i++) {
                row[i] += kk[i] * delta;
                o += row[i] * (qq[i] * q_scale);
            }
            o = sum8_lanes(o);
            if (seg == 0) out[(int64_t)(t0 + tt) * vper + h * dv + j] = o;
        }
        if (t0 + GDN_TCH < d.n_tokens) stash(buf ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < V4; i++)
        ((float4*)S)[i] = make_float4(row[4 * i], row[4 * i + 1], row[4 * i + 2], row[4 * i + 3]);
}

void delta_rule(const DeltaArgs& d, float* state, float* out, int exact, float* work, size_t work_floats, hipStream_t s) {
    if (d.n_tokens <= 0) return;
    if (!exact && delta_rule_chunked(d, state, out, work, work_floats, s)) return;
    float q_scale = 1.0f / sqrtf((float)d.head_k_dim);
    const size_t gate_lds = ((((size_t)d.n_tokens * 2 + 3) & ~(size_t)3) + 4 * GDN_TCH * d.head_k_dim + 2 * GDN_TCH * 32) * sizeof(float);
    if (!exact && d.head_v_dim % 32 == 0 && (d.head_k_dim == 64 || d.head_k_dim == 128) && gate_lds <= 96 * 1024) {
        const int blocks = d.n_v_heads * (d.head_v_dim / 32);
        if (d.head_k_dim == 64) hipLaunchKernelGGL(delta_rule_fast_k<64>, dim3(blocks), dim3(256), gate_lds, s, d, state, out, q_scale);
        else hipLaunchKernelGGL(delta_rule_fast_k<128>, dim3(blocks), dim3(256), gate_lds, s, d, state, out, q_scale);
        return;
    }
    int blocks = d.n_v_heads * ((d.head_v_dim + DX_ROWS - 1) / DX_ROWS);
    switch (d.head_k_dim) {
        case 32: hipLaunchKernelGGL(delta_rule_k<32>, dim3(blocks), dim3(128), 0, s, d, state, out, q_scale); break;
        case 64: hipLaunchKernelGGL(delta_rule_k<64>, dim3(blocks), dim3(128), 0, s, d, state, out, q_scale); break;
        case 128: hipLaunchKernelGGL(delta_rule_k<128>, dim3(blocks), dim3(128), 0, s, d, state, out, q_scale); break;
        default: break;  // the caller validates head_k_dim
    }
}

}  // namespace itk
