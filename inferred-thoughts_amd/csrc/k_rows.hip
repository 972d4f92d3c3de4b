// Runs of row-wise ops of a batch pass as one launch each (fast mode).
//
// Between two products of a batch the loop (src/model/qwen35.rs:956-1328, 1630-1700) has three to six ops that each read and
// write a few hundred kilobytes: a launch apiece is 4.7 us of dispatch for a tenth of that in memory time, and on long
// batches a pass over memory each.  Here a row stays in the registers of its wave or block from one op of a run to the
// next.  Every value is formed as the kernels it replaces form it (f64 sums of squares, round-half-away Q8_0 blocks with
// the scale through f16, softmax with f32 sums); only the order of the long sums differs.  All of it is bound by memory or,
// below some 500 tokens, by the launch itself, so a row's loads are all issued before its first use.
//
// The split form of a row (what the f16 matrix-core kernels multiply): the Q8_0 value q * d divided by the row's power of
// two and written as f16 hi + lo (22 bits kept), inside every unit of 32 elements in the order in which a lane's operand of
// those kernels takes them: element j at 8 n + 2 (j % 4) + j / 8 % 2 with n = 2 (j / 16) + (j / 4) % 2.
#include <algorithm>

#include "it_device.h"
#include "it_dot.h"
#include "it_reduce.h"
#include "kernels.h"

namespace itk {
namespace {

IT_DEV float row_reduce_max(float v, float* red, int tid, int waves) {
    v = group_max<64>(v);
    if (waves == 1) return v;
    if ((tid & 63) == 0) red[tid >> 6] = v;
    __syncthreads();
    v = red[0];
    for (int w = 1; w < waves; w++) v = fmaxf(v, red[w]);
    return v;
}

// The split form of four neighbouring elements: their quants times d (the block's scale over the row's power of two).  The
// elements that lie between them in the operand order are two lanes away: of such a pair one lane writes the hi parts of all
// eight, 16 bytes, and the other the lo parts.  i: number of the four in the row.
IT_DEV void put_split(uint32_t quants, float d, int i, int64_t row_at, const SplitOut& o) {
    uint32_t h[4], l[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const float x = (float)(int8_t)(quants >> (8 * k)) * d;
        const _Float16 hi = (_Float16)x;
        const _Float16 lo = (_Float16)(x - (float)hi);
        h[k] = __builtin_bit_cast(uint16_t, hi);
        l[k] = __builtin_bit_cast(uint16_t, lo);
    }
    const bool second = (i >> 1) & 1;             // elements 8 .. 15 of their sixteen
    uint32_t keep[4], give[2], got[2];
#pragma unroll
    for (int k = 0; k < 4; k++) keep[k] = second ? l[k] : h[k];
#pragma unroll
    for (int k = 0; k < 2; k++) {
        give[k] = second ? h[2 * k] | (h[2 * k + 1] << 16) : l[2 * k] | (l[2 * k + 1] << 16);
        got[k] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)give[k], 0x4E, 0xf, 0xf, true);   // lane ^ 2
    }
    const uint32_t other[4] = {got[0] & 0xffffu, got[0] >> 16, got[1] & 0xffffu, got[1] >> 16};
    uint32_t w[4];
#pragma unroll
    for (int k = 0; k < 4; k++) w[k] = second ? other[k] | (keep[k] << 16) : keep[k] | (other[k] << 16);
    const int j0 = 4 * (i & 7), n = 2 * (j0 >> 4) + ((j0 >> 2) & 1);
    *(uint4*)((second ? o.l : o.h) + row_at + 32 * (i >> 3) + 8 * n) = make_uint4(w[0], w[1], w[2], w[3]);
}

// The Q8_0 (and, xh given, the split) form of a row held four neighbouring elements a thread: thread `tid` of T holds
// float4 number tid + T * v.  A block of 32 is eight neighbouring lanes.
template <int T, int NV>
IT_DEV void put_forms(const float4 (&val)[NV], int64_t row, int n4, int tid, const QuantOut& o, float* red) {
    const int64_t base = row * n4;
    float dq[NV];
    uint32_t qq[NV];
    float top = 0.0f;
#pragma unroll
    for (int v = 0; v < NV; v++) {
        const int i = tid + T * v;
        const float4 a = val[v];
        float amax = fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w)));
        amax = group_max<8>(amax);
        const float d = amax / 127.0f;
        const float id = d != 0.0f ? 1.0f / d : 0.0f;
        const float r[4] = {roundf(a.x * id), roundf(a.y * id), roundf(a.z * id), roundf(a.w * id)};
        uint32_t packed = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float c = fminf(fmaxf(r[k], -128.0f), 127.0f);
            const int q = (r[k] != r[k]) ? 0 : (int)c;
            packed |= ((uint32_t)(q & 0xff)) << (8 * k);
        }
        dq[v] = it_f16_to_f32(it_f32_to_f16(d));
        qq[v] = packed;
        if (i < n4) {
            ((uint32_t*)o.quants)[base + i] = packed;
            if ((i & 7) == 0) o.scales[(base + i) >> 3] = dq[v];
            top = fmaxf(top, fabsf(dq[v]));
        }
    }
    if (!o.split.h) return;
    top = row_reduce_max(top, red, tid, T / 64) * 127.0f;
    int ex = 0;
    if (top > 0.0f) (void)frexpf(top, &ex);       // top = m * 2^ex, m in [0.5, 1)
    ex = max(-100, min(100, ex));
    const float down = ldexpf(1.0f, -ex);
    if (tid == 0) o.split.scale[row] = ldexpf(1.0f, ex);
#pragma unroll
    for (int v = 0; v < NV; v++) {
        const int i = tid + T * v;
        if (i >= n4) continue;
        put_split(qq[v], dq[v] * down, i, base * 4, o.split);
    }
}

// ------------------------------------------------------------------ the residual row
// [FINISH ->] x += y [-> rms norm [-> copy] [-> Q8_0, split]]: a block per token, the row in registers throughout.
// NU: picks per token of the FINISH in front (their rows and the gated shared row summed in pick order), 0: no FINISH,
// -1: any number.  y null: the norm alone, so that a row's normed values do not depend on what was issued with it.
template <int NV, int NU>
__global__ __launch_bounds__(256) void residual_row_k(ResidualP p) {
    __shared__ float red[4];
    __shared__ double redd[4];
    const int tid = threadIdx.x, n4 = p.n >> 2;
    const int64_t t = blockIdx.x;
    float4 y[NV], x[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) {
        const int i = tid + 256 * v;
        const int64_t at = t * n4 + min(i, n4 - 1);
        x[v] = ((const float4*)p.x)[at];
        if (NU == 0) y[v] = p.y ? ((const float4*)p.y)[at] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    if constexpr (NU != 0) {
        const int nu = NU > 0 ? NU : p.n_used;
        const float g = fx_sigmoid(p.logit[t]);
        const float* rw = p.rw + t * nu;
#pragma unroll
        for (int v = 0; v < NV; v++) {
            const int i = min(tid + 256 * v, n4 - 1);
            const float4* r = (const float4*)p.rows + t * nu * n4 + i;
            const float4 sh = ((const float4*)p.shared)[t * n4 + i];
            float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
            if constexpr (NU > 0) {
                float4 rr[NU];
#pragma unroll
                for (int e = 0; e < NU; e++) rr[e] = r[(int64_t)e * n4];
#pragma unroll
                for (int e = 0; e < NU; e++) {
                    const float we = rw[e];
                    a.x += we * rr[e].x; a.y += we * rr[e].y; a.z += we * rr[e].z; a.w += we * rr[e].w;
                }
            } else {
                for (int e = 0; e < nu; e++) {
                    const float we = rw[e];
                    const float4 re = r[(int64_t)e * n4];
                    a.x += we * re.x; a.y += we * re.y; a.z += we * re.z; a.w += we * re.w;
                }
            }
            a.x += sh.x * g; a.y += sh.y * g; a.z += sh.z * g; a.w += sh.w * g;
            y[v] = a;
            if (tid + 256 * v < n4) ((float4*)p.y)[t * n4 + i] = a;
        }
    }
    double part = 0.0;
#pragma unroll
    for (int v = 0; v < NV; v++) {
        const int i = tid + 256 * v;
        if (p.y) { x[v].x += y[v].x; x[v].y += y[v].y; x[v].z += y[v].z; x[v].w += y[v].w; }
        if (i < n4) {
            if (p.y) ((float4*)p.x)[t * n4 + i] = x[v];
            part += (double)(x[v].x * x[v].x);
            part += (double)(x[v].y * x[v].y);
            part += (double)(x[v].z * x[v].z);
            part += (double)(x[v].w * x[v].w);
        } else {
            x[v] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
    }
    if (!p.w) return;
    part = wave_sum_f64_tail(part);
    if ((tid & 63) == 63) redd[tid >> 6] = part;
    __syncthreads();
    const float mean = (float)((redd[0] + redd[1] + redd[2] + redd[3]) / (double)p.n);
    const float scale = 1.0f / sqrtf(mean + p.eps);
#pragma unroll
    for (int v = 0; v < NV; v++) {
        const int i = tid + 256 * v;
        if (i >= n4) continue;
        const float4 w = ((const float4*)p.w)[i];
        x[v] = make_float4(x[v].x * scale * w.x, x[v].y * scale * w.y, x[v].z * scale * w.z, x[v].w * scale * w.w);
        ((float4*)p.out)[t * n4 + i] = x[v];
        if (p.copy) ((float4*)p.copy)[t * n4 + i] = x[v];
    }
    if (p.q.quants) put_forms<256, NV>(x, t, n4, tid, p.q, red);
}

// ------------------------------------------------------------------ [silu-mul | sigmoid-mul ->] Q8_0 [-> split]
template <int T, int NV, int OP>
__global__ __launch_bounds__(256) void mul_forms_k(float* __restrict__ a, const float* __restrict__ b, int64_t n_rows, int n4, QuantOut o) {
    __shared__ float red[4];
    const int tid = threadIdx.x % T;
    const int64_t row = (int64_t)blockIdx.x * (256 / T) + threadIdx.x / T;
    if (row >= n_rows) return;    // (whole waves; with T = 256 a block has one row and none leaves)
    float4 v[NV], u[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const int64_t at = row * n4 + min(tid + T * k, n4 - 1);
        v[k] = ((const float4*)a)[at];
        if (OP) u[k] = ((const float4*)b)[at];
    }
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const int i = tid + T * k;
        if (OP == 1) {
            v[k].x = fx_silu(v[k].x) * u[k].x; v[k].y = fx_silu(v[k].y) * u[k].y;
            v[k].z = fx_silu(v[k].z) * u[k].z; v[k].w = fx_silu(v[k].w) * u[k].w;
        } else if (OP == 2) {
            v[k].x *= fx_sigmoid(u[k].x); v[k].y *= fx_sigmoid(u[k].y); v[k].z *= fx_sigmoid(u[k].z); v[k].w *= fx_sigmoid(u[k].w);
        }
        if (i >= n4) v[k] = make_float4(0.f, 0.f, 0.f, 0.f);
        else if (OP) ((float4*)a)[row * n4 + i] = v[k];
    }
    put_forms<T, NV>(v, row, n4, tid, o, red);
}

// the split form alone, from a Q8_0 form that is there (a row of any length)
__global__ __launch_bounds__(256) void split_rows_k(const int8_t* __restrict__ q, const float* __restrict__ sc, int n_in, SplitOut o) {
    __shared__ float red[4];
    const int tid = threadIdx.x, nb = n_in >> 5;
    const int64_t row = blockIdx.x;
    float mx = 0.0f;
    for (int b = tid; b < nb; b += 256) mx = fmaxf(mx, fabsf(sc[row * nb + b]));
    mx = row_reduce_max(mx, red, tid, 4) * 127.0f;
    int ex = 0;
    if (mx > 0.0f) (void)frexpf(mx, &ex);
    ex = max(-100, min(100, ex));
    const float down = ldexpf(1.0f, -ex);
    if (tid == 0) o.scale[row] = ldexpf(1.0f, ex);
    for (int i = tid; i < n_in / 4; i += 256) {
        const uint32_t qq = ((const uint32_t*)(q + row * n_in))[i];
        put_split(qq, sc[row * nb + (i >> 3)] * down, i, row * n_in, o);
    }
}

// ------------------------------------------------------------------ attention's rows before the scores
// Per token: the query half of every head of the projected [q | gate] rows normed and rotated, its gate half copied out,
// the key heads normed, rotated and stored (f32 and, as f16, in the cache), the value heads stored in the cache
// (qwen35.rs:1141-1223): ten ops.  A wave per head, PER neighbouring elements a lane; a rotation's two elements are PER
// whole lanes apart.
template <int PER>
__global__ __launch_bounds__(256) void attn_rows_k(AttnRowsP p) {
    constexpr int HD = 64 * PER;
    const int lane = threadIdx.x & 63;
    const int per_tok = p.n_head + 2 * p.n_kv;
    const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (w >= (int64_t)p.n_tok * per_tok) return;
    const int64_t t = w / per_tok;
    const int h = (int)(w - t * per_tok);
    const bool is_q = h < p.n_head, is_k = !is_q && h < p.n_head + p.n_kv;
    const int kvh = is_q ? 0 : is_k ? h - p.n_head : h - p.n_head - p.n_kv;
    const float* src = is_q ? p.qg + (t * p.n_head + h) * 2 * HD : (is_k ? p.k : p.v) + (t * p.n_kv + kvh) * HD;
    const int e0 = lane * PER;
    float v[PER], g[PER];
    auto load = [&](const float* at, float (&o)[PER]) __attribute__((always_inline)) {
        if constexpr (PER == 4) {
            const float4 a = *(const float4*)at;
            o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w;
        } else if constexpr (PER == 2) {
            const float2 a = *(const float2*)at;
            o[0] = a.x; o[1] = a.y;
        } else {
            o[0] = at[0];
        }
    };
    auto store = [&](float* at, const float (&o)[PER]) __attribute__((always_inline)) {
        if constexpr (PER == 4) *(float4*)at = make_float4(o[0], o[1], o[2], o[3]);
        else if constexpr (PER == 2) *(float2*)at = make_float2(o[0], o[1]);
        else at[0] = o[0];
    };
    load(src + e0, v);
    if (is_q) {
        load(src + HD + e0, g);
        store(p.g + (t * p.n_head + h) * HD + e0, g);
    }
    if (is_q || is_k) {
        const float* nw = is_q ? p.q_w : p.k_w;
        double part = 0.0;
#pragma unroll
        for (int e = 0; e < PER; e++) part += (double)(v[e] * v[e]);
        const double sum = __shfl(wave_sum_f64_tail(part), 63, 64);
        const float mean = (float)(sum / (double)HD);
        const float scale = 1.0f / sqrtf(mean + (is_q ? p.q_eps : p.k_eps));
#pragma unroll
        for (int e = 0; e < PER; e++) v[e] = v[e] * scale * nw[e0 + e];
        const int hl = p.half / PER;               // lanes of one half of the rotated elements
        const int partner = lane < hl ? lane + hl : lane - hl;
        const float2* cs = p.table + (int64_t)(p.pos + t) * p.half;
#pragma unroll
        for (int e = 0; e < PER; e++) {
            const float other = __shfl(v[e], partner & 63, 64);
            if (lane < 2 * hl) {
                const float2 c = cs[(lane < hl ? e0 : e0 - p.half) + e];
                v[e] = lane < hl ? v[e] * c.x - other * c.y : other * c.y + v[e] * c.x;
            }
        }
        store((is_q ? p.q + (t * p.n_head + h) * HD : p.k + (t * p.n_kv + kvh) * HD) + e0, v);
    }
    if (!is_q) {
        uint16_t* d = (is_k ? p.k_slab + p.k_at : p.v_slab + p.v_at) + (t * p.n_kv + kvh) * HD + e0;
        uint16_t o[PER];
#pragma unroll
        for (int e = 0; e < PER; e++) o[e] = it_f32_to_f16(v[e]);
        if constexpr (PER == 4) *(uint2*)d = make_uint2(o[0] | ((uint32_t)o[1] << 16), o[2] | ((uint32_t)o[3] << 16));
        else if constexpr (PER == 2) *(uint32_t*)d = o[0] | ((uint32_t)o[1] << 16);
        else d[0] = o[0];
    }
}

// ------------------------------------------------------------------ softmax -> route
// A wave per token, NE probabilities a lane in registers: softmax (the row is written, as its op would), then a pick a
// round: one reduction for the value, a ballot per register for the lowest expert that has it (src/ops/mod.rs:1191-1216).
template <int NE>
__global__ __launch_bounds__(256) void softmax_route_k(float* __restrict__ x, int n_tok, int n_expert, int n_used,
                                                       int32_t* __restrict__ ids, float* __restrict__ weights) {
    const int lane = threadIdx.x & 63;
    const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= n_tok) return;
    float* row = x + t * n_expert;
    float v[NE];
    float m = -INFINITY;
#pragma unroll
    for (int i = 0; i < NE; i++) {
        const int e = lane + 64 * i;
        v[i] = e < n_expert ? row[e] : -INFINITY;
        m = fmaxf(m, v[i]);
    }
    m = group_max<64>(m);
    float part = 0.0f;
#pragma unroll
    for (int i = 0; i < NE; i++) {
        v[i] = lane + 64 * i < n_expert ? it_expf(v[i] - m) : 0.0f;
        part += v[i];
    }
    const float sum = group_sum<64>(part);
#pragma unroll
    for (int i = 0; i < NE; i++) {
        const int e = lane + 64 * i;
        v[i] = e < n_expert ? v[i] / sum : -1.0f;
        if (e < n_expert) row[e] = v[i];
    }
    float picked_p = 0.0f, s = 0.0f;  // lane r keeps pick r's probability
    int picked_id = 0;
    for (int r = 0; r < n_used; r++) {
        float best = v[0];
#pragma unroll
        for (int i = 1; i < NE; i++) best = fmaxf(best, v[i]);
        best = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, group_max_tail<64>(best)), 63));
        int id = best >= 0.0f ? -1 : r;   // (probabilities that are not numbers: some expert)
#pragma unroll
        for (int i = 0; i < NE; i++) {    // taken and absent experts hold -1
            const unsigned long long has = __ballot(v[i] == best);
            if (id < 0 && has) id = 64 * i + __builtin_ctzll(has);
        }
        s += best;                         // pick order, as the CPU path adds them
        if (lane == r) {
            picked_p = best;
            picked_id = id;
        }
#pragma unroll
        for (int i = 0; i < NE; i++)
            if (lane + 64 * i == id) v[i] = -1.0f;
    }
    if (lane < n_used) {   // (n_used 0: the softmax alone)
        ids[t * n_used + lane] = picked_id;
        weights[t * n_used + lane] = picked_p / fmaxf(s, 6.103515625e-5f);
    }
}

bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

bool residual_row(const ResidualP& p, hipStream_t s) {
    if (p.n_tok <= 0 || p.n_tok > (1 << 24) || p.n % 32 || p.n > 8192 || !al16(p.x) || !al16(p.y)) return false;
    if (p.w && (!al16(p.w) || !al16(p.out) || (p.copy && !al16(p.copy)))) return false;
    if (p.rows && (!al16(p.rows) || !al16(p.shared))) return false;
    const dim3 grid(p.n_tok), block(256);
#define IT_RES(NV, NU) hipLaunchKernelGGL((residual_row_k<NV, NU>), grid, block, 0, s, p)
#define IT_RES_NU(NV)                          \
    do {                                       \
        if (!p.rows) IT_RES(NV, 0);            \
        else if (p.n_used == 4) IT_RES(NV, 4); \
        else if (p.n_used == 8) IT_RES(NV, 8); \
        else if (p.n_used == 10) IT_RES(NV, 10); \
        else IT_RES(NV, -1);                   \
    } while (0)
    if (p.n <= 1024) IT_RES_NU(1);
    else if (p.n <= 2048) IT_RES_NU(2);
    else if (p.n <= 4096) IT_RES_NU(4);
    else IT_RES_NU(8);
#undef IT_RES_NU
#undef IT_RES
    return true;
}

bool mul_forms(float* a, const float* b, int op, int64_t n_rows, int row, const QuantOut& o, hipStream_t s) {
    if (n_rows <= 0 || n_rows > (1 << 30) || row <= 0 || row % 32 || row > 8192 || !al16(a) || (op && !al16(b)) || (reinterpret_cast<uintptr_t>(o.quants) & 3)) return false;
    const int n4 = row / 4;
#define IT_MF(T, NV, OP) hipLaunchKernelGGL((mul_forms_k<T, NV, OP>), dim3((unsigned)((n_rows + 256 / T - 1) / (256 / T))), dim3(256), 0, s, a, b, n_rows, n4, o)
#define IT_MF_OP(T, NV)               \
    do {                              \
        if (op == 1) IT_MF(T, NV, 1); \
        else if (op == 2) IT_MF(T, NV, 2); \
        else IT_MF(T, NV, 0);         \
    } while (0)
    if (row <= 256) IT_MF_OP(64, 1);
    else if (row <= 512) IT_MF_OP(64, 2);
    else if (row <= 1024) IT_MF_OP(64, 4);
    else if (row <= 2048) IT_MF_OP(256, 2);
    else if (row <= 4096) IT_MF_OP(256, 4);
    else IT_MF_OP(256, 8);
#undef IT_MF_OP
#undef IT_MF
    return true;
}

void split_rows(const int8_t* quants, const float* scales, int64_t n_rows, int row, const SplitOut& o, hipStream_t s) {
    if (n_rows <= 0) return;
    hipLaunchKernelGGL(split_rows_k, dim3((unsigned)n_rows), dim3(256), 0, s, quants, scales, row, o);
}

bool attn_rows(const AttnRowsP& p, int head_dim, hipStream_t s) {
    const int per = head_dim / 64;
    if (head_dim % 64 || (per != 1 && per != 2 && per != 4) || p.half % per || p.half <= 0 || 2 * p.half > head_dim) return false;
    if (!al16(p.qg) || !al16(p.q) || !al16(p.g) || !al16(p.k) || !al16(p.v) || ((reinterpret_cast<uintptr_t>(p.k_slab + p.k_at) | reinterpret_cast<uintptr_t>(p.v_slab + p.v_at)) & 7)) return false;
    const int64_t waves = (int64_t)p.n_tok * (p.n_head + 2 * p.n_kv);
    const dim3 grid((unsigned)((waves + 3) / 4)), block(256);
    if (per == 1) hipLaunchKernelGGL(attn_rows_k<1>, grid, block, 0, s, p);
    else if (per == 2) hipLaunchKernelGGL(attn_rows_k<2>, grid, block, 0, s, p);
    else hipLaunchKernelGGL(attn_rows_k<4>, grid, block, 0, s, p);
    return true;
}

bool softmax_route(float* x, int n_tok, int n_expert, int n_used, int32_t* ids, float* weights, hipStream_t s) {
    if (n_tok <= 0 || n_used < 0 || n_used > 16 || n_used > n_expert || n_expert > 1024) return false;
    const dim3 grid((n_tok + 3) / 4), block(256);
    if (n_expert <= 64) hipLaunchKernelGGL(softmax_route_k<1>, grid, block, 0, s, x, n_tok, n_expert, n_used, ids, weights);
    else if (n_expert <= 256) hipLaunchKernelGGL(softmax_route_k<4>, grid, block, 0, s, x, n_tok, n_expert, n_used, ids, weights);
    else if (n_expert <= 512) hipLaunchKernelGGL(softmax_route_k<8>, grid, block, 0, s, x, n_tok, n_expert, n_used, ids, weights);
    else hipLaunchKernelGGL(softmax_route_k<16>, grid, block, 0, s, x, n_tok, n_expert, n_used, ids, weights);
    return true;
}

}  // namespace itk
