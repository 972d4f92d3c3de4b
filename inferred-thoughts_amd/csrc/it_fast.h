// Device pieces shared by the single-token kernels of the fast mode (k_fast.hip) and the layer chain (k_chain.hip):
// 16-byte weight chunks owned by lanes, the matching activation chunks, the per-chunk integer dots, the Q8_0
// quantization of a quad held in registers, and the block-wide router (softmax + top-k of the logits).
//
// A "chunk" is 16 bytes of a repacked weight row: 16 Q8_0 quants (half a block) or 32 NVFP4 nibbles (two
// sub-blocks).  A row of `cpr` chunks is spread over L = min(64, cpr) lanes, CPL = cpr / L chunks each.
#pragma once
#include "it_device.h"
#include "it_dot.h"
#include "it_reduce.h"
#include "kernels.h"

namespace itk {
namespace fastk {

template <int FMT, int CPL> struct XChunks {
    uint4 a[CPL], b[CPL];  // b: second half of an NVFP4 chunk's 32 activations
    float d[CPL];
};
template <int CPL> struct WChunks {
    uint4 w[CPL];
    uint32_t sc[CPL];
};

// activation chunks of lane `sub` from the quantized activation in LDS
template <int FMT, int CPL, int L>
IT_DEV void load_x(XChunks<FMT, CPL>& x, const int8_t* xq, const float* xs, int sub) {
#pragma unroll
    for (int k = 0; k < CPL; k++) {
        const int c = k * L + sub;
        if (FMT == W_Q8_0) {
            x.a[k] = *(const uint4*)(xq + c * 16);
            x.d[k] = xs[c >> 1];
        } else {
            x.a[k] = *(const uint4*)(xq + c * 32);
            x.b[k] = *(const uint4*)(xq + c * 32 + 16);
            x.d[k] = xs[c];
        }
    }
}

template <int FMT, int CPL, int L>
IT_DEV void load_w(WChunks<CPL>& t, const uint8_t* q, const uint8_t* s, int n_in, int64_t row, int sub, bool live) {
    if (!live) {
#pragma unroll
        for (int k = 0; k < CPL; k++) {
            t.w[k] = make_uint4(0, 0, 0, 0);
            t.sc[k] = 0;
        }
        return;
    }
    const uint8_t* rp = q + row * (FMT == W_Q8_0 ? n_in : n_in >> 1);
    const uint16_t* sp = (const uint16_t*)s + row * (n_in >> 5);
#pragma unroll
    for (int k = 0; k < CPL; k++) {
        const int c = k * L + sub;
        {   // read once per token: no reason to keep it in the caches
            typedef unsigned v4u __attribute__((ext_vector_type(4)));
            const v4u nt = __builtin_nontemporal_load((const v4u*)(rp + c * 16));
            t.w[k] = make_uint4(nt.x, nt.y, nt.z, nt.w);
        }
        t.sc[k] = FMT == W_Q8_0 ? sp[c >> 1] : sp[c];
    }
}

// An NVFP4 chunk against the activation through gfx950's own conversions: v_cvt_scalef32_pk_f16_fp4 turns one byte (two
// e2m1 nibbles) into two f16 and v_dot2_f32_f16 multiplies them with two f16 activations, 2 instructions for 2 elements
// where nibbles -> int8 through v_perm_b32 + v_dot4 takes 7 for 4.  The activations are the Q8_0 quants as f16 (exact),
// paired as the nibbles of a byte are (element j with element 8 + j of a 16-element sub-block); every product and sum is
// a multiple of 0.5 below 2^24, so the f32 accumulation is exact and the result is the integer path's, bit for bit.
// The sub-block scales come from v_cvt_pk_f32_fp8 (OCP e4m3; the format's ue4m3 is half of that, and the e2m1 values
// here are half of the integer path's doubled ones: the two factors of 2 cancel; code 0x7f is 0 as in it_ue4m3_to_f32).
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef float f2v __attribute__((ext_vector_type(2)));
struct XN {
    uint32_t p[16];   // sub-block A: pairs (j, 8 + j) j = 0..7, then sub-block B
    float d;
};
// In LDS such an activation is four planes, one of each quarter of a 32-element unit's sixteen pairs: unit u's quarter q is
// 16 bytes at q * (16 * units) + 16 * u, so that the lanes of a load read neighbours.
IT_DEV void load_xn(XN& x, const uint8_t* xh, int units, int u, float d) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const uint4 t = *(const uint4*)(xh + (q * units + u) * 16);
        x.p[4 * q] = t.x;
        x.p[4 * q + 1] = t.y;
        x.p[4 * q + 2] = t.z;
        x.p[4 * q + 3] = t.w;
    }
    x.d = d;
}
// four quants each of elements j .. j + 3 (lo) and 8 + j .. (hi) of a sub-block as f16 pairs, exact: a byte plus 128 in the
// low bits of 1,024's f16, less 1,152
IT_DEV uint4 quant_pairs(uint32_t lo, uint32_t hi) {
    const uint32_t a = lo ^ 0x80808080u, b = hi ^ 0x80808080u;
    auto pair = [&](uint32_t sel) {
        const h2v v = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(b, a, sel) | 0x64006400u) - h2v{(_Float16)1152.0f, (_Float16)1152.0f};
        return __builtin_bit_cast(uint32_t, v);
    };
    return make_uint4(pair(0x0c040c00u), pair(0x0c050c01u), pair(0x0c060c02u), pair(0x0c070c03u));
}
// the chunk of an activation whose int8 quants are in registers: elements 0 .. 15 and 16 .. 31
IT_DEV void make_xn(XN& x, const uint4 a, const uint4 b, float d) {
    const uint4 t[4] = {quant_pairs(a.x, a.z), quant_pairs(a.y, a.w), quant_pairs(b.x, b.z), quant_pairs(b.y, b.w)};
#pragma unroll
    for (int q = 0; q < 4; q++) {
        x.p[4 * q] = t[q].x;
        x.p[4 * q + 1] = t[q].y;
        x.p[4 * q + 2] = t[q].z;
        x.p[4 * q + 3] = t[q].w;
    }
    x.d = d;
}
// the word of the lane two further on in its quad
IT_DEV uint32_t word_ahead2(uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xee, 0xf, 0xf, true); }   // quad_perm [2, 3, 2, 3]
#define IT_FP4_STEP(acc, word, sel, pi) \
    acc = __builtin_amdgcn_fdot2(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, 1.0f, sel), __builtin_bit_cast(h2v, x.p[pi]), acc, false)
// a 32-element chunk's two terms onto `acc`
IT_DEV float dot_xn_add(float acc, const uint4 w, uint32_t sc2, const XN& x) {
    float sa = 0.0f, sb = 0.0f;
    IT_FP4_STEP(sa, w.x, 0, 0); IT_FP4_STEP(sa, w.x, 1, 1); IT_FP4_STEP(sa, w.x, 2, 2); IT_FP4_STEP(sa, w.x, 3, 3);
    IT_FP4_STEP(sa, w.y, 0, 4); IT_FP4_STEP(sa, w.y, 1, 5); IT_FP4_STEP(sa, w.y, 2, 6); IT_FP4_STEP(sa, w.y, 3, 7);
    IT_FP4_STEP(sb, w.z, 0, 8); IT_FP4_STEP(sb, w.z, 1, 9); IT_FP4_STEP(sb, w.z, 2, 10); IT_FP4_STEP(sb, w.z, 3, 11);
    IT_FP4_STEP(sb, w.w, 0, 12); IT_FP4_STEP(sb, w.w, 1, 13); IT_FP4_STEP(sb, w.w, 2, 14); IT_FP4_STEP(sb, w.w, 3, 15);
    const uint32_t sc = sc2 & 0x7f7fu;
    const f2v s2 = __builtin_amdgcn_cvt_pk_f32_fp8((int)sc, false);
    const float dA = (sc & 0x7fu) == 0x7fu ? 0.0f : s2.x, dB = (sc >> 8) == 0x7fu ? 0.0f : s2.y;
    acc += (x.d * dA) * sa;
    acc += (x.d * dB) * sb;
    return acc;
}
IT_DEV float dot_xn(const WChunks<1>& t, const XN& x) { return dot_xn_add(0.0f, t.w[0], t.sc[0], x); }
#undef IT_FP4_STEP

template <int FMT, int CPL>
IT_DEV float dot_chunks(const WChunks<CPL>& t, const XChunks<FMT, CPL>& x) {
    float acc = 0.0f;
#pragma unroll
    for (int k = 0; k < CPL; k++) {
        if (FMT == W_Q8_0) {
            int s = 0;
            s = dot4(t.w[k].x, x.a[k].x, s);
            s = dot4(t.w[k].y, x.a[k].y, s);
            s = dot4(t.w[k].z, x.a[k].z, s);
            s = dot4(t.w[k].w, x.a[k].w, s);
            acc += (float)s * (it_f16_to_f32((uint16_t)t.sc[k]) * x.d[k]);
        } else {
            float tA, tB;
            unit_nvfp4(t.w[k], t.sc[k], x.a[k], x.b[k], x.d[k], &tA, &tB);
            acc += tA;
            acc += tB;
        }
    }
    return acc;
}

// the row's dot, complete in the LAST lane of its L-lane group
template <int L> IT_DEV float reduce_lanes(float v) { return group_sum_tail<L>(v); }

// ------------------------------------------------------------------ activation prologue
// Q8_0 block quantization (naive.rs:652-675) of the quad a thread holds; the 8 threads of a
// 32-block are neighbours in a wave.  Dead threads pass zeros and write nothing.
// Q8_0 (naive.rs:652-675) of one quad of a block of 32 whose largest magnitude is `amax`: four quants a word, and the block's
// step d = amax / 127 before its rounding to f16.  With every wave of a block at it, the single-token stages were bound by
// these instructions: the exact divisions and roundf take 90 of them, this 35, with the same bits (eight chained layers of a
// token 241.7 -> 235.2 us with F32 routers, 227.5 -> 221.0 with Q8_0 ones, a second wait of a stage no longer sleeping included).
//   * amax / 127 as a product with one fused correction (Markstein 1990) is the rounded quotient for every finite float
//     (all 2^31 of them compared);
//   * 1 / d by v_rcp_f32 with one fused Newton step is the rounded reciprocal from 2^-100 to 2^100 (all compared on the card);
//     blocks outside that range, of zeros, infinities or NaN go the long way;
//   * roundf(x) = trunc(x + copysign(0.5 - 2^-25, x)) for |x| <= 127.5 (all compared); the conversion to an integer truncates
//     and makes 0 of NaN.
IT_DEV uint32_t quant_word(float4 v, float amax, float* d_out) {
    constexpr float R127 = 1.0f / 127.0f;
    const float q0 = amax * R127;
    float d = fmaf(fmaf(-127.0f, q0, amax), R127, q0);
    uint32_t packed = 0;
    if (__builtin_expect(d >= 0x1p-100f && d <= 0x1p100f, 1)) {
        const float r0 = __builtin_amdgcn_rcpf(d);
        const float id = fmaf(r0, fmaf(-d, r0, 1.0f), r0);
        const float x[4] = {v.x * id, v.y * id, v.z * id, v.w * id};
        uint32_t q[4];
#pragma unroll
        for (int i = 0; i < 4; i++) asm("v_cvt_i32_f32 %0, %1" : "=v"(q[i]) : "v"(x[i] + copysignf(0x1.fffffep-2f, x[i])));
        packed = __builtin_amdgcn_perm(q[1], q[0], 0x0c0c0400u) | __builtin_amdgcn_perm(q[3], q[2], 0x04000c0cu);
    } else {
        d = amax / 127.0f;
        const float id = d != 0.0f ? 1.0f / d : 0.0f;
        const float r[4] = {roundf(v.x * id), roundf(v.y * id), roundf(v.z * id), roundf(v.w * id)};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float c = fminf(fmaxf(r[i], -128.0f), 127.0f);
            const int q = (r[i] != r[i]) ? 0 : (int)c;
            packed |= ((uint32_t)(q & 0xff)) << (8 * i);
        }
    }
    *d_out = d;
    return packed;
}
IT_DEV float quad_amax(float4 v) { return fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))); }
IT_DEV void quant_quad(float4 v, bool live, int qi, int8_t* xq, float* xs) {
    const float amax = group_max<8>(quad_amax(v));
    if (!live) return;
    float d;
    *(uint32_t*)(xq + qi * 4) = quant_word(v, amax, &d);
    if ((qi & 7) == 0) xs[qi >> 3] = it_f16_to_f32(it_f32_to_f16(d));
}

IT_DEV double quad_sumsq(float4 v) {
    double s = (double)(v.x * v.x);
    s += (double)(v.y * v.y);
    s += (double)(v.z * v.z);
    s += (double)(v.w * v.w);
    return s;
}

// ------------------------------------------------------------------ router in a block
// softmax over n_expert logits, the n_used largest by (probability descending, id ascending),
// weights = picked probabilities over their sum in pick order (src/ops/mod.rs:1191-1216,
// naive.rs:362-376).  Every thread of the block calls this.  After it returns, ids[r] and
// wts[r] (LDS, 16 entries, zero past n_used) hold pick r and its probability; the return
// value is the weights' denominator, the same in every thread.
// n_expert <= 4 * THREADS, n_used <= 16.
//
// Selection.  A key is one of the n_used largest only if fewer than n_used of the block's half waves hold a larger one: that
// leaves some fifteen of 512 keys, which are put side by side and ranked against one another.  (Ranking every key among the 64 of
// its wave and then each wave's best against one another is 96 dependent compare-and-count pairs a thread, 17 cycles each: 1.4 us
// of a decode layer's 28 where this takes 0.77.)
// Probabilities are non-negative, so their bit patterns order like the values; a pick is
// compared as the 64-bit key (probability bits, ~id): larger key = earlier pick, keys are
// unique, and key 0 is no key.
template <int THREADS, int PER_THREAD> struct TopLds {
    unsigned n;                                                       // candidates
    __attribute__((aligned(16))) unsigned best[THREADS / 32];        // largest value of each half wave
    __attribute__((aligned(16))) unsigned long long cand[PER_THREAD * THREADS];
};
template <int THREADS> struct RouteLds {
    float redf[2 * (THREADS / 64)];
    TopLds<THREADS, 4> top;
};

IT_DEV unsigned long long route_key(float p, int e) {
    return ((unsigned long long)__float_as_uint(p) << 32) | (unsigned long long)(~(unsigned)e);
}

template <int CTRL, int ROWS> IT_DEV unsigned dpp_umax(unsigned v) {
    return max(v, (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, ROWS, 0xf, false));
}
// the half waves' largest values; a barrier of the block follows, then top_pick.  (Every thread calls both.)
template <int THREADS, int PER_THREAD>
IT_DEV void top_begin(TopLds<THREADS, PER_THREAD>& sh, unsigned largest) {
    largest = dpp_umax<0xB1, 0xf>(largest);        // lane ^ 1
    largest = dpp_umax<0x4E, 0xf>(largest);        // lane ^ 2
    largest = dpp_umax<0x141, 0xf>(largest);       // mirrored in 8
    largest = dpp_umax<0x140, 0xf>(largest);       // in 16
    largest = dpp_umax<0x142, 0xa>(largest);       // lane 15 of rows 0 and 2 into rows 1 and 3
    if ((threadIdx.x & 31) == 16) sh.best[threadIdx.x >> 5] = largest;
    if (threadIdx.x == 0) sh.n = 0;
}
// put(rank, key) for the n_used largest of the block's keys (key[k], k < K; 0: none); holds a barrier, and one follows before what
// put writes is read
template <int THREADS, int PER_THREAD, int N, class Put>
IT_DEV void top_pick(TopLds<THREADS, PER_THREAD>& sh, const unsigned long long (&key)[N], int K, int n_used, Put put) {
    static_assert(N <= PER_THREAD);
    const int tid = threadIdx.x, lane = tid & 63;
    unsigned best[THREADS / 32];
#pragma unroll
    for (int i = 0; i < THREADS / 128; i++) {
        const uint4 q = ((const uint4*)sh.best)[i];
        best[4 * i] = q.x, best[4 * i + 1] = q.y, best[4 * i + 2] = q.z, best[4 * i + 3] = q.w;
    }
#pragma unroll
    for (int k = 0; k < N; k++) {
        if (k >= K) break;
        const unsigned mine = (unsigned)(key[k] >> 32);
        int above0 = 0, above1 = 0;
#pragma unroll
        for (int i = 0; i < THREADS / 32; i += 2) {
            above0 += best[i] > mine ? 1 : 0;
            above1 += best[i + 1] > mine ? 1 : 0;
        }
        const bool in = key[k] != 0ull && above0 + above1 < n_used;
        const unsigned long long all = __ballot(in);
        if (all == 0ull) continue;
        unsigned at = 0;
        if (lane == 0) at = __hip_atomic_fetch_add(&sh.n, (unsigned)__popcll(all), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        at = __builtin_amdgcn_readfirstlane(at) + __builtin_amdgcn_mbcnt_hi((unsigned)(all >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)all, 0));
        if (in) sh.cand[at] = key[k];
    }
    __syncthreads();
    // eight threads a candidate
    const int n = (int)sh.n, part = tid & 7;
    for (int c0 = 0; c0 < n; c0 += THREADS / 8) {
        const int c = c0 + (tid >> 3);
        const unsigned long long me = c < n ? sh.cand[c] : ~0ull;
        int rank = 0;
        for (int j = part; j < n; j += 8) rank += sh.cand[j] > me ? 1 : 0;
        rank += __builtin_amdgcn_update_dpp(0, rank, 0xB1, 0xf, 0xf, true);
        rank += __builtin_amdgcn_update_dpp(0, rank, 0x4E, 0xf, 0xf, true);
        rank += __builtin_amdgcn_update_dpp(0, rank, 0x141, 0xf, 0xf, true);
        if (part == 0 && c < n && rank < n_used) put(rank, me);
    }
}

// this thread's logits (up to four experts, THREADS apart): fetched ahead of the activation prologue so that the
// two loads share one trip to memory
template <int THREADS>
__device__ __forceinline__ void route_fetch(const float* logits, int n_expert, float l[4]) {
    const int K = (n_expert + THREADS - 1) / THREADS;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int e = threadIdx.x + k * THREADS;
        l[k] = (k < K && e < n_expert) ? logits[e] : -INFINITY;
    }
}

// EXACT: the CPU path's exponentials (etab: their table, in LDS) and its sum in the order of the experts (terms: n_expert floats of
// LDS, 16-byte aligned), a chain of eight cycles an expert in one wave.
template <int THREADS, bool EXACT = false>
__device__ __forceinline__ float block_route(const float l[4], int n_expert, int n_used, RouteLds<THREADS>& sh, int* ids, float* wts,
                                             const uint64_t* etab = nullptr, float* terms = nullptr) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    constexpr int NW = THREADS / 64;
    const int K = (n_expert + THREADS - 1) / THREADS;  // experts per thread that can be live
    float m = -INFINITY;
#pragma unroll
    for (int k = 0; k < 4; k++) m = fmaxf(m, l[k]);
    if (tid < 16) wts[tid] = 0.0f;
    m = group_max_tail<64>(m);
    if (lane == 63) sh.redf[wave] = m;
    __syncthreads();
    m = sh.redf[0];
#pragma unroll
    for (int i = 1; i < NW; i++) m = fmaxf(m, sh.redf[i]);
    float v[4];
    float part = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int e = tid + k * THREADS;
        if constexpr (EXACT) {
            if (k >= K) break;
            v[k] = it_expf_by(l[k] - m, etab);
            if (e < n_expert) terms[e] = v[k];
        } else {
            v[k] = (k < K && e < n_expert) ? fx_expf(l[k] - m) : 0.0f;
            part += v[k];
        }
    }
    float sum = 0.0f;
    if constexpr (EXACT) {
        __syncthreads();
        if (wave == 0) sh.redf[NW] = fold_terms(terms, n_expert);   // (every lane: the same reads)
        __syncthreads();
        sum = sh.redf[NW];
    } else {
        part = group_sum_tail<64>(part);
        if (lane == 63) sh.redf[NW + wave] = part;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NW; i++) sum += sh.redf[NW + i];
    }
    unsigned long long key[4];
    unsigned largest = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int e = tid + k * THREADS;
        if (!EXACT || k < K) v[k] = v[k] / sum;
        key[k] = (k < K && e < n_expert) ? route_key(v[k], e) : 0ull;
        largest = max(largest, (unsigned)(key[k] >> 32));
    }
    top_begin(sh.top, largest);
    __syncthreads();
    top_pick(sh.top, key, K, n_used, [&](int rank, unsigned long long pick) {
        ids[rank] = (int)~(unsigned)(pick & 0xffffffffull);
        wts[rank] = __uint_as_float((unsigned)(pick >> 32));
    });
    __syncthreads();
    float s = 0.0f;
#pragma unroll
    for (int r4 = 0; r4 < 4; r4++) {
        const float4 w = ((const float4*)wts)[r4];
        s += w.x;
        s += w.y;
        s += w.z;
        s += w.w;
    }
    return fmaxf(s, 6.103515625e-5f);
}

}  // namespace fastk
}  // namespace itk
