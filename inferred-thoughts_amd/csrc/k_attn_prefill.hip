// Causal attention for a batch of queries (prefill) on the f16 matrix cores, one pass over the keys.
//
// Same function as /root/reference src/ops/naive.rs:137-203 (scores, softmax, weighted values per
// head; query i of a batch of n_q sees positions 0 .. n_pos - n_q + i), computed tile by tile with a
// running maximum and sum per query instead of a full score row.  Fast mode only: the sums are not
// in the CPU path's order.
//
// A block owns 128 query rows of one KV head: 128 / G tokens x the G query heads that share the head.
// It walks the keys in tiles of 64; a tile's K and V are brought to LDS as stored ([key][dim], f16) by loads that go
// straight there, two tiles of each, and serve all 128 rows.  Each wave owns 32 rows and forms
//     S^T = K Q^T   (32 keys x 32 queries per MFMA tile, A = K from LDS, B = Q from registers)
//     O^T = V^T P^T (32 dims x 32 queries per MFMA tile, A = V^T from LDS, B = P from registers)
// so a lane holds, for ITS query (column l % 32), 16 of the 32 keys of a score tile and 16 of the 32
// dims of an output tile: the running maximum, the rescaling and the final division stay inside
// the lane (one exchange with lane l ^ 32), and the probabilities go from the score accumulators
// to the next MFMA's B operand without leaving the registers (the k order of an MFMA is free as
// long as both operands agree: lane group g's eight probabilities of step j are keys
// 16 j + 4 g + {0..3} and 8 more; V is read at those keys by the transposing LDS read, which gives
// lane i of 16 four keys' value of column i).
// The rows of 2 * HD bytes lie whole in LDS; which 16-byte piece of a row lies where is turned by the row, for K so that
// rows read together hit different banks, for V so that eight keys' 64-byte blocks do (swap_k, swap_v).
// The query is scaled by scale * log2(e) and split into an f16 pair (hi + lo, 22 bits kept); K, V
// are f16 in the cache; probabilities are rounded to f16 (relative 2^-11 each, unbiased).
//
// MFMA operand layout (32x32x16, f16): lane l supplies 8 k values of row (l % 32), k group l / 32,
// for A and for B; it receives D for column l % 32 and rows 8 * (i / 4) + 4 * (l / 32) + i % 4.
#include "it_device.h"
#include "it_dot.h"
#include "it_launch.h"
#include "kernels.h"

#include <algorithm>

namespace itk {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef short s4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s4 ls4;
typedef __attribute__((address_space(3))) uint8_t* lptr;
constexpr int KT = 64;          // keys per tile
constexpr float GROW = 8.0f;    // the running maximum follows when the scores pass it by more than this (log2): probabilities stay below 2^8

// the 16-byte piece of row `key` that lies at piece p of its row in LDS (and the other way round)
template <int HD>
IT_DEV int swap_k(int key) { return HD >= 128 ? key & 15 : (key >> 1) & 7; }
template <int HD>
IT_DEV int swap_v(int key) { return HD == 256 ? (key & 7) << 2 : HD == 128 ? (key & 3) << 2 : ((key >> 1) & 1) << 2; }

// formed here, not later where it is first read
IT_DEV void here(float& x, h8& v) {
    uint4 t = __builtin_bit_cast(uint4, v);
    asm volatile("" : "+v"(x), "+v"(t.x), "+v"(t.y), "+v"(t.z), "+v"(t.w));
    v = __builtin_bit_cast(h8, t);
}

constexpr float NONE = -1e30f;  // the maximum of a row that has seen no key

// Partial results of n_split shares: the sums [token][head][share][HD], then maximum (log2) and weight of each.
IT_DEV float* part_stats(float* part, const AttnArgs& a, int hd) { return part + (int64_t)a.n_q * a.n_head * gridDim.z * hd; }

template <int V>
struct Is { static constexpr int value = V; };

// What bounds it: the matrix cores' instructions (96 per wave and tile at head_dim 256: 64 for the scores, the query being a
// pair, 32 for the values), with one wave on each SIMD, since a row's query pair and sums take about 300 registers.  So
// nothing else may stand between them: the softmax of a tile runs in the shadow of the next tile's scores, a tile's loads
// are asked for one tile ahead, and there is one barrier per tile.  5,700 queries, 16 heads of 256 on 2: 0.42 ms, 960 TFLOP/s
// as issued (0.68 ms when a tile was fetched through registers, V turned on its way into LDS, and softmax and products
// took turns between two barriers); 30,000 in four batches: 10.3 ms (16.9).
template <int HD, int G>
__global__ __launch_bounds__(256) void attend_prefill_k(AttnArgs a, float* __restrict__ out, float* __restrict__ part) {
    constexpr int QT = 128 / G;                     // tokens per block
    constexpr int NS = HD / 16;                     // k steps of a score tile
    constexpr int ND = HD / 32;                     // output tiles along the head dimension
    constexpr int P = HD / 8;                       // 16-byte pieces of a row
    constexpr int NL = HD / 32;                     // loads of a wave per tile of K, and of V (1,024 bytes each)
    constexpr int RL = 512 / HD;                    // rows of one
    constexpr int TILE = KT * HD * 2;               // bytes
    constexpr int V_AT = 2 * TILE;
    extern __shared__ __align__(1024) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, g = lane >> 5;
    const int n_qt = (a.n_q + QT - 1) / QT;
    const int qt = n_qt - 1 - (int)blockIdx.x;      // the longest rows first
    const int kvh = blockIdx.y;
    const int row = 32 * w + r;
    const int token = qt * QT + row / G, head = kvh * G + row % G;
    const bool valid = token < a.n_q;
    const int base_pos = a.n_pos - a.n_q;
    const int pos = valid ? base_pos + token : 0x7fffffff;
    const int qdim = a.n_head * HD;

    const int first_pos = base_pos + qt * QT;                            // smallest position of the block
    const int last_pos = base_pos + min(a.n_q, (qt + 1) * QT) - 1;       // largest
    const int all_kt = last_pos / KT + 1;
    const int kt0 = (int)((int64_t)all_kt * blockIdx.z / gridDim.z);     // this block's share of the tiles
    const int n_kt = (int)((int64_t)all_kt * (blockIdx.z + 1) / gridDim.z);
    const int row_at = token * a.n_head + head;
    if (kt0 == n_kt) {                              // more shares than tiles: weight 0 for the merge
        if (valid && g == 0) *(float2*)(part_stats(part, a, HD) + ((int64_t)row_at * gridDim.z + blockIdx.z) * 2) = make_float2(NONE, 0.0f);
        return;
    }
    const uint32_t at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lptr)lds);

    const int lrow = w * 16 + lane / P;             // this lane's row of the wave's first load
    auto ask_k = [&](int kt, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NL; i++) {
            const int key = lrow + i * RL;
            const uint16_t* from = a.k + kvh * HD + (int64_t)min(kt * KT + key, a.n_pos - 1) * a.kv_dim + 8 * ((lane % P) ^ swap_k<HD>(key));
            to_lds(from, at + buf * TILE + (w * NL + i) * 1024);
        }
    };
    auto ask_v = [&](int kt, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NL; i++) {
            const int key = lrow + i * RL;
            const uint16_t* from = a.v + kvh * HD + (int64_t)min(kt * KT + key, a.n_pos - 1) * a.kv_dim + 8 * ((lane % P) ^ swap_v<HD>(key));
            to_lds(from, at + V_AT + buf * TILE + (w * NL + i) * 1024);
        }
    };
    ask_k(kt0, 0);
    ask_v(kt0, 0);
    ask_k(kt0 + 1, 1);                                    // (past the end: the last key again, never read)

    // this lane's query row, scaled, as an f16 pair
    h8 qh[NS], ql[NS];
    {
        const float qs = a.scale * 1.4426950408889634f;
        const float* qrow = a.q + (int64_t)min(token, a.n_q - 1) * qdim + head * HD + 8 * g;
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const float4 x0 = *(const float4*)(qrow + 16 * s), x1 = *(const float4*)(qrow + 16 * s + 4);
            const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float v = valid ? x[e] * qs : 0.0f;
                const _Float16 hi = (_Float16)v;
                qh[s][e] = hi;
                ql[s][e] = (_Float16)(v - (float)hi);
            }
        }
    }

    const uint8_t* const k_row = lds + r * HD * 2;
    const int k_swap = g ^ swap_k<HD>(r);           // piece 2 s + g of row r (and of row r + 32)
    auto k_frag = [&](int buf, int s, int kk) __attribute__((always_inline)) {
        return *(const h8*)(k_row + buf * TILE + kk * 32 * HD * 2 + (((2 * s) ^ k_swap) << 4));
    };
    const int v_key = 4 * g + ((lane & 15) >> 2);   // key this lane names of the eight of a transposing read
    const uint8_t* const v_row = lds + V_AT + v_key * HD * 2 + ((lane >> 4) & 1) * 32 + (lane & 3) * 8;
    const int v_swap = swap_v<HD>(v_key) << 4;
    auto v_frag = [&](int buf, int j, int dt) __attribute__((always_inline)) {
        const uint8_t* const p = v_row + buf * TILE + 16 * j * HD * 2 + ((64 * dt) ^ v_swap);
        const s4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ls4*)p);
        const s4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ls4*)(p + 8 * HD * 2));
        typedef short s8 __attribute__((ext_vector_type(8)));
        return __builtin_bit_cast(h8, s8(__builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7)));
    };

    v16f o[ND];
#pragma unroll
    for (int dt = 0; dt < ND; dt++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[dt][i] = 0.0f;
    float m = NONE, l = 0.0f;

    // a row sees keys up to its own position
    auto mask = [&](v16f (&sc)[2], int kt) __attribute__((always_inline)) {
        if (kt * KT + KT - 1 > first_pos) {         // some row of the block cannot see the whole tile
#pragma unroll
            for (int kk = 0; kk < 2; kk++)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int key = kt * KT + 32 * kk + 8 * (i >> 2) + 4 * g + (i & 3);
                    if (key > pos) sc[kk][i] = -INFINITY;
                }
        }
    };

    // Tile kt, whose scores are sc: its softmax, beside it (NEXT) tile kt + 1's scores to sn, then its values.
    // B: the half of LDS that holds tile kt.
    auto tile = [&](auto next, auto half, int kt, v16f (&sc)[2], v16f (&sn)[2]) __attribute__((always_inline)) {
        constexpr bool NEXT = decltype(next)::value;
        constexpr int B = decltype(half)::value;
        __builtin_amdgcn_s_waitcnt(0x0070);         // tile kt's V and tile kt + 1's K have landed (vmcnt 0), and this wave has what it read (lgkmcnt 0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (NEXT) {                                 // (every wave is past tile kt's K and tile kt - 1's V)
            ask_v(kt + 1, B ^ 1);
            ask_k(kt + 2, B);
        }
        float mt = -INFINITY, alpha = 1.0f, psum = 0.0f;
        h8 pf[4], kf[2][2], vf[2][4];
        if (NEXT) {
            kf[0][0] = k_frag(B ^ 1, 0, 0);
            kf[0][1] = k_frag(B ^ 1, 0, 1);
#pragma unroll
            for (int kk = 0; kk < 2; kk++)
#pragma unroll
                for (int i = 0; i < 16; i++) sn[kk][i] = 0.0f;
        }
#pragma unroll
        for (int s = 0; s < NS; s++) {
            if (NEXT) {
                if (s + 1 < NS) {
                    kf[(s + 1) & 1][0] = k_frag(B ^ 1, s + 1, 0);
                    kf[(s + 1) & 1][1] = k_frag(B ^ 1, s + 1, 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
                sn[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[s & 1][0], qh[s], sn[0], 0, 0, 0);
                sn[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[s & 1][1], qh[s], sn[1], 0, 0, 0);
                sn[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[s & 1][0], ql[s], sn[0], 0, 0, 0);
                sn[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[s & 1][1], ql[s], sn[1], 0, 0, 0);
            }
            constexpr int NM = NS / 4, NE = NS / 2;     // steps that take the maximum, that form the probabilities
            if (s < NM) {
#pragma unroll
                for (int e = s * (32 / NM); e < (s + 1) * (32 / NM); e++) mt = fmaxf(mt, sc[e >> 4][e & 15]);
                if (s == NM - 1) {
                    mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
                    const float m_new = mt > m + GROW ? mt : m;   // (NONE while the row has seen no key: its probabilities are 0)
                    alpha = __builtin_amdgcn_exp2f(m - m_new);
                    m = m_new;
                }
            } else if (s < NM + NE) {
#pragma unroll
                for (int e = (s - NM) * (32 / NE); e < (s - NM + 1) * (32 / NE); e++) {
                    const float p = __builtin_amdgcn_exp2f(sc[e >> 4][e & 15] - m);
                    psum += p;
                    pf[e >> 3][e & 7] = (_Float16)p;
                }
                here(psum, pf[(s - NM) * 4 / NE]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        l = l * alpha + psum;
        if (__any(alpha != 1.0f)) {
#pragma unroll
            for (int dt = 0; dt < ND; dt++)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    float x = o[dt][i], t;
                    asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\tv_accvgpr_write_b32 %0, %1" : "+a"(x), "=&v"(t) : "v"(alpha));
                    o[dt][i] = x;
                }
            asm volatile("s_nop 4");
        }
        constexpr int W = ND < 4 ? ND : 4, NG = 4 * ND / W;   // output tiles of a group, groups: group q is step q % 4 of tiles W (q / 4) ...
#pragma unroll
        for (int i = 0; i < W; i++) vf[0][i] = v_frag(B, 0, i);
#pragma unroll
        for (int q = 0; q < NG; q++) {
            if (q + 1 < NG) {
#pragma unroll
                for (int i = 0; i < W; i++) vf[(q + 1) & 1][i] = v_frag(B, (q + 1) & 3, W * ((q + 1) >> 2) + i);
                __builtin_amdgcn_sched_barrier(0);  // (ahead of the products, not between)
            }
#pragma unroll
            for (int i = 0; i < W; i++)
                o[W * (q >> 2) + i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[q & 1][i], pf[q & 3], o[W * (q >> 2) + i], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (NEXT) mask(sn, kt + 1);
    };

    v16f s0[2], s1[2];
    __builtin_amdgcn_s_waitcnt(0x0f70);             // tile 0 has landed
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int kk = 0; kk < 2; kk++) {
#pragma unroll
        for (int i = 0; i < 16; i++) s0[kk][i] = 0.0f;
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const h8 kf = k_frag(0, s, kk);
            s0[kk] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qh[s], s0[kk], 0, 0, 0);
            s0[kk] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, ql[s], s0[kk], 0, 0, 0);
        }
    }
    mask(s0, kt0);
    int kt = kt0;
    for (; kt + 2 < n_kt; kt += 2) {
        tile(Is<1>(), Is<0>(), kt, s0, s1);
        tile(Is<1>(), Is<1>(), kt + 1, s1, s0);
    }
    if (kt + 1 < n_kt) {
        tile(Is<1>(), Is<0>(), kt, s0, s1);
        tile(Is<0>(), Is<1>(), kt + 1, s1, s0);
    } else {
        tile(Is<0>(), Is<0>(), kt, s0, s1);
    }

    l += __shfl_xor(l, 32, 64);
    if (valid) {
        const int64_t at_part = (int64_t)row_at * gridDim.z + blockIdx.z;
        if (part && g == 0) *(float2*)(part_stats(part, a, HD) + at_part * 2) = make_float2(m, l);
        const float inv = part ? 1.0f : 1.0f / l;
        float* orow = (part ? part + at_part * HD : out + (int64_t)token * qdim + head * HD) + 4 * g;
#pragma unroll
        for (int dt = 0; dt < ND; dt++)
#pragma unroll
            for (int i4 = 0; i4 < 4; i4++)
                *(float4*)(orow + 32 * dt + 8 * i4) = make_float4(o[dt][4 * i4] * inv, o[dt][4 * i4 + 1] * inv,
                                                                 o[dt][4 * i4 + 2] * inv, o[dt][4 * i4 + 3] * inv);
    }
}

// The shares' sums, weighted and divided: four dims of a row per thread.  Memory: each partial is read once.
__global__ __launch_bounds__(256) void prefill_merge_k(const float* __restrict__ part, int64_t rows, int n_split, int hd4, float* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, row = i / hd4;
    if (row >= rows) return;
    const float2* const st = (const float2*)(part + rows * n_split * hd4 * 4) + row * n_split;
    const float4* const p = (const float4*)part + row * n_split * hd4 + i % hd4;
    float m = st[0].x;
    for (int z = 1; z < n_split; z++) m = fmaxf(m, st[z].x);
    float l = 0.0f;
    float4 o = make_float4(0, 0, 0, 0);
    for (int z = 0; z < n_split; z++) {
        const float2 t = st[z];
        if (t.y <= 0.0f) continue;                  // an empty share's sums were never written
        const float w = __builtin_amdgcn_exp2f(t.x - m);
        const float4 x = p[(int64_t)z * hd4];
        l += w * t.y;
        o.x += w * x.x; o.y += w * x.y; o.z += w * x.z; o.w += w * x.w;
    }
    const float inv = 1.0f / l;
    ((float4*)out)[i] = make_float4(o.x * inv, o.y * inv, o.z * inv, o.w * inv);
}

template <int HD, int G>
bool launch_prefill(const AttnArgs& a, int n_split, float* part, float* out, hipStream_t s) {
    constexpr int QT = 128 / G;
    const size_t lds = (size_t)4 * KT * HD * sizeof(uint16_t);   // two tiles of K, two of V
    if (!lds_allowed<&attend_prefill_k<HD, G>>(lds)) return false;
    hipLaunchKernelGGL((attend_prefill_k<HD, G>), dim3((a.n_q + QT - 1) / QT, a.n_head_kv, n_split), dim3(256), lds, s, a, out,
                       n_split > 1 ? part : nullptr);
    if (n_split > 1) {
        const int64_t rows = (int64_t)a.n_q * a.n_head;
        hipLaunchKernelGGL(prefill_merge_k, dim3((unsigned)((rows * (HD / 4) + 255) / 256)), dim3(256), 0, s, part, rows, n_split, HD / 4, out);
    }
    return true;
}

template <int HD>
bool launch_prefill_g(const AttnArgs& a, int n_split, float* part, float* out, hipStream_t s) {
    switch (a.n_head / a.n_head_kv) {
        case 1: return launch_prefill<HD, 1>(a, n_split, part, out, s);
        case 2: return launch_prefill<HD, 2>(a, n_split, part, out, s);
        case 4: return launch_prefill<HD, 4>(a, n_split, part, out, s);
        case 8: return launch_prefill<HD, 8>(a, n_split, part, out, s);
        case 16: return launch_prefill<HD, 16>(a, n_split, part, out, s);
        default: return false;
    }
}

}  // namespace

// whether the one-pass kernel takes the shape (then the split kernels' scratch is not needed)
bool attend_prefill_takes(const AttnArgs& a, const float* out) {
    if (a.n_pos_dyn || a.n_q <= 16 || a.n_pos < a.n_q || a.n_head_kv <= 0 || a.n_head % a.n_head_kv) return false;
    if (a.kv_dim % 8 || (reinterpret_cast<uintptr_t>(a.k) & 15) || (reinterpret_cast<uintptr_t>(a.v) & 15) ||
        (reinterpret_cast<uintptr_t>(a.q) & 15) || (reinterpret_cast<uintptr_t>(out) & 15))
        return false;
    const int G = a.n_head / a.n_head_kv;
    if (G != 1 && G != 2 && G != 4 && G != 8 && G != 16) return false;
    return a.head_dim == 64 || a.head_dim == 128 || a.head_dim == 256;
}

// Shares the keys are cut into: a batch whose blocks leave compute units idle gets as many as fill them once, as long as a
// share keeps PREFILL_SHARE tiles (2 to 8 measure the same; a tile is 2 us, the merge's launch 5).  16,000 tokens in passes of
// 512, two layers: 44.9 ms with whole rows on 64 of 256 compute units, 38.0 so.
constexpr int PREFILL_SHARE = 4, CUS = 256;
int attend_prefill_splits_max(const AttnArgs& a) {
    const int qt = 128 / (a.n_head / a.n_head_kv);
    return (int)std::max<int64_t>(1, CUS / ((int64_t)((a.n_q + qt - 1) / qt) * a.n_head_kv));
}
int attend_prefill_splits(const AttnArgs& a) {
    return std::max(1, std::min(attend_prefill_splits_max(a), (a.n_pos + KT - 1) / KT / PREFILL_SHARE));
}
// floats of partial results, at any n_pos (so that a context that grows does not make them grow)
size_t attend_prefill_floats(const AttnArgs& a) {
    const int n = attend_prefill_splits_max(a);
    return n > 1 ? (size_t)a.n_q * a.n_head * n * (a.head_dim + 2) : 0;
}

// false: not a shape this kernel takes (the caller uses the split kernels)
bool attend_prefill(const AttnArgs& a, int n_split, float* part, float* out, hipStream_t s) {
    if (!attend_prefill_takes(a, out)) return false;
    switch (a.head_dim) {
        case 64: return launch_prefill_g<64>(a, n_split, part, out, s);
        case 128: return launch_prefill_g<128>(a, n_split, part, out, s);
        case 256: return launch_prefill_g<256>(a, n_split, part, out, s);
        default: return false;
    }
}

}  // namespace itk
