// Attention of one to sixteen queries over the f16 cache (decode, verify batches), split over the keys, on the f16 matrix cores.
//
// Same function as /root/reference src/ops/naive.rs:420-466 (query i of a batch of n_q sees positions 0 .. n_pos - n_q + i),
// fast mode: the sums are not in the CPU path's order.  The live context is cut into n_split equal ranges of keys; a block
// owns one KV head (the G query heads of it), its queries and one range, and leaves its sums, its maximum and its weight
// for the merge ([HD sums][m][l] per query, head and range).
//
// A wave forms, 32 keys at a time (a slice), S^T = K Q^T and O^T = V^T P^T.  A query takes 16 columns: its heads as the high
// f16 halves of the scaled query in columns 0 .. 7, the low halves in 8 .. 15 (one product carries both, a lane move within a
// row of 16 lanes adds them).  A lane has, for its column, some of the slice's keys and some of every output tile's dims, so the
// softmax needs one or two exchanges and the probabilities go to the next product without leaving the registers (the k order
// of a product is free as long as both operands agree).
// K and V go from memory straight to LDS as stored ([key][dim]; which 16-byte piece of a row lies where is turned by the row
// so that rows read together hit different banks); V is read by the transposing LDS read, which gives lane i of 16 four
// keys' value of column i.
//
// What bounds it: short contexts the chain of trips to memory and LDS and the number of instructions a wave issues between
// them (four cycles each), long ones memory.  So one query's waves share nothing but the query: each walks a quarter of the
// range with its own slice of K and of V in LDS, asked for again as soon as it has been read, and the four results are added at
// the end.  Calls one after another on the same operands, with the merge, 16 query heads of 256 on 2 KV heads: 8.3 us at 1,024
// positions, 9.2 at 5,800, 15.6 at 32,000 (4.2 TB/s); five queries at 5,431: 15.0; on 4 KV heads at 31,000: 22.8 (5.6 TB/s); 32 heads of
// 128 on 4 at 30,000: 14.8.  (9.9, 10.3, 21.2, 16.1, 32.7 and 21.5 with K and V through registers, V turned on its way into LDS, a tile
// of 64 keys a block at a time, every wave forming the same scores.)
#include <algorithm>
#include <type_traits>

#include "it_device.h"
#include "it_dot.h"
#include "it_launch.h"
#include "it_reduce.h"
#include "kernels.h"

namespace itk {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef short s4 __attribute__((ext_vector_type(4)));
typedef short s8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s4 ls4;
constexpr int SL = 32;          // keys of a slice
constexpr float NONE = -1e30f;  // the maximum of a column that has seen no key
constexpr float GROW = 8.0f;    // the running maximum follows when the scores pass it by more than this (log2)

// What a row's piece numbers are XORed with in LDS.  Each takes bits of the key's number, so that turn(a + b) is
// turn(a) ^ turn(b) where a and b share no bit.
template <int HD> IT_DEV constexpr int turn_k(int key) { return HD >= 128 ? key & 15 : (key >> 1) & 7; }
template <int HD> IT_DEV constexpr int turn_v16(int key) { return HD == 256 ? (key & 15) << 1 : HD == 128 ? (key & 7) << 1 : (key & 3) << 1; }   // 16-dim tiles
template <int HD> IT_DEV constexpr int turn_v32(int key) { return HD == 256 ? (key & 7) << 2 : HD == 128 ? (key & 3) << 2 : ((key >> 1) & 1) << 2; }   // 32-dim tiles

template <int HD> IT_DEV constexpr int turn_o(int row) { return (HD == 64 ? row & 3 : row) << 2; }   // rows of f32 results: eight rows' four pieces

IT_DEV float ror8(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x128, 0xf, 0xf, true));
}
// all but the last N loads of this wave have landed
template <int N>
IT_DEV void wait_loads() {
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
    asm volatile("" ::: "memory");
}
// what this wave has read of (or written to) LDS is there
IT_DEV void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
IT_DEV void barrier() {
    wait_lds();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
// The same value, not known to be: what is computed from it is computed where it stands (a slice's addresses, formed ahead of
// the loop, would hold a hundred registers through it).
IT_DEV int here(int v) {
    asm volatile("" : "+v"(v));
    return v;
}
// NL loads of a wave, 1,024 bytes each: rows row0 .. of a slice (row0: a multiple of 8, the same in every lane), which are keys
// key0 + row of one KV head, to `to` of LDS (whose array starts at `lds`, address `at`).  `left` of them are there: loads without a row
// of their own are left out (ZERO: zeros instead), in the last one the rows behind are the last one again.
template <int HD, int NL, bool ZERO, typename Turn>
IT_DEV void ask(const uint16_t* head, int kv_dim, int key0, int row0, int left, bool direct, uint8_t* lds, uint32_t at, int to, int lane, Turn turn) {
    constexpr int P = HD / 8, RL = 512 / HD;   // pieces of a row, rows of a load
    const int b = lane / P, live = min(NL, (left + RL - 1) / RL);
    const uint8_t* base = (const uint8_t*)(head + (int64_t)(key0 + row0) * kv_dim);
    const uint32_t x = 16 * ((lane % P) ^ turn(b));
    // (loops, not unrolled: a launch finds the instruction cache cold, and a line of it costs as much as the loop)
#pragma unroll 1
    for (int i = 0; i < live; i++) {
        const int row = min(b, left - 1 - i * RL);
        if (direct) {
            to_lds_at(base, (x ^ (16 * turn(row0 + i * RL))) + __umul24(row, kv_dim * 2), at + to + i * 1024);
        } else {
            *(uint4*)(lds + to + i * 1024 + 16 * lane) = *(const uint4*)(base + (int64_t)row * kv_dim * 2 + (x ^ (16 * turn(row0 + i * RL))));
        }
        base += (int64_t)RL * kv_dim * 2;
    }
    if (ZERO)
#pragma unroll 1
        for (int i = max(0, live); i < NL; i++) *(uint4*)(lds + to + i * 1024 + 16 * lane) = make_uint4(0, 0, 0, 0);
}
// the rows behind the last one of a slice's values, once its loads have landed: their probability is 0, which the matrix cores multiply
template <int HD>
IT_DEV void zero_behind(uint8_t* rows, int left, int n, int lane) {
    constexpr int P = HD / 8, RL = 512 / HD;
    if (left > 0 && left < n && left % RL && lane / P >= left % RL) *(uint4*)(rows + left / RL * 1024 + 16 * lane) = make_uint4(0, 0, 0, 0);
}

// Query rows in LDS: f32 as they come, then, in the place of eight values' 32 bytes, their high and their low f16 halves, scaled.  The
// 16-byte pieces of head h's row are turned by 2 h: sixteen columns' reads hit different banks.
IT_DEV uint32_t pack2(_Float16 a, _Float16 b) { return (uint32_t)__builtin_bit_cast(uint16_t, a) | ((uint32_t)__builtin_bit_cast(uint16_t, b) << 16); }
IT_DEV void split8(float4 a, float4 b, float scale, uint8_t* to) {
    const float x[8] = {a.x * scale, a.y * scale, a.z * scale, a.w * scale, b.x * scale, b.y * scale, b.z * scale, b.w * scale};
    uint32_t hi[4], lo[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const _Float16 h0 = (_Float16)x[2 * e], h1 = (_Float16)x[2 * e + 1];
        hi[e] = pack2(h0, h1);
        lo[e] = pack2((_Float16)(x[2 * e] - (float)h0), (_Float16)(x[2 * e + 1] - (float)h1));
    }
    *(uint4*)to = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    *(uint4*)(to + 16) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
}
// where the results go: one range: the output, else the partial results
struct Result {
    float *part, *out;
    const float* gate;
    int gate_stride, n_split;
    int kpb;                     // keys of a range, a multiple of 32 (0: by the context that the device knows)
    int per;                     // queries of a block, of a few
};
// Contexts that stay one range (and need no merge where the host knows them).  One query: 64 KB of K and of V (heads of 256: 6.3 us
// at 128 keys where a range every 64 keys and the merge take 8.2, 8.9 against 8.2 at 256; of 128: 5.7 against 7.2 at 256, 7.3
// against 6.9 at 384; of 64: 6.7 against 7.2 at 512).  A few: three slices (eight queries, heads of 64: 5.4 us against 6.9; five,
// heads of 256: 10.0 against 10.5).
template <int HD> constexpr int one_range() { return 32768 / HD; }
constexpr int FEW_RANGE = 3 * SL;
// Keys of a range: the context over the ranges, in whole slices.  The same for a context that the device knows and for one that
// the host does: a pass that is issued op by op adds up in the order of the recorded ones of its tag.
__host__ IT_DEV int keys_over(int n_pos, int n_split, int one) {
    const int n = n_pos <= one ? n_pos : (n_pos + n_split - 1) / n_split;
    return (n + SL - 1) & ~(SL - 1);
}
IT_DEV int keys_of_range(int n_pos, const Result& r, int one) { return r.kpb ? r.kpb : keys_over(n_pos, r.n_split, one); }

// the partial result of row (query * n_head + head): its sums, its maximum m (log2 here, natural log as the merge expects) and weight
template <int HD>
IT_DEV float* partial(const Result& r, int64_t row, int split) {
    return r.part + (row * r.n_split + split) * (HD + 2);
}
template <int HD>
IT_DEV void put_stats(const Result& r, int64_t row, int split, float m, float l) {
    *(float2*)(partial<HD>(r, row, split) + HD) = make_float2(m == NONE ? -INFINITY : m * 0.6931471805599453f, l);
}

// ------------------------------------------------------------------ one query
// 16 columns, so 16x16x32 products: lane l supplies 8 k values of row (l % 16), k group l / 16, for A and for B, and receives D
// for column l % 16 and rows 4 * (l / 16) + i.
// With PREP the block forms its query heads itself (norm + rotation), and the wave whose slice holds the new position forms
// that position's key and value rows: they go to the slabs and straight into LDS.
template <int HD> constexpr int one_lds() { return 4 * 2 * SL * HD * 2 + 8 * HD * 4; }   // slices, the query
template <int HD> constexpr int one_blocks() { return HD == 256 ? 1 : HD == 128 ? 2 : 4; }              // of a CU

template <int HD, int G, bool PREP>
__global__ __launch_bounds__(256, one_blocks<HD>()) void attend_one_k(AttnArgs a, TilePrepP pr, int direct, Result res) {
    constexpr int NS = HD / 32, ND = HD / 16;   // k steps of a score tile, output tiles
    constexpr int P = HD / 8;                   // 16-byte pieces of a row
    constexpr int NL = HD / 16;                 // loads of a slice of K, and of V
    constexpr int SLICE = SL * HD * 2, V_AT = 4 * SLICE, Q_AT = 8 * SLICE;
    static_assert(G <= 8, "");
    extern __shared__ __align__(1024) uint8_t lds[];
    __shared__ float st_m[4][8], st_l[4][8];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int kvh = blockIdx.x, h0 = kvh * G, split = blockIdx.y;
    const int n_pos = a.n_pos_dyn ? *a.n_pos_dyn : a.n_pos;
    // the block's keys in whole groups of 32, a quarter for each wave
    const int kpb = keys_of_range(n_pos, res, one_range<HD>());
    const int beg = split * kpb + w * (kpb / 4), end = min(min(n_pos, (split + 1) * kpb), beg + kpb / 4);
    const int n_s = max(0, end - beg + SL - 1) / SL;
    const uint32_t at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lptr)lds);
    const uint16_t *const kh = a.k + kvh * HD, *const vh = a.v + kvh * HD;
    uint8_t* const K = lds + w * SLICE;
    uint8_t* const V = K + V_AT;
    auto whole = [&](int s) __attribute__((always_inline)) { return end - beg - s * SL >= SL; };
    auto ask_k = [&](int s) __attribute__((always_inline)) {
        ask<HD, NL, false>(kh, a.kv_dim, beg + s * SL, 0, end - beg - s * SL, direct, lds, at, w * SLICE, lane, turn_k<HD>);
    };
    auto ask_v = [&](int s) __attribute__((always_inline)) {
        ask<HD, NL, true>(vh, a.kv_dim, beg + s * SL, 0, end - beg - s * SL, direct, lds, at, V_AT + w * SLICE, lane, turn_v16<HD>);
    };

    // ---- the query
    if constexpr (!PREP) {
        constexpr int QP = HD / 4, RQ = 64 / QP;     // 16-byte pieces of a row, rows of a load
#pragma unroll 1
        for (int i = w; i * RQ < G; i += 4) {
            const int head = min(i * RQ + lane / QP, G - 1);
            const float* const from = a.q + (int64_t)(h0 + head) * HD + 4 * ((lane % QP) ^ (2 * head));
            if (direct) to_lds(from, at + Q_AT + i * 1024);
            else *(uint4*)(lds + Q_AT + i * 1024 + 16 * lane) = *(const uint4*)from;
        }
    }
    if (n_s > 0) {
        ask_k(0);
        ask_v(0);
    }
    if constexpr (!PREP) {
        if (n_s > 0 && whole(0)) wait_loads<2 * NL>();
        else wait_loads<0>();
    } else {
        constexpr int LPH = HD / 4, HPP = 64 / LPH;  // lanes per head, heads per wave pass
        const int li = lane % LPH;
        for (int g0 = w * HPP; g0 < G; g0 += 4 * HPP) {
            const int row = g0 + lane / LPH;  // G is a multiple of HPP or smaller than it
            if (row < G) {
                float4 v = ((const float4*)(pr.qg + (int64_t)(h0 + row) * 2 * HD))[li];
                v = head_norm_rope<HD>(v, pr.q_norm, pr.eps, pr.rope, pr.n_rot, n_pos - 1, li);
                *(float4*)(lds + Q_AT + row * HD * 4 + ((li ^ (2 * row)) << 4)) = v;
            }
        }
    }
    barrier();
    if (tid < G * P) {
        uint8_t* const u = lds + Q_AT + tid * 32;
        split8(*(const float4*)u, *(const float4*)(u + 16), a.scale * 1.4426950408889634f, u);
    }
    barrier();
    h8 qf[NS];
    {
        const int row = min(c & 7, G - 1);           // (columns without a head: the last head again, not used)
        const uint8_t* const q = lds + Q_AT + row * HD * 4;
#pragma unroll
        for (int s = 0; s < NS; s++) qf[s] = *(const h8*)(q + (((8 * s + 2 * g + (c >> 3)) ^ (2 * row)) << 4));
    }

    v4f o[ND];
#pragma unroll
    for (int dt = 0; dt < ND; dt++) o[dt] = v4f{0, 0, 0, 0};
    float m = NONE, l = 0.0f;
    const int v_key = 4 * g + (c >> 2);          // key this lane names of the sixteen of a transposing read
    for (int s = 0; s < n_s; s++) {
        const int kb = beg + s * SL, left = end - kb;
        const int fresh = PREP && n_pos - 1 >= kb && n_pos - 1 < min(end, kb + SL) ? n_pos - 1 - kb : -1;   // the new position's row
        if (whole(s)) wait_loads<NL>();
        else wait_loads<0>();
        auto put_row = [&](uint8_t* to, uint16_t* slab, float4 v, int turn, int li) __attribute__((always_inline)) {
            const uint2 hv = make_uint2((uint32_t)it_f32_to_f16(v.x) | ((uint32_t)it_f32_to_f16(v.y) << 16),
                                        (uint32_t)it_f32_to_f16(v.z) | ((uint32_t)it_f32_to_f16(v.w) << 16));
            *(uint2*)(slab + (int64_t)(n_pos - 1) * a.kv_dim + kvh * HD + 4 * li) = hv;
            *(uint2*)(to + fresh * HD * 2 + (((li >> 1) ^ turn) << 4) + 8 * (li & 1)) = hv;
        };
        if (PREP && fresh >= 0) {
            const int li = lane % (HD / 4);
            float4 v = ((const float4*)(pr.kproj + (int64_t)kvh * HD))[li];
            v = head_norm_rope<HD>(v, pr.k_norm, pr.eps, pr.rope, pr.n_rot, n_pos - 1, li);
            if (lane < HD / 4) put_row(K, pr.k_slab, v, turn_k<HD>(fresh), li);
            wait_lds();
        }
        v4f sc[2] = {v4f{0, 0, 0, 0}, v4f{0, 0, 0, 0}}, sd[2] = {v4f{0, 0, 0, 0}, v4f{0, 0, 0, 0}};   // (two chains of products each)
        {
            const int cc = here(c), turn = g ^ turn_k<HD>(cc);   // (row 16 + c: the same turn)
            const uint8_t* const row = K + cc * HD * 2;
            h8 kf[2][4];                         // two steps' rows, the next two's on their way
            auto read = [&](int i) __attribute__((always_inline)) {
#pragma unroll
                for (int e = 0; e < 4; e++) kf[(i >> 1) & 1][e] = *(const h8*)(row + (((4 * (i + (e >> 1))) ^ turn) << 4) + (e & 1) * 16 * HD * 2);
            };
            read(0);
#pragma unroll
            for (int i = 0; i < NS; i += 2) {
                if (i + 2 < NS) read(i + 2);
                __builtin_amdgcn_sched_barrier(0);
                const h8* const f = kf[(i >> 1) & 1];
                sc[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[0], qf[i], sc[0], 0, 0, 0);
                sc[1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[1], qf[i], sc[1], 0, 0, 0);
                sd[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[2], qf[i + 1], sd[0], 0, 0, 0);
                sd[1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[3], qf[i + 1], sd[1], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        wait_lds();
        if (s + 1 < n_s) ask_k(s + 1);
        // high + low halves, the keys past the range, the softmax
        float mt = -INFINITY;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            float v = sc[i >> 2][i & 3] + sd[i >> 2][i & 3];
            v += ror8(v);
            if (16 * (i >> 2) + 4 * g + (i & 3) >= left) v = -INFINITY;
            sc[i >> 2][i & 3] = v;
            mt = fmaxf(mt, v);
        }
        mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
        mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
        const float m_new = mt > m + GROW ? mt : m, alpha = __builtin_amdgcn_exp2f(m - m_new);
        m = m_new;
        float psum = 0.0f;
        h8 pf;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float p = __builtin_amdgcn_exp2f(sc[i >> 2][i & 3] - m);
            psum += p;
            pf[i] = (_Float16)p;
        }
        l = l * alpha + psum;
        if (s > 0 && __any(alpha != 1.0f)) {
#pragma unroll
            for (int dt = 0; dt < ND; dt++) o[dt] *= alpha;
        }
        if (s + 1 < n_s && whole(s + 1)) wait_loads<NL>();
        else wait_loads<0>();
        if (PREP && fresh >= 0 && lane < HD / 4)
            put_row(V, pr.v_slab, ((const float4*)(pr.vproj + (int64_t)kvh * HD))[lane], turn_v16<HD>(fresh), lane);
        zero_behind<HD>(V, left, SL, lane);
        const int vk = here(v_key);
        const uint8_t* const v_row = V + vk * HD * 2 + (c & 3) * 8;
        h8 vf[2][4];                             // four tiles', the next four's on their way
        auto read = [&](int d0) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint8_t* const p = v_row + ((32 * (d0 + e)) ^ (turn_v16<HD>(vk) << 4));   // (key 16 + vk: the same turn)
                const s4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ls4*)p);
                const s4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ls4*)(p + 16 * HD * 2));
                vf[(d0 >> 2) & 1][e] = __builtin_bit_cast(h8, s8(__builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7)));
            }
        };
        read(0);
#pragma unroll
        for (int d0 = 0; d0 < ND; d0 += 4) {
            if (d0 + 4 < ND) read(d0 + 4);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < 4; e++) o[d0 + e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[(d0 >> 2) & 1][e], pf, o[d0 + e], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        wait_lds();
        if (s + 1 < n_s) ask_v(s + 1);
    }

    // ---- the waves' results side by side in LDS (each in its own slice of K), f32 rows, pieces turned by the row
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (lane < G) {
        st_m[w][lane] = m;
        st_l[w][lane] = l;
    }
    if (c < G) {
#pragma unroll
        for (int dt = 0; dt < ND; dt++) *(v4f*)(K + c * HD * 4 + (((4 * dt + g) ^ turn_o<HD>(c)) << 4)) = o[dt];
    }
    barrier();
    constexpr int OP = HD / 4;                   // pieces of a row
#pragma unroll
    for (int i0 = 0; i0 < G * OP; i0 += 256) {
        const int i = i0 + tid, row = i / OP, pc = i % OP;
        if (G * OP < 256 && i >= G * OP) break;
        const float m0 = st_m[0][row], m1 = st_m[1][row], m2 = st_m[2][row], m3 = st_m[3][row];
        const float mm = fmaxf(fmaxf(m0, m1), fmaxf(m2, m3));
        const float wt[4] = {__builtin_amdgcn_exp2f(m0 - mm), __builtin_amdgcn_exp2f(m1 - mm), __builtin_amdgcn_exp2f(m2 - mm), __builtin_amdgcn_exp2f(m3 - mm)};
        float4 sum = make_float4(0, 0, 0, 0);
        float ll = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float4 x = *(const float4*)(lds + k * SLICE + row * HD * 4 + ((pc ^ turn_o<HD>(row)) << 4));
            sum.x += x.x * wt[k]; sum.y += x.y * wt[k]; sum.z += x.z * wt[k]; sum.w += x.w * wt[k];
            ll += st_l[k][row] * wt[k];
        }
        if (res.out) {
            float x[4] = {sum.x / ll, sum.y / ll, sum.z / ll, sum.w / ll};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (res.gate) x[e] *= fx_sigmoid(res.gate[(int64_t)(h0 + row) * res.gate_stride + 4 * pc + e]);
                res.out[(int64_t)(h0 + row) * HD + 4 * pc + e] = x[e];
            }
        } else {
            float2* const q = (float2*)(partial<HD>(res, h0 + row, split) + 4 * pc);   // (8-byte aligned)
            q[0] = make_float2(sum.x, sum.y);
            q[1] = make_float2(sum.z, sum.w);
            if (pc == 0) put_stats<HD>(res, h0 + row, split, mm, ll);
        }
    }
}

// ------------------------------------------------------------------ a few queries
// Up to eight queries a block, a pair of them for each of four waves (of two, where the launcher says four): 32 columns, so 32x32x16 products: lane l supplies 8 k
// values of row (l % 32), k group l / 32, for A and for B, and receives D for column l % 32 and rows 8 * (i / 4) + 4 * (l / 32) + i % 4.
// Heads of 256 take two waves a pair (H), which form the same scores and half of the sums each: one wave's sums, 128 registers a
// lane, would stand alone on its SIMD with everything between two trips to LDS exposed.  The waves bring a slice together, two
// in LDS: the cache is read once whatever the number of queries.
template <int HD> constexpr int few_lds() { return 2 * 2 * SL * HD * 2 + 4 * 16 * HD * 4; }
template <int HD> constexpr int few_waves() { return HD == 256 ? 2 : 1; }                                // of a pair of queries
template <int HD> constexpr int few_blocks() { return HD == 256 ? 1 : HD == 128 ? 2 : 4; }
constexpr int FEW = 8;

template <int HD, int G>
__global__ __launch_bounds__(256 * few_waves<HD>(), few_blocks<HD>() * few_waves<HD>()) void attend_few_k(AttnArgs a, int direct, Result res) {
    constexpr int H = few_waves<HD>(), RW = 8 / H;                         // keys of a slice that a wave brings
    constexpr int NS = HD / 16, ND = HD / 32 / H;   // k steps of a score tile, output tiles of a wave
    constexpr int P = HD / 8;                   // 16-byte pieces of a row
    constexpr int NL = HD / 64 / H;             // loads of a wave per slice of K, and of V
    constexpr int SLICE = SL * HD * 2, STAGE = 2 * SLICE, Q_AT = 2 * STAGE;
    static_assert(G <= 8, "");
    extern __shared__ __align__(1024) uint8_t lds[];
    __shared__ float own_s[4][FEW - 1][32];      // scores (log2) of the keys that not every one of eight queries sees
    __shared__ int own_odd[2][4 * H];                // whether a wave has found an infinity or a NaN among such keys' values (of a slice)
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int pw = w & 3, half = w >> 2;                                   // the wave's pair of queries, its share of the dims
    const int c = lane & 31, g = lane >> 5, z = c >> 4;
    const int kvh = blockIdx.x, h0 = kvh * G, split = blockIdx.y;
    const int t0 = blockIdx.z * res.per, t = t0 + 2 * pw;  // the block's first query, this wave's
    const int n_pos_last = a.n_pos_dyn ? *a.n_pos_dyn : a.n_pos;
    const int n_block = min(res.per, a.n_q - t0);                              // queries of the block
    const int pos_lo = n_pos_last - a.n_q + 1 + t0, pos_hi = pos_lo + n_block - 1;   // keys that its first and its last one see
    const int ahead = t0 % FEW, own_lo = pos_lo - ahead;                   // keys that the first of its eight queries sees (of another block, of four)
    const int my_pos = pos_lo + 2 * pw + z;                                 // (columns without a query: more than there are)
    const bool works = 2 * pw < n_block;                                    // waves without queries bring their share only
    const int kpb = keys_of_range(pos_hi, res, FEW_RANGE);
    const int k0 = split * kpb, k1 = min(pos_hi, k0 + kpb), n_s = max(0, k1 - k0 + SL - 1) / SL;
    const uint32_t at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lptr)lds);
    const uint16_t *const kh = a.k + kvh * HD, *const vh = a.v + kvh * HD;
    auto bring = [&](int s) __attribute__((always_inline)) {
        const int to = (s & 1) * STAGE + w * NL * 1024, left = k1 - k0 - s * SL - RW * w;   // the wave's rows
        ask<HD, NL, false>(kh, a.kv_dim, k0 + s * SL, RW * w, left, direct, lds, at, to, lane, turn_k<HD>);
        ask<HD, NL, true>(vh, a.kv_dim, k0 + s * SL, RW * w, left, direct, lds, at, to + SLICE, lane, turn_v32<HD>);
    };

    // ---- the wave's queries: rows [query][head]
    uint8_t* const Q = lds + Q_AT + pw * 16 * HD * 4;
    constexpr int QU = (2 * G * P / H + 63) / 64;   // units of eight values a lane takes
    float4 q0[QU], q1[QU];
    if (works) {
#pragma unroll
        for (int i = 0; i < QU; i++) {
            const int u = min((i * H + half) * 64 + lane, 2 * G * P - 1), row = u / P;
            const float* const from = a.q + ((int64_t)min(t + row / G, a.n_q - 1) * a.n_head + h0 + row % G) * HD + 8 * (u % P);
            q0[i] = *(const float4*)from;
            q1[i] = *(const float4*)(from + 4);
        }
    }
    if (n_s > 0) bring(0);
    if (n_s > 1) bring(1);
    h8 qf[NS];
    if (works) {
#pragma unroll
        for (int i = 0; i < QU; i++) {
            const int u = min((i * H + half) * 64 + lane, 2 * G * P - 1), row = u / P;
            split8(q0[i], q1[i], a.scale * 1.4426950408889634f, Q + row * HD * 4 + (((2 * (u % P)) ^ (2 * (row % G))) << 4));
        }
    }
    if (H > 1) barrier();
    else wait_lds();
    if (works) {
        const int head = min(c & 7, G - 1);          // (columns without a head: the last head again, not used)
        const uint8_t* const q = Q + (z * G + head) * HD * 4;
#pragma unroll
        for (int s = 0; s < NS; s++) qf[s] = *(const h8*)(q + (((4 * s + 2 * g + ((c >> 3) & 1)) ^ (2 * head)) << 4));
    }

    v16f o[ND];
#pragma unroll
    for (int dt = 0; dt < ND; dt++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[dt][i] = 0.0f;
    float m = NONE, l = 0.0f;
    bool odd_any = false;
    const int v_key = 4 * g + ((lane & 15) >> 2);   // key this lane names of the eight of a transposing read
    for (int s = 0; s < n_s; s++) {
        const int kb = k0 + s * SL, left = k1 - kb;
        uint8_t* const K = lds + (s & 1) * STAGE;
        uint8_t* const V = K + SLICE;
        if (s + 1 < n_s && k1 - kb >= 2 * SL) wait_loads<2 * NL>();        // (the next one is whole: 2 NL loads)
        else wait_loads<0>();
        zero_behind<HD>(V + w * NL * 1024, left - RW * w, RW, lane);
        // A masked key's probability is 0, and the matrix cores multiply it: from the values of keys that only the block's later
        // queries see, infinities and NaN are taken out here and added at the end, to those queries, with the f32 weight under the
        // last maximum (such keys lie in up to two slices, the maximum may move between them, and an f16 weight is 0 from 17 nats on).
        const int own = max(0, own_lo - kb);                               // the slice's first such key
        if (own < SL) {
            bool bad = false;
#pragma unroll 1
            for (int i = max(own, RW * w) * P + lane; i < min(min(SL, left), RW * (w + 1)) * P; i += 64) {
                uint32_t* const x = (uint32_t*)(V + i * 16);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const uint32_t e = x[k], m0 = (e & 0x7c00u) == 0x7c00u ? 0xffffu : 0u, m1 = (e & 0x7c000000u) == 0x7c000000u ? 0xffff0000u : 0u;
                    bad |= (m0 | m1) != 0;
                    x[k] = e & ~(m0 | m1);
                }
            }
            if (lane == 0) own_odd[s & 1][w] = 0;
            if (bad) own_odd[s & 1][w] = 1;
        }
        barrier();
        if (works) {
            v16f sc, sd;                                                   // (two chains of products)
#pragma unroll
            for (int i = 0; i < 16; i++) sc[i] = sd[i] = 0.0f;
            {
                const int cc = here(c), turn = g ^ turn_k<HD>(cc);
                const uint8_t* const row = K + cc * HD * 2;
                h8 kf[2][4];                     // four steps', the next four's on their way
                auto read = [&](int i) __attribute__((always_inline)) {
#pragma unroll
                    for (int e = 0; e < 4; e++) kf[(i >> 2) & 1][e] = *(const h8*)(row + (((2 * (i + e)) ^ turn) << 4));
                };
                read(0);
#pragma unroll
                for (int i = 0; i < NS; i += 4) {
                    if (i + 4 < NS) read(i + 4);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int e = 0; e < 4; e += 2) {
                        sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[(i >> 2) & 1][e], qf[i + e], sc, 0, 0, 0);
                        sd = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[(i >> 2) & 1][e + 1], qf[i + e + 1], sd, 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            // high + low halves, the keys past the range or the column's own position, the softmax
            const int seen = min(left, my_pos - kb);
            float mt = -INFINITY;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                float v = sc[i] + sd[i];
                v += ror8(v);
                if (8 * (i >> 2) + 4 * g + (i & 3) >= seen) v = -INFINITY;
                sc[i] = v;
                mt = fmaxf(mt, v);
            }
            mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
            const float m_new = mt > m + GROW ? mt : m, alpha = __builtin_amdgcn_exp2f(m - m_new);
            m = m_new;
            float psum = 0.0f;
            h8 pf[2];
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const float p = __builtin_amdgcn_exp2f(sc[i] - m);
                psum += p;
                pf[i >> 3][i & 7] = (_Float16)p;
            }
            l = l * alpha + psum;
            if (s > 0 && __any(alpha != 1.0f)) {
#pragma unroll
                for (int dt = 0; dt < ND; dt++)
#pragma unroll
                    for (int i = 0; i < 16; i++) o[dt][i] *= alpha;
            }
            int odd = 0;
            if (own < SL)
#pragma unroll
                for (int k = 0; k < 4 * H; k++) odd |= own_odd[s & 1][k];
            if (odd) {
                odd_any = true;
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int d = kb + 8 * (i >> 2) + 4 * g + (i & 3) - own_lo;
                    if (d >= 0 && d < ahead + n_block - 1) own_s[pw][d][c] = sc[i];
                }
            }
            const int vk = here(v_key);
            const uint8_t* const v_row = V + vk * HD * 2 + ((lane >> 4) & 1) * 32 + (lane & 3) * 8;
            {
                constexpr int W = ND < 4 ? ND : 4;
                h8 vf[2][W];                     // a group of tiles', the next group's on their way
                auto read = [&](int u) __attribute__((always_inline)) {    // group u: keys 16 j .., tiles d0 ..
                    const int j = u & 1, d0 = (u >> 1) * W;
#pragma unroll
                    for (int e = 0; e < W; e++) {
                        const uint8_t* const p = v_row + 16 * j * HD * 2 + ((64 * (half * ND + d0 + e)) ^ (turn_v32<HD>(vk) << 4));
                        const s4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ls4*)p);
                        const s4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ls4*)(p + 8 * HD * 2));
                        vf[u & 1][e] = __builtin_bit_cast(h8, s8(__builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7)));
                    }
                };
                read(0);
#pragma unroll
                for (int u = 0; u < 2 * ND / W; u++) {
                    if (u + 1 < 2 * ND / W) read(u + 1);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int e = 0; e < W; e++)
                        o[(u >> 1) * W + e] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[u & 1][e], pf[u & 1], o[(u >> 1) * W + e], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        if (s + 2 < n_s) {
            barrier();                           // every wave has read the slice
            bring(s + 2);
        }
    }
    if (!works) return;

    // ---- the wave's results, from the registers: two lanes' 32 bytes side by side
    l += __shfl_xor(l, 32, 64);
    const int tq = 2 * pw + z, head = c & 7;
    if ((c & 8) || head >= G || tq >= n_block) return;
    if (odd_any) {
        for (int d = 0; d < ahead + tq; d++) {   // (query tq sees pos_lo + tq keys)
            if (own_lo + d < k0 || own_lo + d >= k1) continue;
            const uint16_t* const v = vh + (int64_t)(own_lo + d) * a.kv_dim + 32 * half * ND + 4 * g;
            const float p = __builtin_amdgcn_exp2f(own_s[pw][d][c] - m);
#pragma unroll
            for (int dt = 0; dt < ND; dt++)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const uint16_t e = v[32 * dt + 8 * (i >> 2) + (i & 3)];
                    if ((e & 0x7c00) == 0x7c00) o[dt][i] += p * it_f16_to_f32(e);
                }
        }
    }
    const int64_t row = (int64_t)(t0 + tq) * a.n_head + h0 + head;
    if (!res.out && g == 0 && half == 0) put_stats<HD>(res, row, split, m, l);
    const float f = res.out ? 1.0f / l : 1.0f;
    typedef float f4 __attribute__((ext_vector_type(4), aligned(4)));
    f4* const to = (f4*)((res.out ? res.out + row * HD : partial<HD>(res, row, split)) + 32 * half * ND + 4 * g);
#pragma unroll
    for (int dt = 0; dt < ND; dt++)
#pragma unroll
        for (int i4 = 0; i4 < 4; i4++)
            to[8 * dt + 2 * i4] = f4{o[dt][4 * i4] * f, o[dt][4 * i4 + 1] * f, o[dt][4 * i4 + 2] * f, o[dt][4 * i4 + 3] * f};
}

// The ranges' results of a (query, head), weighted and divided, spread over the chip: one block per (query, head, 32 output
// dims).  A thread loads the statistics of range `tid` and, before any of them is needed, its share of the sums (group
// tid / 32 of the ranges, dim tid % 32: every load of the block is in flight at once); the block then agrees on the maximum,
// forms the weights exp(m_s - m) in LDS and adds up.  Ranges without keys carry m = -inf, l = 0 and sums of 0 (one whose keys
// all score -inf has the same weight, and 0 times what it found among its values).
constexpr int MERGE_MAX = 256;
template <int MAX>
__global__ __launch_bounds__(256) void attend_merge_wide_k(const float* __restrict__ part, int n_split, int hd,
                                                           float* __restrict__ out, const float* __restrict__ gate,
                                                           int gate_stride) {
    __shared__ float wsplit[256];
    __shared__ float red[8], accs[8][32];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int sg = tid >> 5, i = tid & 31;
    const int d0 = blockIdx.y * 32;
    const float* p = part + (int64_t)blockIdx.x * n_split * (hd + 2);
    const bool has = tid < n_split;
    const float ms = has ? p[(int64_t)tid * (hd + 2) + hd] : -INFINITY;
    const float ls = has ? p[(int64_t)tid * (hd + 2) + hd + 1] : 0.0f;
    float o[MAX / 8];
#pragma unroll
    for (int j = 0; j < MAX / 8; j++) {
        const int sp = sg + 8 * j;
        o[j] = sp < n_split ? p[(int64_t)sp * (hd + 2) + d0 + i] : 0.0f;
    }
    float m = group_max<64>(ms);
    if (lane == 0) red[wave] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float wgt = ms != -INFINITY ? __expf(ms - m) : 0.0f;
    wsplit[tid] = wgt;
    float l = group_sum<64>(ls * wgt);
    if (lane == 0) red[4 + wave] = l;
    __syncthreads();
    l = (red[4] + red[5]) + (red[6] + red[7]);
    float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
    for (int j = 0; j < MAX / 8; j += 2) {
        const float w0 = wsplit[sg + 8 * j], w1 = wsplit[sg + 8 * j + 8];
        a0 += o[j] * w0;
        a1 += o[j + 1] * w1;
    }
    accs[sg][i] = a0 + a1;
    __syncthreads();
    if (tid < 32) {
        float r = (((accs[0][i] + accs[1][i]) + (accs[2][i] + accs[3][i])) + ((accs[4][i] + accs[5][i]) + (accs[6][i] + accs[7][i]))) / l;
        if (gate) r *= fx_sigmoid(gate[(int64_t)blockIdx.x * gate_stride + d0 + i]);
        out[(int64_t)blockIdx.x * hd + d0 + i] = r;
    }
}

template <int HD, int G>
bool launch(const AttnArgs& a, const TilePrepP* prep, int n_split, float* part, float* out, const float* gate, int gate_stride, hipStream_t s) {
    const int direct = !((reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.k) | reinterpret_cast<uintptr_t>(a.v)) & 15) && a.kv_dim < (1 << 20);   // (offsets of 24 bits)
    // Eight queries a block, which read the cache once; four while that leaves one block a CU at most, half of the waves idle but none
    // waiting for another on its SIMD (16 heads of 256 on 2, eight queries at 48 / 512 / 1,024 / 2,048, each launch between two events:
    // 13.2, 16.2, 16.4, 17.5 us with eight, 11.1, 14.2, 14.9, 16.0 with four; on 4 at 2,048, 256 blocks of four, 16.3 and 15.4, at 5,431
    // 20.2 and 23.2).
    const int per = a.n_head_kv * n_split * ((a.n_q + 3) / 4) <= DECODE_CUS ? 4 : FEW;
    const int groups = a.n_q > 1 ? (a.n_q + per - 1) / per : 1;
    // one round of blocks: more of them would leave more results to merge, and have no more bytes in flight
    n_split = std::max(1, std::min(n_split, DECODE_CUS * (a.n_q > 1 ? few_blocks<HD>() : one_blocks<HD>()) / (groups * a.n_head_kv)));
    int kpb = 0;
    if (!a.n_pos_dyn) {
        kpb = keys_over(a.n_pos, n_split, a.n_q > 1 ? FEW_RANGE : one_range<HD>());
        n_split = (a.n_pos + kpb - 1) / kpb;
    }
    const Result res{part, n_split == 1 ? out : nullptr, gate, gate_stride, n_split, kpb, per};
    const dim3 grid(a.n_head_kv, n_split, groups), block(256);
    if (a.n_q > 1) {
        if (!lds_allowed<&attend_few_k<HD, G>>(few_lds<HD>())) return false;
        hipLaunchKernelGGL((attend_few_k<HD, G>), grid, dim3(256 * few_waves<HD>()), few_lds<HD>(), s, a, direct, res);
    } else if (prep) {
        if (!lds_allowed<&attend_one_k<HD, G, true>>(one_lds<HD>())) return false;
        hipLaunchKernelGGL((attend_one_k<HD, G, true>), grid, block, one_lds<HD>(), s, a, *prep, direct, res);
    } else {
        if (!lds_allowed<&attend_one_k<HD, G, false>>(one_lds<HD>())) return false;
        hipLaunchKernelGGL((attend_one_k<HD, G, false>), grid, block, one_lds<HD>(), s, a, TilePrepP{}, direct, res);
    }
    if (n_split == 1) return true;
    const dim3 merge(a.n_q * a.n_head, HD / 32);
    if (n_split <= 64) hipLaunchKernelGGL(attend_merge_wide_k<64>, merge, block, 0, s, part, n_split, HD, out, gate, gate_stride);
    else if (n_split <= 128) hipLaunchKernelGGL(attend_merge_wide_k<128>, merge, block, 0, s, part, n_split, HD, out, gate, gate_stride);
    else hipLaunchKernelGGL(attend_merge_wide_k<256>, merge, block, 0, s, part, n_split, HD, out, gate, gate_stride);
    return true;
}

template <int HD>
bool launch_hd(const AttnArgs& a, const TilePrepP* prep, int n_split, float* part, float* out, const float* gate, int gate_stride, hipStream_t s) {
    switch (a.n_head / a.n_head_kv) {
        case 1: return launch<HD, 1>(a, prep, n_split, part, out, gate, gate_stride, s);
        case 2: return launch<HD, 2>(a, prep, n_split, part, out, gate, gate_stride, s);
        case 4: return launch<HD, 4>(a, prep, n_split, part, out, gate, gate_stride, s);
        case 8: return launch<HD, 8>(a, prep, n_split, part, out, gate, gate_stride, s);
        default: return false;
    }
}

}  // namespace

bool attend_decode_takes(int n_q, int head_dim, int group) {
    return n_q <= DECODE_MAX_Q && (head_dim == 64 || head_dim == 128 || head_dim == 256) && group <= 8;
}
// false: nothing was launched and `out` is untouched (a group size that is not a power of two, LDS that could not be had)
bool attend_decode(const AttnArgs& a, const TilePrepP* prep, int n_split, float* part, float* out, const float* gate, int gate_stride,
                   hipStream_t s) {
    if (n_split < 1 || n_split > MERGE_MAX) return false;
    if (a.head_dim == 64) return launch_hd<64>(a, prep, n_split, part, out, gate, gate_stride, s);
    if (a.head_dim == 128) return launch_hd<128>(a, prep, n_split, part, out, gate, gate_stride, s);
    return launch_hd<256>(a, prep, n_split, part, out, gate, gate_stride, s);
}

}  // namespace itk
