// Per-block integer dots shared by the GEMV kernels and the fused decode kernels.
#pragma once
#include "it_device.h"
#include "kernels.h"

namespace itk {

// ------------------------------------------------------------------ E2M1 nibbles -> int8
// kvalues (doubled E2M1, /root/reference src/quant/mod.rs:265) through two byte
// permutes: magnitude by the low 3 bits, then the sign bit picks +mag or -mag.
IT_DEV uint32_t fp4x4_to_i8x4(uint32_t v) {  // v: four nibbles, one per byte
    const uint32_t TPlo = 0x03020100u, TPhi = 0x0c080604u;
    const uint32_t TNlo = 0xfdfeff00u, TNhi = 0xf4f8fafcu;
    uint32_t idx = v & 0x07070707u;
    uint32_t mag = __builtin_amdgcn_perm(TPhi, TPlo, idx);
    uint32_t neg = __builtin_amdgcn_perm(TNhi, TNlo, idx);
    uint32_t sel = ((v >> 1) & 0x04040404u) | 0x03020100u;
    return __builtin_amdgcn_perm(neg, mag, sel);
}

IT_DEV int dot4(uint32_t a, uint32_t b, int c) { return __builtin_amdgcn_sdot4((int)a, (int)b, c, false); }

// One 32-element unit of a Q8_0 row against activation block `a` (8 dwords).
IT_DEV float unit_q8_0(const uint4 w0, const uint4 w1, uint16_t dw_bits, const uint4 a0, const uint4 a1,
                       float dx) {
    int s = 0;
    s = dot4(w0.x, a0.x, s); s = dot4(w0.y, a0.y, s); s = dot4(w0.z, a0.z, s); s = dot4(w0.w, a0.w, s);
    s = dot4(w1.x, a1.x, s); s = dot4(w1.y, a1.y, s); s = dot4(w1.z, a1.z, s); s = dot4(w1.w, a1.w, s);
    float dw = it_f16_to_f32(dw_bits);
    return (float)s * (dw * dx);
}

// One 32-element unit (two 16-element sub-blocks) of an NVFP4 row.
IT_DEV void unit_nvfp4(const uint4 w, uint32_t sc2, const uint4 a0, const uint4 a1, float dy, float* tA,
                       float* tB) {
    int sa = 0, sb = 0;
    sa = dot4(fp4x4_to_i8x4(w.x & 0x0f0f0f0fu), a0.x, sa);
    sa = dot4(fp4x4_to_i8x4(w.y & 0x0f0f0f0fu), a0.y, sa);
    sa = dot4(fp4x4_to_i8x4((w.x >> 4) & 0x0f0f0f0fu), a0.z, sa);
    sa = dot4(fp4x4_to_i8x4((w.y >> 4) & 0x0f0f0f0fu), a0.w, sa);
    sb = dot4(fp4x4_to_i8x4(w.z & 0x0f0f0f0fu), a1.x, sb);
    sb = dot4(fp4x4_to_i8x4(w.w & 0x0f0f0f0fu), a1.y, sb);
    sb = dot4(fp4x4_to_i8x4((w.z >> 4) & 0x0f0f0f0fu), a1.z, sb);
    sb = dot4(fp4x4_to_i8x4((w.w >> 4) & 0x0f0f0f0fu), a1.w, sb);
    float dA = it_ue4m3_to_f32(sc2 & 0xffu), dB = it_ue4m3_to_f32((sc2 >> 8) & 0xffu);
    *tA = (dy * dA) * (float)sa;
    *tB = (dy * dB) * (float)sb;
}

// ------------------------------------------------------------------ E2M1 nibbles -> f16
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));
// a sub-block's scale for fp4x8_to_f16x8: an e4m3 code moved into an f16's exponent and mantissa fields is the scale times
// 2^-8, subnormal codes included (4 exponent bits with bias 7 against 5 with bias 15; f16 subnormals are computed with, not
// flushed); code 0x7f (not a number) counts as zero, as in the CPU path
IT_DEV h2 e4m3_to_scale(uint32_t code) {
    const uint32_t em = code & 0x7fu;
    const _Float16 sv = __builtin_bit_cast(_Float16, (uint16_t)(em == 0x7fu ? 0u : em << 7));
    return h2{sv, sv};
}
// the eight weights of a dword of nibbles: byte i's low nibble (element i of its sub-block's half) and high nibble (element
// 8 + i) side by side, through the conversion of the matrix cores' own fp4 (times 2^8, which pays for the scale's 2^-8) and
// one packed product; exact.  Half the vector operations of byte permutes and sign bits.
IT_DEV h8v fp4x8_to_f16x8(uint32_t w, h2 scale) {
    const h2 a = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 256.0f, 0) * scale;
    const h2 b = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 256.0f, 1) * scale;
    const h2 c = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 256.0f, 2) * scale;
    const h2 d = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 256.0f, 3) * scale;
    return h8v{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

typedef __attribute__((address_space(3))) void* lptr;
// 16 bytes a lane from memory to LDS, one lane's behind the other's from `to` on (the same in every lane).  Written out because
// the compiler's own form makes every later read of LDS wait for all such loads; here they are waited for by count, in front
// of the barrier of the stage that reads them.  (The LDS address goes in as M0 itself, so that the compiler knows what it holds.)
IT_DEV void to_lds(const void* from, uint32_t to) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "{m0}"(to), "v"(from) : "memory");
}

// The same from base + off (base: the same in every lane, in scalar registers).  A scalar register that a vector instruction has
// written (a v_readlane of the compiler's) may be read by a memory instruction five wait states later; inside a statement the
// compiler does not see that there is one.
IT_DEV void to_lds_at(const void* base, uint32_t off, uint32_t to) {
    asm volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %1, %2" : : "{m0}"(to), "v"(off), "s"(base) : "memory");
}

// operands of the f16 expert tile kernels (k_gemm_f16.hip, k_gemm_f16s.hip)
struct ExpertsF16P {
    const uint8_t *q, *s, *q2, *s2;
    const uint8_t* const *q_tab, *const *s_tab, *const *q2_tab, *const *s2_tab;  // expert placement tables or null
    int64_t q_stride, s_stride;
    const float *scale2, *scale2_up;
    const uint16_t *xh, *xl;
    const float* rscale;
    float* out;
    float* up_out;               // gate / up pair: the up product too (null: only silu(gate) * up)
    int n_in, n_out, x_mode, n_used;
    const int32_t* n_tiles;
    const int4* tiles;           // null: one matrix, tile t holds the pairs from t * (pairs a tile) on, in order
    const int32_t* order;
    int n_pairs;
    float scale_a, scale_b;      // factors of the two products
    TileCount count;
};
IT_DEV int4 tile_of(const ExpertsF16P& p, int tile, int per_tile) {
    return p.tiles ? p.tiles[tile] : make_int4(0, tile * per_tile, min(per_tile, p.n_pairs - tile * per_tile), 0);
}
IT_DEV int n_tiles_of(const ExpertsF16P& p, int per_tile) { return p.tiles ? *p.n_tiles : (p.n_pairs + per_tile - 1) / per_tile; }
IT_DEV int pair_at(const ExpertsF16P& p, int slot) { return p.tiles ? p.order[slot] : slot; }
// one thread per tile: the tile's reads of its expert (expert_count_k)
IT_DEV void count_tile(const ExpertsF16P& p, int64_t e, int cnt) {
    const TileCount& c = p.count;
    if (!c.a || !c.tally) return;
    atomicAdd(c.a + e, (uint32_t)cnt);
    if (c.b) atomicAdd(c.b + e, (uint32_t)cnt);
    const unsigned long long host = (c.tier_a && c.tier_a[e] ? cnt : 0) + (c.b && c.tier_b && c.tier_b[e] ? cnt : 0);
    const unsigned long long all = (unsigned long long)cnt * (c.b ? 2 : 1);
    if (host) atomicAdd(c.tally + 1, host);
    if (all > host) atomicAdd(c.tally, all - host);
}

// Serial ascending fold of T per-block terms from a 16-byte aligned LDS row.  A group is asked for ahead of the one being
// added, in registers of its own; 32 terms a group, whose additions outlast the reads (2,048 terms: 16 a group 10 us).
template <int N>
struct TermGroup {
    float4 v[N / 4];
    IT_DEV void load(const float* p) {
#pragma unroll
        for (int c = 0; c < N / 4; c++) v[c] = ((const float4*)p)[c];
    }
    IT_DEV float add_to(float acc) const {
#pragma unroll
        for (int c = 0; c < N / 4; c++) {
            acc += v[c].x;
            acc += v[c].y;
            acc += v[c].z;
            acc += v[c].w;
        }
        return acc;
    }
};
IT_DEV float fold_terms_from(float acc, const float* tr, int T) {
    constexpr int N = 32;
    int k = 0;
    const int last = T / N * N - N;   // start of the last whole group
    if (last >= 0) {
        TermGroup<N> a, b;
        a.load(tr);
        for (; k + 2 * N <= T; k += 2 * N) {
            b.load(tr + k + N);
            acc = a.add_to(acc);
            a.load(tr + min(k + 2 * N, last));
            acc = b.add_to(acc);
        }
        if (k + N <= T) {
            acc = a.add_to(acc);
            k += N;
        }
    }
    if (k + 16 <= T) {
        TermGroup<16> a;
        a.load(tr + k);
        acc = a.add_to(acc);
        k += 16;
    }
    for (; k < T; k++) acc += tr[k];
    return acc;
}
IT_DEV float fold_terms(const float* tr, int T) { return fold_terms_from(0.0f, tr, T); }

}  // namespace itk
