// =====================================================================================
// NVFP4 expert matmuls on the f16 matrix cores for FEW pairs per expert (fast mode).
//
// The 128-pair tiles of k_gemm_f16.hip pay for themselves from a few dozen pairs per expert on.  A batch
// of 32 .. 1,000 tokens over 512 experts leaves 1 .. 20 pairs per expert: there the work is the expansion
// of every touched expert's nibbles to f16, once, and its stream from HBM; the products are nearly free.
// This kernel keeps the arithmetic of the wide kernel (weights exact in f16 with the sub-block scale folded
// in, activations as an f16 hi + lo pair, f32 accumulation over the whole k range, the row's power of two
// and the expert's scale in the epilogue) on tiles of 16 pairs, MFMA 16x16x32:
//
//  * no LDS in the main loop: a wave is on its own.  Lane l supplies weight row l % 16 and the k group l / 16 of
//    the A operand straight from the nibble bytes it loads from global memory: two 128-bit loads per 256-wide
//    k chunk, units kg and kg + 4, so that the four lanes of a row fetch its whole 128-byte line at once
//    (with one load per 128-wide chunk every line was fetched in two halves, far apart in time: 10 % slower);
//  * the activations of the 16 pairs are stored (the split form, k_rows.hip) in the order the MFMA steps consume
//    them, so a lane's B operands of a chunk are sixteen 128-bit loads (from L2: a batch's activations are a
//    few MB).  They stay in registers while the wave walks its row groups, so every B load feeds
//    `groups` MFMAs;
//  * a wave owns up to 8 groups of 16 rows of ONE matrix and carries their f32 sums in registers across the k
//    chunks; for the gate/up pair two waves of a block take the gate rows and two the same rows of up, whose
//    sums cross to the gate waves through LDS at the end (the only barrier).
//
// MFMA 16x16x32 f16 operands: lane l holds A[l % 16][8 (l / 16) .. + 8], B[8 (l / 16) .. + 8][l % 16] and
// receives D[4 (l / 16) + i][l % 16], i = 0..3.  The k order inside a step is free as long as A and B agree:
// step n of a lane's 32-wide unit takes the elements the n-th dword of the 16 nibble bytes holds (byte i: low nibble element
// 16 (n / 2) + 4 (n % 2) + i, high nibble the same + 8).
#include <algorithm>

#include "it_device.h"
#include "it_dot.h"
#include "it_reduce.h"
#include "kernels.h"

namespace itk {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
constexpr int SK_PAIRS = 16;   // pairs per tile
constexpr int SK_KC = 256;     // k per chunk: two 32-wide units per k group, 128 bytes of nibbles per row
constexpr int SK_G = 8;        // row groups per wave at most
constexpr int SK_AHEAD = 1;    // steps of weights in flight per wave

struct RawW {
    uint4 nib[2];     // units kg and kg + 4 of the chunk: a row's whole 128-byte line is read by its four lanes at once
    uint32_t sc[2];
};

// fragment n (8 weights as f16, sub-block scale folded in) of a lane's 16 nibble bytes
IT_DEV h8 expand_frag(const uint4 nib, const uint32_t rsc, int n) {
    const uint32_t wd = n == 0 ? nib.x : n == 1 ? nib.y : n == 2 ? nib.z : nib.w;
    return fp4x8_to_f16x8(wd, e4m3_to_scale(n < 2 ? rsc : rsc >> 8));
}

// GLU: waves 0 and 1 take the gate matrix, waves 2 and 3 the up matrix of the same rows (a wave streams ONE matrix, so
// its sums and operands fit the registers of four to five waves per SIMD); the up waves pass their sums through LDS.
template <bool GLU>
__global__ __launch_bounds__(256) void experts_f16s_k(ExpertsF16P p, int gpw) {
    __shared__ float4 handoff[GLU ? 2 * SK_G * 64 : 1];
    const int tile = blockIdx.x;
    if (tile >= n_tiles_of(p, SK_PAIRS)) return;
    const int4 td = tile_of(p, tile, SK_PAIRS);
    const int64_t e = td.x;
    const int cnt = td.z;
    if (blockIdx.y == 0 && threadIdx.x == 0) count_tile(p, e, cnt);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, kg = lane >> 4;
    const int n_in = p.n_in, n_chunk = n_in / SK_KC;
    const int z = GLU ? wave >> 1 : 0;                 // which matrix
    const int wslot = GLU ? wave & 1 : wave;           // which share of the block's row groups
    constexpr int WPB = GLU ? 2 : 4;                   // shares per block
    // this wave's row groups: rows g0 * 16 .. of the matrix, `mine` of them (none: the wave only keeps the barrier)
    const int g0 = (blockIdx.y * WPB + wslot) * gpw;
    const int mine = max(0, min(gpw, (p.n_out + 15) / 16 - g0));
    const int pair = pair_at(p, td.y + min(r16, cnt - 1));
    const int xrow = p.x_mode == 0 ? pair : (p.x_mode == 1 ? pair / p.n_used : 0);
    const uint16_t* bh = p.xh + (int64_t)xrow * n_in + 32 * kg;
    const uint16_t* bl = p.xl + (int64_t)xrow * n_in + 32 * kg;
    const uint8_t* wq = z ? it_expert_at(p.q2, p.q2_tab, e, p.q_stride) : it_expert_at(p.q, p.q_tab, e, p.q_stride);
    const uint8_t* ws = z ? it_expert_at(p.s2, p.s2_tab, e, p.s_stride) : it_expert_at(p.s, p.s_tab, e, p.s_stride);

    v4f acc[SK_G];
#pragma unroll
    for (int g = 0; g < SK_G; g++) acc[g] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

    if (mine > 0) {
        // A step is one row group of one chunk: chunk st / mine, group st % mine.  Its weights are loaded SK_AHEAD
        // steps ahead.  (Measured on 512 experts x 10 pairs: two to eight steps ahead, or the next chunk's B operands
        // loaded early, cost a wave per SIMD in registers and were 5 - 25 % slower; the weight stream alone, without
        // the products, takes two thirds of the kernel's time.)
        const int n_steps = n_chunk * mine;
        auto load_step = [&](int st) __attribute__((always_inline)) -> RawW {
            RawW o;
            const int c = st / mine, g = st - c * mine;
            const int64_t row = min((g0 + g) * 16 + r16, p.n_out - 1);
            const int u = 8 * c + kg;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                o.nib[h] = *(const uint4*)(wq + row * (n_in >> 1) + (u + 4 * h) * 16);
                o.sc[h] = *(const uint16_t*)(ws + row * (n_in >> 4) + (u + 4 * h) * 2);
            }
            return o;
        };
        RawW q[SK_AHEAD];
#pragma unroll
        for (int d = 0; d < SK_AHEAD; d++) q[d] = load_step(min(d, n_steps - 1));
        uint4 nh[8], nl[8];
        auto load_b = [&](int c) __attribute__((always_inline)) {
#pragma unroll
            for (int n = 0; n < 8; n++) {
                nh[n] = *(const uint4*)(bh + c * SK_KC + 128 * (n >> 2) + 8 * (n & 3));
                nl[n] = *(const uint4*)(bl + c * SK_KC + 128 * (n >> 2) + 8 * (n & 3));
            }
        };
        load_b(0);
        int st = 0;
        for (int c = 0; c < n_chunk; c++) {
            h8 fh[8], fl[8];
            if (c > 0) load_b(c);
#pragma unroll
            for (int n = 0; n < 8; n++) {
                fh[n] = __builtin_bit_cast(h8, nh[n]);
                fl[n] = __builtin_bit_cast(h8, nl[n]);
            }
            // the groups of a chunk, unrolled so that the sums are indexed by constants
#pragma unroll
            for (int g = 0; g < SK_G; g++) {
                if (g < mine) {
                    const RawW cur = q[0];
                    const RawW nx = load_step(min(st + SK_AHEAD, n_steps - 1));
#pragma unroll
                    for (int d = 0; d + 1 < SK_AHEAD; d++) q[d] = q[d + 1];
                    q[SK_AHEAD - 1] = nx;
#pragma unroll
                    for (int n = 0; n < 8; n++) {
                        const h8 a = expand_frag(cur.nib[n >> 2], cur.sc[n >> 2], n & 3);
                        acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, fh[n], acc[g], 0, 0, 0);
                        acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, fl[n], acc[g], 0, 0, 0);
                    }
                    st++;
                }
            }
        }
    }
    if (GLU) {
        if (z == 1) {
#pragma unroll
            for (int g = 0; g < SK_G; g++)
                handoff[(wslot * SK_G + g) * 64 + lane] = make_float4(acc[g][0], acc[g][1], acc[g][2], acc[g][3]);
        }
        __syncthreads();
        if (z == 1) return;
    }
    if (r16 >= cnt) return;
    const float rsc = p.rscale[xrow];
    const float e2a = p.scale2 ? p.scale2[e] : p.scale_a;
    const float e2b = GLU ? (p.scale2_up ? p.scale2_up[e] : p.scale_b) : e2a;
#pragma unroll
    for (int g = 0; g < SK_G; g++) {
        if (g >= mine) break;
        const int row = (g0 + g) * 16 + 4 * kg;
        if (row >= p.n_out) continue;
        float o[4];
        if (GLU) {
            const float4 up = handoff[(wslot * SK_G + g) * 64 + lane];
            const float u4[4] = {up.x, up.y, up.z, up.w};
#pragma unroll
            for (int i = 0; i < 4; i++) o[i] = fx_silu(acc[g][i] * rsc * e2a) * (u4[i] * rsc * e2b);
            if (p.up_out)
                *(float4*)(p.up_out + (int64_t)pair * p.n_out + row) = make_float4(u4[0] * rsc * e2b, u4[1] * rsc * e2b, u4[2] * rsc * e2b, u4[3] * rsc * e2b);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) o[i] = acc[g][i] * rsc * e2a;
        }
        *(float4*)(p.out + (int64_t)pair * p.n_out + row) = make_float4(o[0], o[1], o[2], o[3]);
    }
}


// The same products with the k range split over the waves of a block.  Above, a wave walks one 128-byte column of its
// rows chunk after chunk, so every DRAM page is opened once per chunk and the stream stops at 3.5 TB/s.  Here the KW
// waves of a row set take one 256-wide chunk EACH (n_in = 256 KW, KW = 1, 2, 4 or 8) and walk the same row groups
// together: the block reads whole rows at a time, a wave's B operands are loaded once for a tile, and both
// matrices of the gate/up pair share them.  The price is a reduction of the KW partial sums of every 16 x 16 tile
// through LDS, a batch of two tiles per wave at a time (a row group of gate and up, or two of one matrix).
//
// A batch is one MFMA 32x32x16 chain: its two tiles are the A operand's 32 rows and the 16 pairs' high and low halves the B
// operand's 32 columns, so a lane expands every weight once and its scale serves the whole row of a half chunk.  Lane l
// supplies row l % 32's half l / 32 of the chunk and receives D[8 (i / 4) + 4 (l / 32) + i % 4][l % 32], i = 0..15.
//
// A wave brings a step (16 rows of its chunk, 2 KB; the scales of two steps with every second one) straight into a ring of its
// own in LDS, two to three steps ahead: no register waits on memory, no other wave is waited for, and a row's 128-byte line is
// one request.  A load writes its lanes' 16 bytes side by side, so a row's eight pieces are permuted by the row's number, so that
// sixteen rows' reads start in different banks.  The persistent grid shares all tiles' batches evenly, and the sums of a batch are
// finished by all eight waves (one wave at a time before).
//
// Bound by the stream of the touched experts' nibbles and the vector work of expanding them, which are about equal.  512 experts,
// ten a token, gate / up of 512 x 2,048 and down, each launch between two events: 204 tokens 137 and 81 us before, 133 and 79 now; 512
// tokens 169 and 98, now 150 and 89.  Of gate / up's 512 tokens, 141 us in a prompt's pass, the loads alone take 106, the work without the
// loads 103.
constexpr int SK_RING = 3;
// four scale codes, 0x7f (not a number: counts as zero) made zero; and the b-th of them as a factor for fp4x8_to_f16x8 (see e4m3_to_scale)
IT_DEV uint32_t scale_codes(uint32_t c) {
    c &= 0x7f7f7f7fu;
    const uint32_t bad = (c + 0x01010101u) & 0x80808080u;
    return c & ~(bad - (bad >> 7));
}
IT_DEV h2 scale_of(uint32_t codes, int b) { return __builtin_bit_cast(h2, __umul24((codes >> (8 * b)) & 0x7fu, 0x800080u)); }
// the same value, not known to be (what is computed from it is not kept in a register from batch to batch)
IT_DEV int here(int v) {
    asm volatile("" : "+v"(v));
    return v;
}
// an address that is the same in every lane, in scalar registers
IT_DEV const uint8_t* scalar(const uint8_t* p) {
    const uint64_t u = (uint64_t)p;
    return (const uint8_t*)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(u >> 32)) << 32) | (uint32_t)__builtin_amdgcn_readfirstlane((int)u));
}
constexpr int SK_WAVE_LDS = SK_RING * 2048 + 2 * 512;     // a wave's steps and scales

template <bool GLU, int KW>
__global__ __launch_bounds__(512, 4) void experts_f16k_k(ExpertsF16P p, int per_tile) {
    constexpr int NM = GLU ? 2 : 1;
    constexpr int GB = 2 / NM;        // row groups per batch
    constexpr int RS = 8 / KW;        // row sets per block
    __shared__ float4 red[8][2][68];  // [wave][tile of the batch][lane, 16 lanes and a space]
    __shared__ __align__(16) uint8_t ring[8 * SK_WAVE_LDS];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kw = wave % KW, rs = wave / KW;
    const int r16 = lane & 15, half = lane >> 5;
    const int n_in = p.n_in, n_groups = (p.n_out + 15) / 16;
    uint8_t* const mine = ring + wave * SK_WAVE_LDS;
    const uint32_t mine_at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lptr)mine);
    const uint32_t row_off = (uint32_t)(lane >> 3) * (n_in >> 1) + kw * 128 + (((lane & 7) ^ ((lane >> 4) & 7)) << 4);
    // The block's share of all tiles' batches, an even one: a run of batches of one tile after the other.  From one and a quarter tiles
    // a block on, whole tiles as well, one of each gridDim.x: an expert's tiles, side by side in the list, go through its rows at the
    // same time on blocks of one XCD and take them from each other's cache lines.  (One after the other in a block's run, they had its
    // rows from memory each time: 512 experts, gate / up and down, 16 / 20 / 28 / 36 pairs an expert: 197 and 112, 254 and 140, 299 and
    // 167, 384 and 204 us so, now 181 and 107, 217 and 127, 252 and 143, 305 and 174.  At 8 and 10 pairs, 1.00 and 1.07 tiles a block,
    // the run alone: 144 and 85, 149 and 90 against 147 and 94, 151 and 94.)
    const unsigned tiles = n_tiles_of(p, SK_PAIRS), blocks = gridDim.x, b = blockIdx.x;
    const int whole = 4 * tiles >= 5 * blocks ? tiles / blocks : 0;
    const int place = blocks % 8 ? b : b % 8 * (blocks / 8) + b / 8;
    const unsigned rest = (tiles - whole * blocks) * per_tile, each = rest / blocks, more = rest - each * blocks;
    // The batches left over: one for each CU before a second one for any (blocks b and b + 256 of two a CU share one; spread over all
    // 512 blocks they fell to both or to neither: gate / up and down of 128 experts of 256 x 512 at 10 pairs 27 and 22 us, now 25 and 21,
    // of 64 of 512 x 2,048 at 16 pairs 46 and 36, now 42 and 33).
    auto run_at = [&](unsigned i) {
        const unsigned a = min(more, 256u), over = blocks == 512 ? (min(i, 256u) * a + (max(i, 256u) - 256u) * (more - a)) >> 8 : min(i, more);
        return (int)(whole * blocks * per_tile + i * each + over);
    };
    int unit = run_at(b), round = 0;
    const int unit1 = run_at(b + 1), first_run = 2 * b >= blocks ? 0 : whole;   // (half of the blocks begin with the run: a CU's two are at different places of their tiles)
    bool first_batch = true;
    while (true) {
    const bool run = round >= first_run && unit < unit1;
    if (!run && round >= whole) break;
    int tile = round * blocks + place, b0 = 0, n_batches = per_tile;
    if (run) {
        tile = (unsigned)unit / (unsigned)per_tile;
        b0 = unit - tile * per_tile;
        n_batches = min(per_tile - b0, unit1 - unit);
        unit += n_batches;
    } else {
        round++;
    }
    const int4 td = tile_of(p, tile, SK_PAIRS);
    const int64_t e = td.x;
    const int cnt = td.z;
    if (b0 == 0 && threadIdx.x == 0) count_tile(p, e, cnt);
    const int pair = pair_at(p, td.y + min(r16, cnt - 1));
    const int xrow = p.x_mode == 0 ? pair : (p.x_mode == 1 ? pair / p.n_used : 0);
    const uint8_t* const wq[2] = {scalar(it_expert_at(p.q, p.q_tab, e, p.q_stride)), GLU ? scalar(it_expert_at(p.q2, p.q2_tab, e, p.q_stride)) : nullptr};
    const uint8_t* const ws[2] = {it_expert_at(p.s, p.s_tab, e, p.s_stride), GLU ? it_expert_at(p.s2, p.s2_tab, e, p.s_stride) : nullptr};

    // step st = batch st / 2, tile st % 2 of it: a row group's gate, then up rows, or two row groups
    const int n_steps = n_batches * 2;
    auto group_of = [&](int st) { return ((b0 + st / 2) * RS + rs) * GB + (GLU ? 0 : st & 1); };
    // (whole groups of 16 rows: a lane's part of an address is fixed, and only the row group's, scalar, moves)
    auto ask = [&](int st, int slot, int z) __attribute__((always_inline)) {
        const uint8_t* const base = (z ? wq[1] : wq[0]) + (int64_t)min(group_of(st), n_groups - 1) * 16 * (n_in >> 1);
        to_lds_at(base, row_off, mine_at + slot * 2048);
        to_lds_at(base + 8 * (n_in >> 1), row_off ^ 64, mine_at + slot * 2048 + 1024);   // (row 8 + r: r / 2 turns by 4 more)
    };
    // scales of batch i: lanes 0 .. 15 its first tile's rows, 16 .. 31 its second's
    const uint8_t* const my_scales = (GLU && lane >= 16 ? ws[1] : ws[0]) + (int64_t)r16 * (n_in >> 4) + kw * 16;
    auto ask_scales = [&](int i) __attribute__((always_inline)) {
        if (lane < 32) to_lds(my_scales + (int64_t)min(group_of(2 * i + (lane >> 4)), n_groups - 1) * 16 * (n_in >> 4), mine_at + SK_RING * 2048 + (i & 1) * 512);
    };
    // Of a batch's tiles this wave finishes 16 / KW pairs' quads (four rows of a pair, of 16), KW lanes a quad: lane q * KW + k has
    // the partial sums of chunk k.  A pair's 16 rows, 64 bytes, are stored side by side.
    const int fk = lane % KW, fkg = (lane / KW) & 3, f16 = kw * (16 / KW) + (lane / KW) / 4;
    const int fpair = pair_at(p, td.y + min(f16, cnt - 1));
    const float rsc = p.rscale[p.x_mode == 0 ? fpair : (p.x_mode == 1 ? fpair / p.n_used : 0)];
    const float e2a = p.scale2 ? p.scale2[e] : p.scale_a;
    const float e2b = GLU ? (p.scale2_up ? p.scale2_up[e] : p.scale_b) : e2a;
    // (in the order of their use: behind a batch's two steps the next one's scales and first step may be out)
    ask_scales(0);
    ask(0, 0, 0);
    ask(1, 1, NM - 1);
    if (n_batches > 1) {
        ask_scales(1);
        ask(2, 2, 0);
    }

    // this wave's B operands, for all batches of the tile: chunk kw of its 16 pairs, the high halves in columns 0 .. 15, the low
    // ones in 16 .. 31; half l / 32 of the chunk.  (Waited for here, by the statement at the end: the compiler counts these loads, but
    // not those to LDS, and left to the loop its waits would drain the stream with every batch.)
    uint4 fx[16];
    {
        const uint16_t* const x = ((lane & 16) ? p.xl : p.xh) + (int64_t)xrow * n_in + kw * SK_KC + 128 * half;
#pragma unroll
        for (int n = 0; n < 16; n++) fx[n] = *(const uint4*)(x + 8 * n);
#pragma unroll
        for (int n = 0; n < 16; n++) asm volatile("" : "+v"(fx[n].x), "+v"(fx[n].y), "+v"(fx[n].z), "+v"(fx[n].w));
    }

    int slot = 0;                             // of the batch's first step
    for (int i = 0; i < n_batches; i++) {
        if (i + 1 < n_batches) __builtin_amdgcn_s_waitcnt(0x0f73);
        else __builtin_amdgcn_s_waitcnt(0x0f70);
        asm volatile("" ::: "memory");
        const int slot1 = slot == SK_RING - 1 ? 0 : slot + 1, slot2 = slot1 == SK_RING - 1 ? 0 : slot1 + 1;
        const uint8_t* const d = mine + ((here(lane) & 16) ? slot1 : slot) * 2048 + r16 * 128;
        uint2 sc = *(const uint2*)(mine + SK_RING * 2048 + (i & 1) * 512 + (lane & 31) * 16 + 8 * half);
        sc = make_uint2(scale_codes(sc.x), scale_codes(sc.y));
        v16f acc;
#pragma unroll
        for (int q = 0; q < 16; q++) acc[q] = 0.0f;
#pragma unroll
        for (int j2 = 0; j2 < 2; j2++) {         // two of the row's four units at a time: 128 registers a lane hold no more
            uint4 nib[2];
#pragma unroll
            for (int j = 0; j < 2; j++) nib[j] = *(const uint4*)(d + (((4 * half + 2 * j2 + j) ^ ((r16 >> 1) & 7)) << 4));
            if (j2 == 1) {
                __builtin_amdgcn_s_waitcnt(0xc07f);     // (read: the slots may be filled again)
                asm volatile("" ::: "memory");
                if (i + 1 < n_batches) ask(2 * i + 3, slot, NM - 1);
                if (i + 2 < n_batches) {
                    ask_scales(i + 2);
                    ask(2 * i + 4, slot1, 0);
                }
            }
#pragma unroll
            for (int n = 0; n < 8; n++) {        // dword n of the two units: sub-block n / 2
                const uint32_t wd = (n & 3) == 0 ? nib[n >> 2].x : (n & 3) == 1 ? nib[n >> 2].y : (n & 3) == 2 ? nib[n >> 2].z : nib[n >> 2].w;
                acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(fp4x8_to_f16x8(wd, scale_of(j2 ? sc.y : sc.x, n >> 1)), __builtin_bit_cast(h8, fx[8 * j2 + n]), acc, 0, 0, 0);
                if (n & 1) __builtin_amdgcn_sched_barrier(0);
            }
        }
        slot = slot2;
        // High and low halves' products stand in lanes l and l ^ 16, the first tile's rows in the first eight values, the second's
        // in the others: rows of 16 lanes change places, and a lane has eight sums of one tile.
        float4 part[2];
        {
            float v[8];
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const float a = acc[q], b = acc[8 + q];      // (a bit_cast of a vector's element itself reads the first one)
                const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
                const unsigned s0 = sw[0], s1 = sw[1];
                v[q] = __uint_as_float(s0) + __uint_as_float(s1);
            }
            part[0] = make_float4(v[0], v[1], v[2], v[3]);     // rows 4 half ..
            part[1] = make_float4(v[4], v[5], v[6], v[7]);     // rows 8 + 4 half ..
        }
        if (!first_batch) __builtin_amdgcn_s_barrier();      // (the last batch's sums have been read)
        first_batch = false;
        asm volatile("" ::: "memory");
        red[wave][(lane >> 4) & 1][17 * half + r16] = part[0];
        red[wave][(lane >> 4) & 1][17 * (half + 2) + r16] = part[1];
        __builtin_amdgcn_s_waitcnt(0xc07f);
        __builtin_amdgcn_s_barrier();             // (not __syncthreads: the loads ahead stay out)
        asm volatile("" ::: "memory");
        // the KW partial sums of a quad of either tile, then its outputs dealt over its lanes: four of a gate / up pair, eight
        // of two groups
        float sum[2][4];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const float4 v = red[rs * KW + fk][t][17 * fkg + f16];
            sum[t][0] = group_sum<KW>(v.x);
            sum[t][1] = group_sum<KW>(v.y);
            sum[t][2] = group_sum<KW>(v.z);
            sum[t][3] = group_sum<KW>(v.w);
        }
        constexpr int OUTS = GLU ? 4 : 8, OPL = OUTS >= 4 * KW ? 4 : OUTS > KW ? OUTS / KW : 1;   // outputs of a quad, of a lane at a time
#pragma unroll
        for (int f0 = 0; f0 < OUTS; f0 += OPL * KW) {                        // (more than once only for KW = 1)
            const int first = f0 + fk * OPL, tile_of_it = GLU ? 0 : first >> 2;
            const int g = group_of(2 * i + tile_of_it), row = g * 16 + 4 * fkg + (first & 3);
            const bool live = g < n_groups && f16 < cnt && first < OUTS;
            if (!live) continue;
            typedef float fo __attribute__((ext_vector_type(OPL)));
            fo o, u;
#pragma unroll
            for (int q = 0; q < OPL; q++) {
                float v = 0.0f, w = 0.0f;
#pragma unroll
                for (int c = f0; c < f0 + OPL * KW && c < OUTS; c += OPL) {
                    v = c == f0 || first == c ? sum[GLU ? 0 : (c + q) >> 2][(c + q) & 3] : v;
                    if (GLU) w = c == f0 || first == c ? sum[1][(c + q) & 3] : w;
                }
                u[q] = w * rsc * e2b;
                o[q] = GLU ? fx_silu(v * rsc * e2a) * u[q] : v * rsc * e2a;
            }
            *(fo*)(p.out + (int64_t)fpair * p.n_out + row) = o;
            if (GLU && p.up_out) *(fo*)(p.up_out + (int64_t)fpair * p.n_out + row) = u;
        }
    }
    }
}

}  // namespace

bool experts_f16s_takes(const ExpertsView& w, const ExpertsView* up, int n_picks, const float* out) {
    if (n_picks < 32 || w.n_expert > 1024 || w.fmt != W_NVFP4 || w.n_in % SK_KC || w.n_out % 4) return false;
    if ((reinterpret_cast<uintptr_t>(w.q) & 15) || w.q_stride % 16 || w.s_stride % 2 || (reinterpret_cast<uintptr_t>(w.scales) & 1) ||
        (reinterpret_cast<uintptr_t>(out) & 15))
        return false;
    if (up && (up->fmt != w.fmt || up->n_in != w.n_in || up->n_out != w.n_out || (reinterpret_cast<uintptr_t>(up->q) & 15) ||
               (reinterpret_cast<uintptr_t>(up->scales) & 1) || up->q_stride != w.q_stride || up->s_stride != w.s_stride))
        return false;
    return true;
}

bool experts_gemm_f16s(const ExpertsView& w, const ExpertsView* up, const int32_t* ids, int n_picks, int n_used,
                       int x_mode, const SplitOut& x, float* out, int32_t* work, size_t work_ints, bool grouped,
                       const TileCount& count, float scale_a, float scale_b, hipStream_t s, float* up_out) {
    if (!x.h || !experts_f16s_takes(w, up, n_picks, out) || (reinterpret_cast<uintptr_t>(up_out) & 15)) return false;
    if (ids && (!work || work_ints < experts_group_work_ints(n_picks, w.n_expert))) return false;
    if (n_used < 1) n_used = 1;
    // the layout of the int8 tile kernel's grouping (tiles of 16 pairs): either may reuse the other's
    const int max_tiles = ids ? w.n_expert + n_picks / SK_PAIRS + 1 : (n_picks + SK_PAIRS - 1) / SK_PAIRS;
    int32_t* n_tiles = ids ? work : nullptr;
    int4* tiles = ids ? (int4*)(work + 16) : nullptr;
    int32_t* order = ids ? work + 16 + (size_t)(max_tiles + 1) * 4 : nullptr;
    if (ids && !grouped) moe_group(ids, n_picks, w.n_expert, SK_PAIRS, n_tiles, tiles, order, s);
    ExpertsF16P p{};
    p.q = (const uint8_t*)w.q;
    p.s = (const uint8_t*)w.scales;
    p.q2 = up ? (const uint8_t*)up->q : nullptr;
    p.s2 = up ? (const uint8_t*)up->scales : nullptr;
    p.q_stride = w.q_stride;
    p.s_stride = w.s_stride;
    p.q_tab = w.q_tab;
    p.s_tab = w.s_tab;
    p.q2_tab = up ? up->q_tab : nullptr;
    p.s2_tab = up ? up->s_tab : nullptr;
    p.scale2 = w.scale2;
    p.scale2_up = up ? up->scale2 : nullptr;
    p.xh = x.h;
    p.xl = x.l;
    p.rscale = x.scale;
    p.n_pairs = n_picks;
    p.scale_a = scale_a;
    p.scale_b = scale_b;
    p.count = count;
    p.out = out;
    p.up_out = up_out;
    p.n_in = w.n_in;
    p.n_out = w.n_out;
    p.x_mode = x_mode;
    p.n_used = n_used;
    p.n_tiles = n_tiles;
    p.tiles = tiles;
    p.order = order;
    const int groups = (w.n_out + 15) / 16;
    const int likely_tiles = ids ? std::min(n_picks, w.n_expert) + n_picks / SK_PAIRS : max_tiles;
    const int n_chunk = w.n_in / SK_KC;
    const bool scales16 = w.s_stride % 16 == 0 && !(reinterpret_cast<uintptr_t>(w.scales) & 15) && !(up && (reinterpret_cast<uintptr_t>(up->scales) & 15));
    if (scales16 && w.n_out % 16 == 0 && (n_chunk == 1 || n_chunk == 2 || n_chunk == 4 || n_chunk == 8)) {
        // k split over the waves: a batch is 2 / NM row groups per row set, 8 / n_chunk row sets per block.  Two blocks a CU,
        // which share all tiles' batches evenly: with a tile or half a tile a block, 512 tokens over 512 experts were 1,054
        // blocks on 512 places, a third round of 30 (157 -> 141 us for gate / up, 87 -> 79 for down).
        const int per_batch = (up ? 1 : 2) * (8 / n_chunk);
        const int per_tile = (groups + per_batch - 1) / per_batch;
        const dim3 grid((unsigned)std::min<int64_t>((int64_t)std::min(n_picks, max_tiles) * per_tile, 512));
#define IT_F16K(G, K) hipLaunchKernelGGL((experts_f16k_k<G, K>), grid, dim3(512), 0, s, p, per_tile)
        if (up) {
            if (n_chunk == 8) IT_F16K(true, 8); else if (n_chunk == 4) IT_F16K(true, 4); else if (n_chunk == 2) IT_F16K(true, 2); else IT_F16K(true, 1);
        } else {
            if (n_chunk == 8) IT_F16K(false, 8); else if (n_chunk == 4) IT_F16K(false, 4); else if (n_chunk == 2) IT_F16K(false, 2); else IT_F16K(false, 1);
        }
#undef IT_F16K
        return true;
    }
    // other row lengths: every wave walks the whole k range of its own rows
    int gpw = SK_G;
    const int wpb = up ? 2 : 4;   // shares of a block's row groups (the gate/up pair puts two waves on each)
    while (gpw > 1 && (int64_t)likely_tiles * ((groups + wpb * gpw - 1) / (wpb * gpw)) < 2048) gpw >>= 1;
    const dim3 grid(std::min(n_picks, max_tiles), (groups + wpb * gpw - 1) / (wpb * gpw));
    if (up) hipLaunchKernelGGL(experts_f16s_k<true>, grid, dim3(256), 0, s, p, gpw);
    else hipLaunchKernelGGL(experts_f16s_k<false>, grid, dim3(256), 0, s, p, gpw);
    return true;
}

}  // namespace itk
