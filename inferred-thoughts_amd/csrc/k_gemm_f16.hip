// =====================================================================================
// NVFP4 expert matmuls on the f16 matrix cores (fast mode).
//
// An NVFP4 weight is (doubled e2m1 value) x (halved e4m3 sub-block scale): at most six significant
// bits, so it is EXACT in f16, and so is every product with an f16 activation in the f32
// accumulator.  The Q8_0 activation x = q * dx is divided by a power of two that brings its row
// into [-1, 1] and split into two f16 numbers (x = hi + lo, 22 bits kept); the power of two comes
// back in the epilogue.  With the scales inside the operands the whole k range accumulates in the
// MFMA accumulator: no per-block scaling on the vector ALU, which bounds the int8 kernels above.
// What differs from the CPU path is the f32 summation order and the 2^-22 of the split.
//
// A block owns one tile of up to 128 (token, pick) pairs of one expert and 128 rows of the
// gate AND up matrices (GLU) or 256 rows of one matrix, with eight waves.  A wave owns two sets of
// 32 rows (gate and up rows of the same index, or two row groups) and half of the token tiles
// (waves 0-3 the first one or two groups of 32 pairs, waves 4-7 the next), so a token fragment
// read from LDS feeds four MFMAs (two sets, hi and lo) and the f32 sums of a wave stay within the
// registers that two waves per SIMD leave.  Weight nibbles go through LDS as full 128-byte lines to
// the owning lane's registers (a lane owns 16 contiguous bytes of a row per 64-wide k slab: the
// k order inside an MFMA is free once the scales are folded in) and are expanded there
// (fp4x8_to_f16x8).
//
// MFMA operand layout (32x32x16, f16): lane l supplies 8 k values of row (l % 32), k group
// l / 32, for both A (weight rows) and B (tokens); it receives D for token l % 32 and weight
// rows 8 * (i / 4) + 4 * (l / 32) + i % 4, i = 0..15.
#include "it_device.h"
#include "it_dot.h"
#include "it_launch.h"
#include "kernels.h"

// Phase stamps for tuning: a build with -DIT_STAMPS records the 100 MHz wall clock of one block's first
// lane at the marked points of five consecutive k slabs; the library build compiles them away.
#ifdef IT_STAMPS
__device__ long long it_gemm_stamps[32];
__device__ int it_gemm_stamp_tile, it_gemm_stamp_slab, it_gemm_stamp_glu;
// (five consecutive slabs of one block, six stamps each)
#define GEMM_STAMP(i)                                                                                                  \
    do {                                                                                                               \
        if ((int)blockIdx.x == it_gemm_stamp_tile && (GLU ? 1 : 0) == it_gemm_stamp_glu && s >= it_gemm_stamp_slab && \
            s < it_gemm_stamp_slab + 5 && tid == 0)                                                                    \
            it_gemm_stamps[6 * (s - it_gemm_stamp_slab) + (i)] = wall_clock64();                                       \
    } while (0)
#else
#define GEMM_STAMP(i) \
    do {              \
    } while (0)
#endif

namespace itk {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
constexpr int FK = 64;          // k per slab
constexpr int FBS = FK + 8;     // LDS row stride of a token slab, in f16 (144 bytes: eight lanes' 16-byte reads hit every bank once)
constexpr int FPAIRS = 128;     // pairs per tile
constexpr int FSUPER = 256;     // k per weight staging step (one 128-byte line of nibbles per row)
constexpr int FWS = 128 + 16;   // LDS row stride of a weight segment, in bytes

template <bool GLU, int T>
__device__ __forceinline__ void experts_f16_body(const ExpertsF16P& p, const int4 td, const int row_block, uint16_t* Bh, uint16_t* Bl,
                                                 uint8_t* Wn, uint8_t* Wsc, const int* xrow_s, const int* pair_s) {
    const int64_t e = td.x;
    const int cnt = td.z;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave8 = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave = wave8 & 3;      // which 32 (GLU) or 64 rows of the block
    const int th = wave8 >> 2;       // which half of the tile's token groups: T groups each
    const int r = lane & 31, kg = lane >> 5;
    const int n_in = p.n_in;
    // the two row sets of this wave
    const int rows_per_block = GLU ? 128 : 256;
    const int rb0 = row_block * rows_per_block + (GLU ? 32 : 64) * wave;
    const int rbase[2] = {rb0, GLU ? rb0 : rb0 + 32};
    const uint8_t* wq0 = it_expert_at(p.q, p.q_tab, e, p.q_stride);
    const uint8_t* ws0 = it_expert_at(p.s, p.s_tab, e, p.s_stride);
    const uint8_t* wq[2] = {wq0, GLU ? it_expert_at(p.q2, p.q2_tab, e, p.q_stride) : wq0};
    const uint8_t* ws[2] = {ws0, GLU ? it_expert_at(p.s2, p.s2_tab, e, p.s_stride) : ws0};
    // this wave's row segments in the block's weight buffer: GLU [set][wave][row], else [wave][set][row]
    const int myseg[2] = {GLU ? 32 * wave + r : 64 * wave + r, GLU ? 128 + 32 * wave + r : 64 * wave + 32 + r};
    // the segments this thread loads (four rows, one 16-byte piece of each row's 128 nibble bytes) and, for the
    // first 256 threads, the segment whose 16 scale bytes it loads
    const int piece = tid & 7;
    const uint8_t* wload[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int seg = (tid >> 3) + 64 * i;
        const int z = GLU ? seg >> 7 : 0;
        const int64_t row = min(row_block * rows_per_block + (GLU ? seg & 127 : seg), p.n_out - 1);
        // (picked by a conditional, not by an index into the array: a pointer that went through an indexed array is a
        // generic pointer to the compiler, and loads through it are flat loads that every LDS wait has to drain)
        wload[i] = (z ? wq[1] : wq[0]) + row * (n_in >> 1) + piece * 16;
    }
    const uint8_t* sload;
    {
        const int st = tid & 255;
        const int z = GLU ? st >> 7 : 0;
        const int64_t row = min(row_block * rows_per_block + (GLU ? st & 127 : st), p.n_out - 1);
        sload = (z ? ws[1] : ws[0]) + row * (n_in >> 4);
    }

    // Software pipeline.  Weights come in super-slabs of 256 k: every thread loads full 128-byte lines of
    // eight rows (coalesced) one super-slab ahead and parks them in the other LDS weight buffer; a lane
    // then reads its own 16 nibble bytes and 2 scale bytes of the NEXT 64-wide slab and expands them to
    // f16 fragments one at a time between the MFMA groups of the current slab.  Tokens run one slab
    // ahead through registers into the other LDS token buffer.  Inside a slab the token fragments of the
    // next MFMA group are read from LDS while the current group is on the matrix unit.  Loads and LDS
    // stores are dealt out between the MFMA groups one or two at a time (loads over the first groups,
    // the stores of what they brought over the later ones), and the slab's one barrier stands in front
    // of its last group.
    const int n_super = n_in / FSUPER;
    uint4 rw[4], rsw;
    uint4 rbh[T], rbl[T];   // 64 * T tokens x 8 segments of 16 bytes = 512 * T segments per array
    rsw = make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; i++) rw[i] = rsw;
    // the token rows this thread stages: fixed for the whole k loop
    const uint16_t* xhp[T];
    const uint16_t* xlp[T];
#pragma unroll
    for (int u = 0; u < T; u++) {
        const int idx = tid + u * 512, tok = idx >> 3, seg = idx & 7;
        const int64_t at = (int64_t)xrow_s[tok] * n_in + seg * 8;
        xhp[u] = p.xh + at;
        xlp[u] = p.xl + at;
    }
    auto fetch_w = [&](int S) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; i++) rw[i] = *(const uint4*)(wload[i] + S * (FSUPER / 2));
        rsw = *(const uint4*)(sload + S * (FSUPER / 16));
    };
    // The same loads one at a time, to be issued between MFMA groups: a burst of 16-byte loads from all four
    // waves backs up the load unit (about 200 cycles an instruction) and the matrix unit idles behind it.
    // q < 2 T: piece q of the next slab's tokens; then the five loads of the next super-slab.
    constexpr int N_LOADS = 2 * T + 5, LPG = (N_LOADS + 4 * T - 1) / (4 * T);
    auto fetch_one = [&](int q, int s_next, int S_next, bool x_on, bool w_on) __attribute__((always_inline)) {
        if (q < 2 * T) {
            if (x_on) {
                if (q & 1) rbl[q >> 1] = *(const uint4*)(xlp[q >> 1] + s_next * FK);
                else rbh[q >> 1] = *(const uint4*)(xhp[q >> 1] + s_next * FK);
            }
        } else if (q < N_LOADS && w_on) {
            const int i = q - 2 * T;
            if (i < 4) rw[i] = *(const uint4*)(wload[i] + S_next * (FSUPER / 2));
            else rsw = *(const uint4*)(sload + S_next * (FSUPER / 16));
        }
    };
    auto stash_w = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; i++) *(uint4*)(Wn + (b * 256 + (tid >> 3) + 64 * i) * FWS + piece * 16) = rw[i];
        if (tid < 256) *(uint4*)(Wsc + (b * 256 + tid) * 16) = rsw;
    };
    auto fetch_x = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < T; u++) {
            rbh[u] = *(const uint4*)(xhp[u] + s * FK);
            rbl[u] = *(const uint4*)(xlp[u] + s * FK);
        }
    };
    auto stash_x = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < T; u++) {
            const int idx = tid + u * 512, tok = idx >> 3, seg = idx & 7;
            uint16_t* dh = Bh + (buf * FPAIRS + tok) * FBS + seg * 8;
            uint16_t* dl = Bl + (buf * FPAIRS + tok) * FBS + seg * 8;
            *(uint4*)dh = rbh[u];
            *(uint4*)dl = rbl[u];
        }
    };
    // The same stores one at a time, to go between the MFMA groups of the slab's second half: issued together at the
    // slab's end, the stores of all eight waves are a burst that the LDS works off while no wave has a product to issue,
    // and every wave's first read of the next slab queues behind it (measured with the stores, or the barrier behind
    // them, taken out: a third of the kernel's time).
    // (one address register per staged row: buffer, hi / lo half and part are constant offsets from it; Bl lies
    // 2 * FPAIRS * FBS behind Bh)
    uint16_t* xdst[T];
#pragma unroll
    for (int u = 0; u < T; u++) {
        const int idx = tid + u * 512;
        xdst[u] = Bh + (idx >> 3) * FBS + (idx & 7) * 8;
    }
    auto stash_x_part = [&](int buf, int i) __attribute__((always_inline)) {   // i < 2 T
        // (picked by conditionals, like the weights' below)
        const uint4 v = i == 0 ? rbh[0] : i == 1 ? rbl[0] : i == 2 ? rbh[T - 1] : rbl[T - 1];
        uint16_t* d = i < 2 ? xdst[0] : xdst[T - 1];
        *(uint4*)(d + buf * FPAIRS * FBS + (i & 1) * 2 * FPAIRS * FBS) = v;
    };
    auto stash_w_part = [&](int b, int i) __attribute__((always_inline)) {   // i < 5
        // (the register set picked by conditionals: indexed by a value the compiler does not fold early enough, the
        // array would live in scratch memory)
        const uint4 v = i == 0 ? rw[0] : i == 1 ? rw[1] : i == 2 ? rw[2] : rw[3];
        if (i < 4) *(uint4*)(Wn + (b * 256 + (tid >> 3) + 64 * i) * FWS + piece * 16) = v;
        else if (tid < 256) *(uint4*)(Wsc + (b * 256 + tid) * 16) = rsw;
    };
    // this lane's nibbles and scales of slab j of the super-slab in weight buffer b
    uint4 ra[2];
    uint32_t rs[2];
    auto read_nib = [&](int b, int j) __attribute__((always_inline)) {
#pragma unroll
        for (int z = 0; z < 2; z++) {
            ra[z] = *(const uint4*)(Wn + (b * 256 + myseg[z]) * FWS + 32 * j + 16 * kg);
            rs[z] = *(const uint16_t*)(Wsc + (b * 256 + myseg[z]) * 16 + 4 * j + 2 * kg);
        }
    };
    // fragment n of set z from ra / rs
    auto expand = [&](int z, int n) __attribute__((always_inline)) -> h8 {
        const uint32_t wd = n == 0 ? ra[z].x : n == 1 ? ra[z].y : n == 2 ? ra[z].z : ra[z].w;
        return fp4x8_to_f16x8(wd, e4m3_to_scale(n < 2 ? rs[z] : rs[z] >> 8));
    };
    struct Tok { h8 h, l; };
    auto read_tok = [&](int buf, int n, int tt) __attribute__((always_inline)) -> Tok {
        // bytes 16 * kg + 4 * n .. + 3 of the row's slab: in the split form's order one run of eight elements
        const int at = (buf * FPAIRS + 32 * (T * th + tt) + r) * FBS + 32 * kg + 8 * n;
        return Tok{__builtin_bit_cast(h8, *(const uint4*)(Bh + at)), __builtin_bit_cast(h8, *(const uint4*)(Bl + at))};
    };

    const bool live_half = __builtin_amdgcn_readfirstlane(32 * T * th < cnt ? 1 : 0) != 0;
    const bool live_last = __builtin_amdgcn_readfirstlane(32 * (T * th + T - 1) < cnt ? 1 : 0) != 0;   // its last group of 32 as well
    // (59 and 80 pairs an expert, prompts of 3,000 and 4,096 over two layers: 3,068 -> 3,034 and 3,848 -> 3,815 us without a dead group's products)
    v16f acc[2][T];
#pragma unroll
    for (int z = 0; z < 2; z++)
#pragma unroll
        for (int tt = 0; tt < T; tt++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[z][tt][i] = 0.0f;

    fetch_w(0);
    fetch_x(0);
    stash_w(0);
    stash_x(0);
    __syncthreads();
    h8 af[2][2][4];   // [slab parity][set][fragment]
    read_nib(0, 0);
#pragma unroll
    for (int z = 0; z < 2; z++)
#pragma unroll
        for (int n = 0; n < 4; n++) af[0][z][n] = expand(z, n);
    if (live_half) read_nib(0, 1);   // (a row has at least one super-slab: slab 1 is there)
    Tok first = read_tok(0, 0, 0);
    // One super-slab (four slabs) per trip so that every register array is indexed by a constant.
    // The slab's barrier stands IN FRONT of its last MFMA group, whose operands are in registers by then: behind it every
    // wave asks for the first token fragment and the nibbles of what comes next and then still has that group to issue,
    // so the wait for the slowest wave and the LDS round trip of the first read run under products instead of between
    // two slabs.  Everything that the barrier orders is ahead of it: the last read of this slab's token buffer, the
    // stores of the next slab's tokens and of the next super-slab's weights.
    for (int S = 0; S < n_super; S++) {
        const int wb = S & 1;
        const bool more_w = S + 1 < n_super;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int par = j & 1;
            const int s = 4 * S + j;
            const bool more = j < 3 || more_w;
            const bool more2 = j < 2 || more_w;
            GEMM_STAMP(0);
            GEMM_STAMP(1);
            Tok cur = first;
#pragma unroll
            for (int n = 0; n < 4; n++) {
                // one fragment pair of the next slab between the MFMA groups of this one
                if (more && live_half) {   // a wave set without pairs expands nothing: its SIMD belongs to the wave that has them
#pragma unroll
                    for (int z = 0; z < 2; z++) af[par ^ 1][z][n] = expand(z, n);
                }
#pragma unroll
                for (int tt = 0; tt < T; tt++) {
                    Tok nxt = cur;
                    const int g1 = n * T + tt + 1;
                    if (g1 < 4 * T) nxt = read_tok(par, g1 / T, g1 % T);
#pragma unroll
                    for (int q = (g1 - 1) * LPG; q < g1 * LPG; q++) fetch_one(q, s + 1, S + 1, more, j == 0 && more_w);
                    // the next super-slab's weights (loaded a slab ago) over this slab's first groups, the next slab's
                    // tokens (asked for in this slab's first groups) over the groups of its second half but the last
                    if (j == 1 && more_w) {
                        constexpr int WPG = T == 1 ? 2 : 1;
#pragma unroll
                        for (int i = (g1 - 1) * WPG; i < g1 * WPG; i++)
                            if (i < 5) stash_w_part(wb ^ 1, i);
                    }
                    if (more && g1 > 2 * T && g1 < 4 * T) {
                        constexpr int PPG = (2 * T + 2 * T - 2) / (2 * T - 1);
#pragma unroll
                        for (int i = (g1 - 2 * T - 1) * PPG; i < (g1 - 2 * T) * PPG; i++)
                            if (i < 2 * T) stash_x_part(par ^ 1, i);
                    }
                    if (g1 == 4 * T) {
                        GEMM_STAMP(2);
                        __syncthreads();
                        GEMM_STAMP(3);
                        if (more) first = read_tok(par ^ 1, 0, 0);
                        // (the nibbles of the slab after next: this slab's expansions are done)
                        if (more2 && live_half) read_nib(j < 2 ? wb : wb ^ 1, (j + 2) & 3);
                    }
                    __builtin_amdgcn_sched_barrier(0);   // the reads stay ahead of the products they overlap
                    if (tt < T - 1 ? live_half : live_last) {   // a wave set whose token groups lie past the tile's pairs only helps with the staging
#pragma unroll
                        for (int z = 0; z < 2; z++) {
                            acc[z][tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[par][z][n], cur.h, acc[z][tt], 0, 0, 0);
                            acc[z][tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[par][z][n], cur.l, acc[z][tt], 0, 0, 0);
                        }
                    }
                    cur = nxt;
                }
            }
            GEMM_STAMP(4);
            GEMM_STAMP(5);
        }
    }

    const float e2a = p.scale2 ? p.scale2[e] : p.scale_a;
    const float e2b = GLU ? (p.scale2_up ? p.scale2_up[e] : p.scale_b) : e2a;
    // The down product's results go through LDS (every read of the slabs is in front of the last barrier), so that a pair's 256 leave
    // side by side, past the caches that they would fill twice over: 32 of a store's 64 lanes in rows of their own took 113 of 453
    // us of 5,700 tokens' products over 512 experts, ten a token; 417 so (3,000 tokens 290 -> 271).  Two, four or eight row
    // blocks of a tile in one pipeline, each one's results stored under the next one's products: 443, 466, 529.
    constexpr int OSTR = 256 + 4;
    static_assert(FPAIRS * OSTR * 4 <= 4 * FPAIRS * FBS * 2 + 2 * 256 * (FWS + 16), "");
    float* const O = (float*)Bh;
#pragma unroll
    for (int tt = 0; tt < T; tt++) {
        const int slot = 32 * (T * th + tt) + r;
        if (slot >= cnt) continue;
        const int64_t pair = pair_s[slot];
        const float rsc = p.rscale[xrow_s[slot]];
#pragma unroll
        for (int i4 = 0; i4 < 4; i4++) {
            if (GLU) {
                const int row = rbase[0] + 8 * i4 + 4 * kg;
                if (row >= p.n_out) continue;
                float o[4], u[4];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float g = acc[0][tt][4 * i4 + i] * rsc * e2a;
                    u[i] = acc[1][tt][4 * i4 + i] * rsc * e2b;
                    o[i] = fx_silu(g) * u[i];
                }
                *(float4*)(p.out + pair * p.n_out + row) = make_float4(o[0], o[1], o[2], o[3]);
                if (p.up_out) *(float4*)(p.up_out + pair * p.n_out + row) = make_float4(u[0], u[1], u[2], u[3]);
            } else {
#pragma unroll
                for (int z = 0; z < 2; z++) {
                    *(float4*)(O + slot * OSTR + 64 * wave + 32 * z + 8 * i4 + 4 * kg) =
                        make_float4(acc[z][tt][4 * i4] * rsc * e2a, acc[z][tt][4 * i4 + 1] * rsc * e2a,
                                    acc[z][tt][4 * i4 + 2] * rsc * e2a, acc[z][tt][4 * i4 + 3] * rsc * e2a);
                }
            }
        }
    }
    if (!GLU) {
        __syncthreads();
        const int row = row_block * 256 + 4 * lane;
        if (row < p.n_out) {
            typedef float fv4 __attribute__((ext_vector_type(4)));
            for (int slot = wave8; slot < cnt; slot += 8)
                __builtin_nontemporal_store(*(const fv4*)(O + slot * OSTR + 4 * lane), (fv4*)(p.out + (int64_t)pair_s[slot] * p.n_out + row));
        }
    }
}

template <bool GLU>
__global__ __launch_bounds__(512) void experts_f16_k(ExpertsF16P p) {
    extern __shared__ __align__(16) uint16_t flds[];
    uint16_t* Bh = flds;                          // [2][128][FBS]
    uint16_t* Bl = flds + 2 * FPAIRS * FBS;       // [2][128][FBS]
    uint8_t* Wn = (uint8_t*)(flds + 4 * FPAIRS * FBS);   // [2][256][FWS]: nibble bytes of 256 row segments x 256 k
    uint8_t* Wsc = Wn + 2 * 256 * FWS;             // [2][256][16]: their scale bytes
    __shared__ int xrow_s[FPAIRS], pair_s[FPAIRS];
    // Blocks go to the 8 XCDs in turn.  The row blocks of one tile read the same token rows (k slab by k slab, each
    // row block once: far more bytes than the weights): they take consecutive places on ONE XCD, so that they run
    // side by side and all but the first find the rows in that XCD's L2.
    const int n_rb = (p.n_out + (GLU ? 128 : 256) - 1) / (GLU ? 128 : 256);
    const int lin = blockIdx.x;
    const int tile = 8 * (lin / (8 * n_rb)) + (lin & 7), row_block = (lin >> 3) % n_rb;
    if (tile >= n_tiles_of(p, FPAIRS)) return;
    const int4 td = tile_of(p, tile, FPAIRS);
    const int cnt = td.z;
    if (row_block == 0 && threadIdx.x == 0) count_tile(p, td.x, cnt);
    if (threadIdx.x < FPAIRS) {
        const int pair = pair_at(p, td.y + min((int)threadIdx.x, cnt - 1));
        pair_s[threadIdx.x] = pair;
        xrow_s[threadIdx.x] = p.x_mode == 0 ? pair : (p.x_mode == 1 ? pair / p.n_used : 0);
    }
    __syncthreads();
    // waves 0..3 take the first T token groups of the tile, waves 4..7 the next T
    if (cnt <= 64) experts_f16_body<GLU, 1>(p, td, row_block, Bh, Bl, Wn, Wsc, xrow_s, pair_s);
    else experts_f16_body<GLU, 2>(p, td, row_block, Bh, Bl, Wn, Wsc, xrow_s, pair_s);
}

}  // namespace

size_t experts_f16_work_ints(int n_picks, int n_expert) {
    return 16 + (size_t)(n_expert + n_picks / FPAIRS + 2) * 4 + (size_t)n_picks;
}

bool experts_f16_takes(const ExpertsView& w, const ExpertsView* up, int n_picks, const float* out) {
    if (n_picks < 32 || w.n_expert > 1024 || w.fmt != W_NVFP4 || w.n_in % FSUPER || w.n_out % 4) return false;
    if ((reinterpret_cast<uintptr_t>(w.q) & 15) || w.q_stride % 16 || w.s_stride % 16 || (reinterpret_cast<uintptr_t>(w.scales) & 15) ||
        (reinterpret_cast<uintptr_t>(out) & 15))
        return false;
    if (up && (up->fmt != w.fmt || up->n_in != w.n_in || up->n_out != w.n_out || (reinterpret_cast<uintptr_t>(up->q) & 15) ||
               (reinterpret_cast<uintptr_t>(up->scales) & 15) || up->q_stride != w.q_stride || up->s_stride != w.s_stride))
        return false;
    const size_t lds = (size_t)4 * FPAIRS * FBS * sizeof(uint16_t) + (size_t)2 * 256 * (FWS + 16);
    return lds_allowed<&experts_f16_k<true>>(lds) && lds_allowed<&experts_f16_k<false>>(lds);
}

bool experts_gemm_f16(const ExpertsView& w, const ExpertsView* up, const int32_t* ids, int n_picks, int n_used,
                      int x_mode, const SplitOut& x, float* out, int32_t* work, size_t work_ints, bool grouped,
                      const TileCount& count, float scale_a, float scale_b, hipStream_t s, float* up_out) {
    if (!x.h || !experts_f16_takes(w, up, n_picks, out) || (reinterpret_cast<uintptr_t>(up_out) & 15)) return false;
    if (ids && (!work || work_ints < experts_f16_work_ints(n_picks, w.n_expert))) return false;
    if (n_used < 1) n_used = 1;
    const size_t lds = (size_t)4 * FPAIRS * FBS * sizeof(uint16_t) + (size_t)2 * 256 * (FWS + 16);
    const int max_tiles = ids ? w.n_expert + n_picks / FPAIRS + 1 : (n_picks + FPAIRS - 1) / FPAIRS;
    int32_t* n_tiles = ids ? work : nullptr;
    int4* tiles = ids ? (int4*)(work + 16) : nullptr;
    int32_t* order = ids ? work + 16 + (size_t)(max_tiles + 1) * 4 : nullptr;
    if (ids && !grouped) moe_group(ids, n_picks, w.n_expert, FPAIRS, n_tiles, tiles, order, s);
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
    const int tiles8 = (max_tiles + 7) / 8 * 8;   // (the kernel deals tiles to the XCDs in groups of eight)
    if (up) hipLaunchKernelGGL(experts_f16_k<true>, dim3(tiles8 * ((w.n_out + 127) / 128)), dim3(512), lds, s, p);
    else hipLaunchKernelGGL(experts_f16_k<false>, dim3(tiles8 * ((w.n_out + 255) / 256)), dim3(512), lds, s, p);
    return true;
}

}  // namespace itk

#ifdef IT_STAMPS
// tuning builds only: the stamps of the selected block, then the next selection
extern "C" int it_hip_debug_gemm_stamps(long long* out, int block, int slab, int glu) {
    if (hipDeviceSynchronize() != hipSuccess) return -1;
    if (hipMemcpyFromSymbol(out, HIP_SYMBOL(it_gemm_stamps), 32 * 8) != hipSuccess) return -1;
    if (hipMemcpyToSymbol(HIP_SYMBOL(it_gemm_stamp_tile), &block, 4) != hipSuccess ||
        hipMemcpyToSymbol(HIP_SYMBOL(it_gemm_stamp_slab), &slab, 4) != hipSuccess ||
        hipMemcpyToSymbol(HIP_SYMBOL(it_gemm_stamp_glu), &glu, 4) != hipSuccess)
        return -1;
    return 0;
}
#endif
