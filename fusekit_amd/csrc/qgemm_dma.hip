// Multi-row quantised matmul from 65 activation rows: tiles whose operands come straight from memory into LDS
// (global_load_lds: no registers, no LDS stores, nothing for the vector ALU to do) and whose weights are dequantised in
// registers by the wave that multiplies them, T(s q + b), the arithmetic of qgemm.hip's tiles.  Direct calls and prompt
// passes into a bf16 cache.  The task families fusekit_qgemm* plan qgemm.hip's tiles: their launch geometry (fk_plan_geometry:
// blocks, LDS, one kernel or two) is part of what a task list's owner sees and is tested; they have not been moved here.
//
// What bounds it is how much other work goes with the matrix instructions.  One v_mfma_f32_16x16x32_bf16 takes 16 cycles and
// hides two vector instructions of its wave, no more (measured: 18.5 cycles with one or two behind each, 22.5 with three, 28
// and more with four), two waves of a SIMD do not hide each other's better, and unpacking int4 costs 2.1 vector instructions
// a weight.  So a wave takes as many activation rows as its registers hold, 256 (the sums are half of the register file), and
// the unpacking is laid between the matrix instructions by hand, one or two at a time; with 128 rows a wave, two waves a SIMD,
// the same tile took 20 % longer, with the unpacking where the compiler puts it 35 %.  The rest is the requests: 38 cycles of
// a wave for each kilobyte, spread over a step's tiles.
//     us (before: the tiles of qgemm.hip; from 1024 rows dequantise + library), 4-bit weights, warm:
//     gate / up pair 9728 x 2560:    128 rows 34.8 -> 29.5   512 rows 99.2 -> 65.3   2048 rows 284 -> 222   4096 rows 446 -> 375
//     q / k / v 6144 x 2560:         512 rows 41.9 -> 33.6   768 rows 63.8 -> 50.2
//     2560 x 9728:                   512 rows 50.4 -> 46.8;  0.5B class, pair 4864 x 896, 200 rows: 39.6 -> 12.9
// (4096 rows of the pair are 1.09 PFLOP/s of the 1.16 that a large library product reaches on this card.)
#include <string.h>

#include <type_traits>

#include "dma_device.hpp"
#include "fk_host.hpp"
#include "gemv_kernel.hpp"

namespace fk {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

// acc += weights x activations with the accumulators in the AGPR half of the register file (left to itself the compiler keeps
// what is beyond 256 registers there and moves it back and forth).  The statement hides the instruction from the hazard
// recogniser: its operands are written at least a tile ahead, and the sums are read behind settle_matrix_ops().
__device__ __forceinline__ void mfma_acc(f32x4_t& acc, const uint32_t (&w)[4], const fk_u32x4_t& x) {
    const fk_u32x4_t wv = {w[0], w[1], w[2], w[3]};
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(wv), "v"(x));
}

struct QgemmDmaArgs {
    const uint16_t* x;  // [M, K] bf16
    uint32_t M, K, gpr;
    uint32_t slabs;        // slabs of 64 k per split (even)
    uint32_t total_slabs;  // K / 64
    uint32_t n_blocks, m_blocks, tiles;   // tiles = n_blocks * m_blocks
    uint32_t ksplit, n_seg, row_cols;     // row_cols: columns of a row of partial sums
    float* partial;   // [ksplit, M, row_cols] or null (one split: finished outputs)
    float* partial2;  // the up matrix of a pair
    const uint16_t* res;
    int variant;
    struct Seg {
        const unsigned char* w;
        const unsigned char* sc;
        const unsigned char* bi;
        uint16_t* y;
        const uint16_t* bias;
        uint32_t N, nb_end, col0, pad;
    } seg[3];   // a fan-out's matrices, or gate and up
};

// Eight int4 codes as bf16 weights T(s q + b).  A nibble in the low bits of a half word is the fp16 subnormal code * 2^-24
// (* 2^-20 four bits higher), so one mixed-precision FMA takes it as it lies: fma(code * 2^-24, s * 2^24, b) is
// fma(code, s, b) to the bit.
// (Pinned where they stand: left alone, the compiler moves an unpacked value to its use, behind all the matrix work, and takes
// the masked words apart again to permute bytes for every pair.)
__device__ __forceinline__ void pin(uint32_t& v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void pin(float& v) { asm volatile("" : "+v"(v)); }
template <int P>
__device__ __forceinline__ float half_of(uint32_t v) { return (float)__builtin_bit_cast(f16x2_t, v)[P]; }
template <int B>
__device__ __forceinline__ float byte_of(uint32_t v) { return (float)((v >> (8 * B)) & 0xffu); }

constexpr uint32_t dma_row_bytes(WKind kind) { return kind == W_Q4 ? 32u : 64u; }   // of a weight row and slab
constexpr uint32_t dma_waves(int gk) { return 4u * gk; }
// activations, codes, scales and biases (of 128 k)
constexpr uint32_t dma_stage_bytes(WKind kind, int gk, uint32_t wtn) { return 32768u + 4u * wtn * (dma_row_bytes(kind) * gk + 8u); }
// stages that fit into the LDS: four or three
constexpr uint32_t dma_stages(WKind kind, int gk, uint32_t wtn) { return 4u * dma_stage_bytes(kind, gk, wtn) <= 163840u ? 4u : 3u; }
constexpr uint32_t dma_lds_bytes(WKind kind, int gk, uint32_t wtn) { return dma_stages(kind, gk, wtn) * dma_stage_bytes(kind, gk, wtn); }

// SiLU(g) * u of the rounded sums, the variant with one rounding at the end, as swiglu_bits has it, with e^x and 1 / d from the
// hardware's 2^x and reciprocal instead of expf and a divide (128 outputs a lane: those take 8 us of a 90 us launch).
//     e^x 2^-32 = 2^(e - 32) 2^a: e is the nearest integer to x log2 e (adding 1.5 2^23, here less 32, rounds to integers and
//     leaves e - 32 in the low bits, from where it goes into the exponent of 2^a), a what is left, with log2 e in two parts:
//     the float next to it and the rest.  |a| <= 1/2, so 2^a keeps its last bits whatever x is.
//     x is held to -64 .. 110: below, 1 + e^x is 1; above, the result is zero (g < -110).  So nothing is infinite on the way.
//     d = (1 + e^x) 2^-32, 1 / d by the reciprocal and one Newton step: the reciprocal of 1 + e^x itself is subnormal from
//     2^126 on, which the instruction gives as zero; of d it is so only for results that are zero.
// Against 64 bits over all bf16 gates no further off than expf and the divide (largest error, units in the last place of fp32,
// here / there: gates in -4 .. -1 1.49 / 1.57, -20 .. -4 1.39 / 1.40, -88.7 .. -20 1.33 / 1.33, -1 .. 0 2.19 / 2.19, above zero
// 1.82 / 1.82; root mean square 0.546 / 0.546, 0.535 / 0.542, 0.557 / 0.555, 0.314 / 0.314, at most 0.534 / 0.539; rounded to bf16 all of
// them right; below -88.7, where expf overflows and leaves -0 u, this still has the value).
__device__ __forceinline__ float swiglu_fast(float acc_g, float acc_u) {
    constexpr float kRound = 12582912.0f - 32.0f;
    const float g = round_bf16(acc_g), u = round_bf16(acc_u);
    const float x = __builtin_amdgcn_fmed3f(-g, -64.0f, 110.0f);
    const float y = fmaf(x, 1.44269504f, kRound), e = y - kRound;
    const float a = fmaf(x, 1.92596299e-8f, fmaf(x, 1.44269504f, -e));
    const float d = __uint_as_float(__float_as_uint(__builtin_amdgcn_exp2f(a)) + (__float_as_uint(y) << 23)) + 0x1p-32f;
    const float r0 = __builtin_amdgcn_rcpf(d), r = fmaf(fmaf(-d, r0, 1.0f), r0, r0);
    return ((r * 0x1p-32f) * g) * u;
}
template <bool FAST>
__device__ __forceinline__ void store_swiglu(const QgemmDmaArgs& a, uint32_t m, uint32_t n, uint32_t N, const f32x4_t& g, const f32x4_t& u) {
    if (m >= a.M || n >= N) return;
    uint2 o;
    if constexpr (FAST)
        o = make_uint2(pack_bf16(swiglu_fast(g[0], u[0]), swiglu_fast(g[1], u[1])), pack_bf16(swiglu_fast(g[2], u[2]), swiglu_fast(g[3], u[3])));
    else
        o = make_uint2(swiglu_bits(g[0], u[0], a.variant, 1.0f) | (swiglu_bits(g[1], u[1], a.variant, 1.0f) << 16),
                       swiglu_bits(g[2], u[2], a.variant, 1.0f) | (swiglu_bits(g[3], u[3], a.variant, 1.0f) << 16));
    *reinterpret_cast<uint2*>(a.seg[0].y + (size_t)m * N + n) = o;
}

// GK = 1: a block of four waves, 256 activation rows x 4 WTN weight rows; a wave multiplies all 256 rows by WTN weight rows
// (its unpacked weights serve 16 tiles).  GK = 2: two groups of four waves, 128 x 4 WTN; the groups take slabs of 64 k in
// turn and their sums are added at the end.
template <WKind KIND, int GK, int WTN, bool PAIR>
__global__ __launch_bounds__(256 * GK, GK) void qgemm_dma_kernel(const QgemmDmaArgs a) {
    extern __shared__ uint4 lds_raw[];
    unsigned char* const lds = reinterpret_cast<unsigned char*>(lds_raw);
    constexpr int NJ = WTN / 16, NI = 16 / GK;
    constexpr uint32_t WAVES = dma_waves(GK), AR = 32u / WAVES;   // AR: activation requests of a wave per stage
    constexpr uint32_t BM = GK == 1 ? 256u : 128u, BN = 4u * WTN;
    constexpr uint32_t ROWB = dma_row_bytes(KIND);
    constexpr uint32_t A_BYTES = 32768u, W_BYTES = BN * ROWB, STAGE = dma_stage_bytes(KIND, GK, WTN);
    constexpr uint32_t NST = dma_stages(KIND, GK, WTN);
    constexpr uint32_t SC0 = A_BYTES + W_BYTES * GK, SC_BYTES = BN * 4u;
    constexpr uint32_t NWI = W_BYTES * GK / 1024u, CW = (NWI + WAVES - 1u) / WAVES;
    constexpr uint32_t NSI = BN / 64u, CS = (2u * NSI + WAVES - 1u) / WAVES;
    constexpr int REQ = (int)(AR + CW + CS);   // requests of a wave per stage
    static_assert(REQ <= NI, "one request per tile of a step");
    constexpr bool SPLIT_PAIR = PAIR && (NJ & 1);   // gate and up rows in different waves
    static_assert(!(SPLIT_PAIR && GK == 2), "pairs in different waves: groups along the activation rows only");

    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t gk = GK == 2 ? wave >> 2 : 0u, wn = wave & 3u, l16 = lane & 15u, kb = lane >> 4;

    // The tile: consecutive blocks go to the XCDs in turn, so each XCD takes one stretch of the list, in which four
    // m tiles of the same n are neighbours (their L2 then serves the weight rows, and the activation rows of a few n).
    // (the divisions run on the vector unit: their results are brought back to scalar registers, where the requests' addresses live)
    const uint32_t ks = __builtin_amdgcn_readfirstlane(blockIdx.x / a.tiles);
    uint32_t nb, mb;
    {
        const uint32_t b = blockIdx.x - ks * a.tiles, xcd = b & 7u, q = a.tiles >> 3, r = a.tiles & 7u;
        const uint32_t t = xcd * q + (xcd < r ? xcd : r) + (b >> 3);
        const uint32_t per = 4u * a.n_blocks, mg = t / per, in = t - mg * per;
        const uint32_t mh = a.m_blocks - 4u * mg < 4u ? a.m_blocks - 4u * mg : 4u;
        nb = __builtin_amdgcn_readfirstlane(in / mh);
        mb = __builtin_amdgcn_readfirstlane(4u * mg + in - nb * mh);
    }
    uint32_t si = 0;
    if (!PAIR && a.n_seg > 1u) {
        si = nb >= a.seg[0].nb_end ? (nb >= a.seg[1].nb_end ? 2u : 1u) : 0u;
        nb -= si ? a.seg[si - 1u].nb_end : 0u;
    }
    const uint32_t N = a.seg[si].N, m0 = mb * BM, n0 = nb * (PAIR ? BN / 2u : BN);
    const uint32_t slab0 = ks * a.slabs;
    const uint32_t n_slabs = a.total_slabs - slab0 < a.slabs ? a.total_slabs - slab0 : a.slabs;

    // ---- what this lane requests per stage: AR pieces of activations, CW of weights, CS of scales / biases
    uint32_t xoff[AR];
#pragma unroll
    for (int i = 0; i < (int)AR; ++i) {
        const uint32_t idx = wave * AR + (uint32_t)i, sub = GK == 2 ? idx >> 4 : 0u;
        const uint32_t m = m0 + (GK == 2 ? idx & 15u : idx) * 8u + (lane >> 3);
        // (a row's 16-byte pieces lie in LDS in the order p ^ (row / 2 % 8): the fragment reads of 16 rows meet all 64 banks)
        xoff[i] = (m < a.M ? m : a.M - 1u) * a.K * 2u + sub * 128u + (((lane & 7u) ^ ((lane >> 4) + 4u * (i & 1))) * 16u);
    }
    auto row_of = [&](uint32_t r, uint32_t* mat) {
        uint32_t n;
        if constexpr (!PAIR) {
            *mat = si;
            n = n0 + r;
        } else if constexpr (!SPLIT_PAIR) {
            const uint32_t w = r / (uint32_t)WTN, q = r % (uint32_t)WTN, h = (uint32_t)WTN / 2u;
            *mat = q >= h ? 1u : 0u;
            n = n0 + w * h + (q >= h ? q - h : q);
        } else {
            *mat = r >= BN / 2u ? 1u : 0u;
            n = n0 + (r >= BN / 2u ? r - BN / 2u : r);
        }
        return n < N ? n : N - 1u;   // rows past the end read the last row; never stored
    };
    const unsigned char *wptr[CW], *sptr[CS];
    uint32_t w_to[CW], s_to[CS];
#pragma unroll
    for (uint32_t i = 0; i < CW; ++i) {
        const uint32_t idx = (wave + i * WAVES) % NWI, sub = idx / (NWI / GK), piece = (idx % (NWI / GK)) * 64u + lane;   // (a surplus wave repeats another's request)
        uint32_t mat;
        const uint32_t n = row_of(piece * 16u / ROWB, &mat);
        wptr[i] = (PAIR ? (mat ? a.seg[1].w : a.seg[0].w) : a.seg[si].w) + ((size_t)n * a.total_slabs + slab0 + sub) * ROWB + piece * 16u % ROWB;
        w_to[i] = A_BYTES + idx * 1024u;
    }
#pragma unroll
    for (uint32_t i = 0; i < CS; ++i) {
        const uint32_t idx = (wave + i * WAVES) % (2u * NSI), bias = idx >= NSI ? 1u : 0u, blk = idx - bias * NSI;
        uint32_t mat;
        const uint32_t n = row_of(blk * 64u + lane, &mat);
        const unsigned char* base = PAIR ? (bias ? (mat ? a.seg[1].bi : a.seg[0].bi) : (mat ? a.seg[1].sc : a.seg[0].sc))
                                         : (bias ? a.seg[si].bi : a.seg[si].sc);
        sptr[i] = base + (size_t)n * a.gpr * 2u + slab0 * 2u;
        s_to[i] = SC0 + bias * SC_BYTES + blk * 256u;
    }
    const unsigned char* xk = reinterpret_cast<const unsigned char*>(a.x) + (size_t)slab0 * 128u;
    // request R (of REQ) for the stage at `to`; advance: go on to the next slab behind it (the last one is requested again
    // by the stages that have no slab, so that every wait counts the same)
    uint32_t requested = 0;
    const uint32_t n_stages = n_slabs / GK;
    auto issue = [&](auto which, uint32_t to) {
        constexpr uint32_t R = (uint32_t)decltype(which)::value;
        if constexpr (R < CW) {
            dma16(to + w_to[R], wptr[R]);
        } else if constexpr (R < CW + CS) {
            dma4(to + s_to[R - CW], sptr[R - CW]);
        } else if constexpr (R < (uint32_t)REQ) {
            dma16(to + (wave * AR + R - CW - CS) * 1024u, xoff[R - CW - CS], xk);
        }
    };
    auto advance = [&]() {
        ++requested;
        const bool on = requested < n_stages;
        const uint32_t dw = on ? ROWB * GK : 0u, ds = on && (GK == 2 || (requested & 1u) == 0u) ? 4u : 0u;   // (GK = 1: two slabs share a dword of scales)
#pragma unroll
        for (uint32_t i = 0; i < CW; ++i) wptr[i] += dw;
#pragma unroll
        for (uint32_t i = 0; i < CS; ++i) sptr[i] += ds;
        xk += on ? 128u * GK : 0u;
    };
    auto issue_all = [&](uint32_t to) {
        static_for<REQ>([&](auto which) { issue(which, to); });
        advance();
    };

    f32x4_t acc[NI][NJ];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // the wave's fragments: activation row l16 of tile i, weight row l16 of tile j; in step st lane quarter kb holds
    // k = 16 kb + 8 st .. + 7 of the slab, of both operands
    const uint32_t arow = gk * 16384u + l16 * 128u;
    const uint32_t asw[2] = {((2u * kb) ^ (l16 >> 1)) * 16u, ((2u * kb + 1u) ^ (l16 >> 1)) * 16u};
    const uint32_t wrow = A_BYTES + gk * W_BYTES + (wn * (uint32_t)WTN + l16) * ROWB + kb * (ROWB / 4u);
    const uint32_t srow = SC0 + (wn * (uint32_t)WTN + l16) * 4u;

    // The pipeline of a wave: while the matrix instructions of a step (32 k) run, row fragments are read RING - 1 tiles ahead
    // and the next step's weights are unpacked, a few values behind each tile's matrix instructions.
    constexpr int RING = 4;
    fk_u32x4_t af[RING];
    uint4 codes[NJ];
    uint32_t wf[2][NJ][4], lo = 0, hi = 0;
    float fa = 0.f, fb = 0.f;
    float sf[NJ], s20[NJ], bf[NJ];
    auto read_codes = [&](uint32_t stage, uint32_t half) {   // half: the slab's of the 128 k that share a set
        const unsigned char* base = lds + stage;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if constexpr (KIND == W_Q4) {
                const uint2 v = *reinterpret_cast<const uint2*>(base + wrow + j * 16 * (int)ROWB);
                codes[j] = make_uint4(v.x, v.y, 0u, 0u);
            } else {
                codes[j] = *reinterpret_cast<const uint4*>(base + wrow + j * 16 * (int)ROWB);
            }
            const uint32_t s2 = *reinterpret_cast<const uint32_t*>(base + srow + j * 64);
            const uint32_t b2 = *reinterpret_cast<const uint32_t*>(base + srow + SC_BYTES + j * 64);
            const uint32_t take = half ? 0x03020c0cu : 0x01000c0cu;
            sf[j] = __uint_as_float(__builtin_amdgcn_perm(s2, s2, take));
            bf[j] = __uint_as_float(__builtin_amdgcn_perm(b2, b2, take));
            if constexpr (KIND == W_Q4) {
                s20[j] = sf[j] * 1048576.0f;
                sf[j] *= 16777216.0f;
            }
        }
    };
    auto read_row = [&](uint32_t stage, int st, int i) {
        af[i % RING] = *reinterpret_cast<const fk_u32x4_t*>(lds + stage + arow + asw[st] + i * 2048);
    };
    // A step's weights in NJ * 9 parts of at most two vector instructions: so many run under a 16-cycle matrix instruction
    // (one or two between each: 18.5 cycles; three 22.5, four 28 and more).  int4: a word's 17 instructions; half H of it gives
    // dwords H and H + 2.  int8: byte converts, multiply-adds and packs of the two words.
    auto unpack = [&](auto step, auto part) {
        constexpr int ST = decltype(step)::value, J = decltype(part)::value / 9, P = decltype(part)::value % 9;
        uint32_t(&out)[4] = wf[ST][J];
        if constexpr (KIND == W_Q4) {
            const uint32_t w = ST ? codes[J].y : codes[J].x;
            if constexpr (P == 0) { lo = w & 0x000F000Fu; pin(lo); hi = w & 0x00F000F0u; pin(hi); }
            if constexpr (P == 1 || P == 6) { fa = fmaf(half_of<0>(lo), sf[J], bf[J]); pin(fa); fb = fmaf(half_of<0>(hi), s20[J], bf[J]); pin(fb); }
            if constexpr (P == 2 || P == 7) { out[P == 7] = pack_bf16(fa, fb); pin(out[P == 7]); fa = fmaf(half_of<1>(lo), sf[J], bf[J]); pin(fa); }
            if constexpr (P == 3 || P == 8) { fb = fmaf(half_of<1>(hi), s20[J], bf[J]); pin(fb); out[2 + (P == 8)] = pack_bf16(fa, fb); pin(out[2 + (P == 8)]); }
            if constexpr (P == 4) { hi = w >> 8; pin(hi); lo = hi & 0x000F000Fu; pin(lo); }
            if constexpr (P == 5) { hi = hi & 0x00F000F0u; pin(hi); }
        } else if constexpr (P < 8) {
            constexpr int D = P / 2, B = 2 * (D % 2);   // dword D from bytes B, B + 1 of a word
            const uint32_t w = D / 2 ? (ST ? codes[J].w : codes[J].y) : (ST ? codes[J].z : codes[J].x);
            if constexpr (P % 2 == 0) { fa = byte_of<B>(w); pin(fa); fb = byte_of<B + 1>(w); pin(fb); }
            if constexpr (P % 2 == 1) { out[D] = pack_bf16(fmaf(fa, sf[J], bf[J]), fmaf(fb, sf[J], bf[J])); pin(out[D]); }
        }
    };
    // Step ST of the slab at `stage`; `next`: the stage of the step behind it, whose codes have been requested (behind the
    // last step a stage is read whose values nobody uses).
    // FILLS: requests for the stage `fill` go out between the tiles (all at once they hold every wave up behind the barrier).
    auto multiply = [&](auto step, uint32_t stage, uint32_t next, auto fills, uint32_t fill) {
        constexpr int ST = decltype(step)::value, PARTS = NJ * 9, SLOTS = (NI - 2) * NJ;   // (the first two tiles: the codes are on their way)
        static_for<NI>([&](auto tile) {
            constexpr int I = decltype(tile)::value, A = I + RING - 1;
            if constexpr (A < NI)
                read_row(stage, ST, A);
            else
                read_row(next, ST ^ 1, A - NI);
            if constexpr (decltype(fills)::value) issue(tile, fill);
            static_for<NJ>([&](auto col) {   // a matrix instruction, then a little vector work under it
                constexpr int J = decltype(col)::value, SLOT = (I - 2) * NJ + J;
                mfma_acc(acc[I][J], wf[ST][J], af[I % RING]);
                if constexpr (SLOT >= 0) {
                    constexpr int P0 = SLOT * PARTS / SLOTS, P1 = (SLOT + 1) * PARTS / SLOTS;
                    static_for<P1 - P0>([&](auto n) { unpack(std::integral_constant<int, ST ^ 1>{}, std::integral_constant<int, P0 + decltype(n)::value>{}); });
                }
            });
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // Slab k: its second step opens with a wait for this wave's requests of slab k + 1 and a barrier, behind which that slab
    // is everybody's (the step reads its codes and first rows).  Requests for slab k + NST - 1 go into the stage of slab k - 1,
    // which nobody reads behind the first barrier of slab k: from the first step on with three stages (a barrier of its own),
    // in the second with four; either way two slabs are on their way.
    typedef std::integral_constant<int, 0> Step0;
    typedef std::integral_constant<int, 1> Step1;
    typedef std::integral_constant<bool, NST == 3> Fill0;
    typedef std::integral_constant<bool, NST == 4> Fill1;
    issue_all(0);
    issue_all(STAGE);
    if constexpr (NST == 4) issue_all(2u * STAGE);
    wait_loads<REQ * (int)(NST - 2u)>();
    barrier();
    read_codes(0, gk);
#pragma unroll
    for (int i = 0; i < RING - 1; ++i) read_row(0, 0, i);
    static_for<NJ * 9>([&](auto part) { unpack(Step0{}, part); });
    uint32_t st = 0, fill = (NST - 1u) * STAGE, odd = 0;   // byte offsets of the stages
    auto after = [&](uint32_t s) { return s + STAGE == NST * STAGE ? 0u : s + STAGE; };
#pragma unroll 1
    for (uint32_t k = 0; k < n_stages; ++k) {
        const uint32_t next = after(st);
        if constexpr (NST == 3) barrier();
        multiply(Step0{}, st, st, Fill0{}, fill);
        wait_loads<REQ>();
        barrier();
        odd ^= 1u;
        read_codes(next, GK == 2 ? gk : odd);
        multiply(Step1{}, st, next, Fill1{}, fill);
        advance();
        st = next;
        fill = after(fill);
    }
    wait_loads<0>();
    settle_matrix_ops();
    barrier();

    // ---- outputs: register r of a lane is weight row 4 kb + r of its tile, activation row l16
    constexpr int NR = NI / GK;   // row tiles that this wave finishes, from mrow0
    const uint32_t mrow0 = m0 + gk * 64u;
    f32x4_t* const ex = reinterpret_cast<f32x4_t*>(lds) + (size_t)(SPLIT_PAIR ? wn & 1u : wn) * NI * NJ * 64u + lane;
    if constexpr (GK == 2) {   // each group finishes half of the rows: the other half's sums go to the other group
        static_for<NI>([&](auto i) {
            constexpr int I = decltype(i)::value;
            if ((I >= NR) != (gk != 0u)) static_for<NJ>([&](auto j) { ex[(I * NJ + decltype(j)::value) * 64] = take(acc[I][decltype(j)::value]); });
        });
        __syncthreads();
        static_for<NR>([&](auto i) {
            static_for<NJ>([&](auto j) {
                constexpr int I = decltype(i)::value, J = decltype(j)::value;
                const f32x4_t own = gk ? take(acc[I + NR][J]) : take(acc[I][J]), o = ex[((gk ? I + NR : I) * NJ + J) * 64];
                acc[I][J] = gk ? o + own : own + o;   // the first group's sums first, whichever group adds
            });
        });
    }
    const bool finished = a.partial == nullptr;
    if constexpr (SPLIT_PAIR) {
        if (!finished) {
            float* p = wn >= 2u ? a.partial2 : a.partial;
            static_for<NR>([&](auto i) {
                static_for<NJ>([&](auto j) {
                    constexpr int I = decltype(i)::value, J = decltype(j)::value;
                    const uint32_t m = mrow0 + I * 16u + l16, n = n0 + (wn & 1u) * (uint32_t)WTN + J * 16u + 4u * kb;
                    if (m < a.M && n < N) *reinterpret_cast<f32x4_t*>(p + ((size_t)ks * a.M + m) * N + n) = take(acc[I][J]);
                });
            });
            return;
        }
        // the up waves hand their sums to the gate waves through LDS, and take every second row tile back finished half-way:
        // gate wave w finishes the even row tiles, up wave w + 2 the odd ones
        static_for<NR>([&](auto i) {
            constexpr int I = decltype(i)::value;
            if ((wn >= 2u) != (I % 2 != 0)) static_for<NJ>([&](auto j) { ex[(I * NJ + decltype(j)::value) * 64] = take(acc[I][decltype(j)::value]); });
        });
        __syncthreads();
        auto finish = [&](auto fast) {
            static_for<NR / 2>([&](auto i) {
                static_for<NJ>([&](auto j) {
                    constexpr int I = decltype(i)::value * 2, J = decltype(j)::value;
                    const bool up = wn >= 2u;
                    const f32x4_t own = up ? take(acc[I + 1][J]) : take(acc[I][J]), o = ex[((up ? I + 1 : I) * NJ + J) * 64];
                    const uint32_t m = mrow0 + (up ? I + 1 : I) * 16u + l16, n = n0 + (wn & 1u) * (uint32_t)WTN + J * 16u + 4u * kb;
                    store_swiglu<decltype(fast)::value>(a, m, n, N, up ? o : own, up ? own : o);
                });
            });
        };
        a.variant == 1 ? finish(std::true_type{}) : finish(std::false_type{});
    } else if constexpr (PAIR) {
        // (What is done with the sums is chosen once: chosen at every output, the code that a tile's end runs through lies
        // scattered over 110 KB, more than the instruction cache holds: 4096 rows of the 9728 x 2560 pair 402 us, this way 372.)
        auto each = [&](auto store) {
            static_for<NR>([&](auto i) {
                static_for<NJ / 2>([&](auto j) {
                    constexpr int I = decltype(i)::value, J = decltype(j)::value;
                    store(mrow0 + I * 16u + l16, n0 + wn * (WTN / 2u) + J * 16u + 4u * kb, take(acc[I][J]), take(acc[I][J + NJ / 2]));
                });
            });
        };
        if (!finished)
            each([&](uint32_t m, uint32_t n, const f32x4_t& g, const f32x4_t& u) {
                if (m >= a.M || n >= N) return;
                *reinterpret_cast<f32x4_t*>(a.partial + ((size_t)ks * a.M + m) * N + n) = g;
                *reinterpret_cast<f32x4_t*>(a.partial2 + ((size_t)ks * a.M + m) * N + n) = u;
            });
        else if (a.variant == 1)
            each([&](uint32_t m, uint32_t n, const f32x4_t& g, const f32x4_t& u) { store_swiglu<true>(a, m, n, N, g, u); });
        else
            each([&](uint32_t m, uint32_t n, const f32x4_t& g, const f32x4_t& u) { store_swiglu<false>(a, m, n, N, g, u); });
    } else {
        uint16_t* y = a.seg[si].y;
        const uint16_t* bias = a.seg[si].bias;
        static_for<NJ>([&](auto j) {
            constexpr int J = decltype(j)::value;
            const uint32_t n = n0 + wn * (uint32_t)WTN + J * 16u + 4u * kb;
            if (n >= N) return;
            if (!finished) {
                static_for<NR>([&](auto i) {
                    const uint32_t m = mrow0 + decltype(i)::value * 16u + l16;
                    if (m < a.M) *reinterpret_cast<f32x4_t*>(a.partial + ((size_t)ks * a.M + m) * a.row_cols + a.seg[si].col0 + n) = take(acc[decltype(i)::value][J]);
                });
                return;
            }
            const uint2 b2 = bias ? *reinterpret_cast<const uint2*>(bias + n) : make_uint2(0u, 0u);
            uint2 r2[NR];   // (requested together: under the row test each load would be waited for by itself)
            if (a.res)
                static_for<NR>([&](auto i) {
                    const uint32_t m = mrow0 + decltype(i)::value * 16u + l16;
                    r2[decltype(i)::value] = *reinterpret_cast<const uint2*>(a.res + (size_t)(m < a.M ? m : a.M - 1u) * N + n);
                });
            static_for<NR>([&](auto i) {
                constexpr int I = decltype(i)::value;
                const uint32_t m = mrow0 + I * 16u + l16;
                f32x4_t v = take(acc[I][J]);
                if (bias) {
                    v[0] += bf16_lo(b2.x); v[1] += bf16_hi(b2.x); v[2] += bf16_lo(b2.y); v[3] += bf16_hi(b2.y);
                }
                if (a.res) {
                    v[0] += bf16_lo(r2[I].x); v[1] += bf16_hi(r2[I].x); v[2] += bf16_lo(r2[I].y); v[3] += bf16_hi(r2[I].y);
                }
                if (m < a.M) *reinterpret_cast<uint2*>(y + (size_t)m * N + n) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
            });
        });
    }
}

namespace {

template <WKind KIND, bool PAIR>
const void* dma_func(int gk, int wtn) {
#define FK_DMA(GK, WTN) \
    if (gk == GK && wtn == WTN) return reinterpret_cast<const void*>(&qgemm_dma_kernel<KIND, GK, WTN, PAIR>);
    FK_DMA(1, 64) FK_DMA(1, 48) FK_DMA(1, 32) FK_DMA(2, 32)
    if constexpr (KIND == W_Q4) FK_DMA(2, 64)
#undef FK_DMA
    return nullptr;
}

struct DmaChoice {
    int gk = 1, wtn = 64;
    uint32_t split = 1;
};

// Which tile, and how many k splits: the least of rounds x (stages x time of a stage + time of a tile) + second kernel, with
// the times as measured on a full chip (us; int4, int8 within 4 %), rounds = tiles over CUs rounded up.  By the times per flop
// the largest tile would always win (1.77 us for 256 x 256 x 64 is 1.2 PFLOP/s over 256 CUs, 256 x 128 takes 1.0): the smaller
// ones are there for what the last round leaves empty.  Depends on the rows in steps of 128 only, so that a workspace sized
// for a multiple of 128 rows serves the counts below it.
DmaChoice dma_choose(uint32_t cus, uint32_t bits, uint32_t M, uint32_t N, uint32_t K, bool pair) {
    static const struct {
        int gk, wtn;
        float stage_us, tile_us;
    } forms[] = {{1, 64, 1.77f, 6.f}, {1, 48, 1.36f, 6.f}, {1, 32, 1.0f, 4.f}, {2, 64, 1.95f, 5.f}, {2, 32, 1.28f, 4.f}};
    const uint32_t rows = (M + 127u) / 128u * 128u, pairs_k = K / 128u;
    DmaChoice best;
    float best_us = 1e30f;
    for (const auto& f : forms) {
        if (f.gk == 2 && f.wtn == 64 && bits != 4) continue;   // (its stages do not fit the LDS)
        const uint32_t bm = f.gk == 1 ? 256u : 128u, bn = 4u * f.wtn;
        const uint32_t tiles = ((rows + bm - 1u) / bm) * (((pair ? 2u : 1u) * N + bn - 1u) / bn);
        for (uint32_t split = 1; split <= 12u && split <= pairs_k; ++split) {
            const uint32_t per = (pairs_k + split - 1u) / split;   // 128 k each
            if (split > 1 && ((pairs_k + per - 1u) / per != split || tiles * split > cus)) continue;
            const uint32_t rounds = (tiles * split + cus - 1u) / cus;
            float us = (float)rounds * ((float)(f.gk == 1 ? 2u * per : per) * f.stage_us + f.tile_us);
            if (split > 1) us += 3.f + (float)(split + 1u) * 4e-6f * (float)rows * (float)N * (pair ? 2.f : 1.f) / 3.5f;
            if (us < best_us) {
                best_us = us;
                best.gk = f.gk;
                best.wtn = f.wtn;
                best.split = split;
            }
        }
    }
    return best;
}

}  // namespace

uint32_t qgemm_dma_split(uint32_t bits, uint32_t M, uint32_t N, uint32_t K, bool pair) {
    const DeviceFacts* dev;
    if (M < 65u || K % 128u || device_facts(&dev) != FK_OK) return 1u;
    return dma_choose((uint32_t)dev->cus, bits, M, N, K, pair).split;
}

// (K < 768: the pipeline fills and drains over less than six stages of 128 k; there the tiles of qgemm.hip are as fast)
bool qgemm_takes_dma(const DmaRequest& rq) {
    if (rq.M < 65u || !rq.x || !rq.workspace || !rq.W[0] || rq.W[0]->k < 768u) return false;
    for (uint32_t i = 0; i < rq.n_mats; ++i) {
        const fk_weight* W = rq.W[i];
        if (!W || !W->w || !W->scales || !W->biases || !(rq.y[i] || (rq.pair && i)) || W->n == 0 || W->k != rq.W[0]->k || (rq.pair && W->n != rq.W[0]->n)) return false;
        if (W->group != 64 || W->k % 128u || W->n % 4u || (W->bits != 4 && W->bits != 8) || W->bits != rq.W[0]->bits) return false;
        if (((uintptr_t)W->w & 15u) || ((uintptr_t)W->scales & 3u) || ((uintptr_t)W->biases & 3u)) return false;
        if (((uintptr_t)rq.bias[i] | (uintptr_t)rq.y[i]) & 7u) return false;
    }
    uint64_t outputs = 0;
    for (uint32_t i = 0; i < rq.n_mats; ++i) outputs += (uint64_t)rq.M * rq.W[i]->n;
    return outputs <= 0x7fffffffull && (uint64_t)rq.M * rq.W[0]->k * 2u < (1ull << 32) && (((uintptr_t)rq.x | (uintptr_t)rq.workspace) & 15u) == 0 && ((uintptr_t)rq.res & 7u) == 0;
}

fk_status plan_qgemm_dma(const DmaRequest& rq, Launch* main, Launch* reduce) {
    const DeviceFacts* dev;
    FK_TRY(device_facts(&dev));
    const uint32_t K = rq.W[0]->k;
    uint32_t n_total = 0;
    for (uint32_t i = 0; i < (rq.pair ? 1u : rq.n_mats); ++i) n_total += rq.W[i]->n;
    const DmaChoice c = dma_choose((uint32_t)dev->cus, rq.W[0]->bits, rq.M, n_total, K, rq.pair);
    const int gk = c.gk, wtn = c.wtn;
    const uint32_t split = c.split;
    const uint32_t bm = gk == 1 ? 256u : 128u, bn = 4u * wtn, per = rq.pair ? bn / 2u : bn;
    QgemmDmaArgs a;
    memset(&a, 0, sizeof(a));
    a.x = rq.x;
    a.M = rq.M;
    a.K = K;
    a.gpr = K / 64u;
    a.total_slabs = K / 64u;
    a.slabs = ((a.total_slabs / 2u + split - 1u) / split) * 2u;
    a.ksplit = (a.total_slabs + a.slabs - 1u) / a.slabs;
    a.m_blocks = (rq.M + bm - 1u) / bm;
    a.n_seg = rq.pair ? 1u : rq.n_mats;
    a.row_cols = n_total;
    a.res = rq.res;
    a.variant = rq.variant;
    uint32_t nb = 0, col = 0;
    for (uint32_t i = 0; i < 3; ++i) {
        const uint32_t j = i < rq.n_mats ? i : rq.n_mats - 1u;
        const fk_weight* W = rq.W[j];
        auto& s = a.seg[i];
        s.w = static_cast<const unsigned char*>(static_cast<const void*>(W->w));
        s.sc = reinterpret_cast<const unsigned char*>(W->scales);
        s.bi = reinterpret_cast<const unsigned char*>(W->biases);
        s.y = rq.y[j];
        s.bias = rq.bias[j];
        s.N = W->n;
        if (i < a.n_seg) nb += (W->n + per - 1u) / per;
        s.nb_end = i < a.n_seg ? nb : 0xffffffffu;
        s.col0 = col;
        if (i + 1u < a.n_seg) col += W->n;
    }
    a.n_blocks = nb;
    a.tiles = nb * a.m_blocks;
    if (a.ksplit > 1u) {
        a.partial = static_cast<float*>(rq.workspace);
        a.partial2 = a.partial + (size_t)a.ksplit * rq.M * n_total;
    }
    const bool q4 = rq.W[0]->bits == 4;
    main->func = q4 ? (rq.pair ? dma_func<W_Q4, true>(gk, wtn) : dma_func<W_Q4, false>(gk, wtn))
                    : (rq.pair ? dma_func<W_Q8, true>(gk, wtn) : dma_func<W_Q8, false>(gk, wtn));
    main->grid = dim3(a.tiles * a.ksplit, 1, 1);
    main->block = dim3(64u * dma_waves(gk), 1, 1);
    main->shmem = dma_lds_bytes(q4 ? W_Q4 : W_Q8, gk, wtn);
    FK_TRY(raise_dynamic_lds(main->func, main->shmem));
    main->set_args(a);
    *reduce = Launch();
    if (rq.sums) *rq.sums = FanSums{a.ksplit > 1u ? a.partial : nullptr, a.ksplit, n_total};
    if (a.ksplit > 1u && !rq.sums) plan_qgemm_dma_reduce(rq, n_total, a.ksplit, reduce);
    return FK_OK;
}

}  // namespace fk
