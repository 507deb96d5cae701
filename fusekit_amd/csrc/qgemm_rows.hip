// Multi-row matmul for up to 64 activation rows: y[M, N] = epilogue(x[M, K] @ dequant(W)^T) in ONE launch, for a single
// matrix, a gate / up pair with SwiGLU, or up to three matrices over the same rows (q / k / v), the rows RMS-normalised
// on the way in if asked.  Replaces the reference's small-M kernels (fusekit_qmv_wide_impl, src/codegen/msl.rs:462-546;
// fusekit_qmv_fast_m_impl, :1307-1485; policy src/codegen/kernels/mod.rs:164-186), the emitters compiled with active_m > 1
// (src/codegen/kernels/rmsnorm_qkv.rs:53-736, rmsnorm_gateup_swiglu.rs:20-330) and its qMM path up to 64 rows
// (src/codegen/msl.rs:2318-2440, src/codegen/kernels/mod.rs:1442-1475).
//
// What bounds these launches is latency first (a 0.5B-class projection is half a megabyte) and the address rate of the
// vector memory unit second.  So no second kernel and no workspace: a block owns 16 (32) weight rows over ALL of K and its
// eight waves split K into runs of quantisation groups; they meet in LDS, are added in wave order and the epilogue follows.
// v_mfma_f32_16x16x32_bf16 with the weights as the B operand.  Its fragments want neighbouring lanes in different rows;
// requested that way from memory (sixteen lines per instruction, a stride that is a power of two) 64 rows of 2560 x 4096
// took 30 us, so every wave requests whole 128-byte lines, eight lanes a row, and turns them round in its OWN piece of LDS
// (LDS operations of a wave execute in order: the main loop has no barrier).  Two slabs of weights and two groups of
// activations are in flight per wave.  The arithmetic is that of the exact form: the integer codes enter as exact bf16
// values, a group's dot product is accumulated from zero in fp32 and folded as s * dot + b * Sx; Sx, the group's activation
// sum, is one more matrix instruction per step against a B operand of ones, which leaves it in the very registers the fold
// needs.
// 37 rows of int4, one call in a chain, before (32 x 32 x 16 tiles, split-k sums, second kernel) / now: 896 x 896 12.8 / 3.6
// us, 4864 x 896 pair 26.3 / 6.9, 896 x 4864 17.8 / 7.0, 2560 x 4096 19.8 / 9.5, 9728 x 2560 pair 53.0 / 24.6; 8 rows (a
// form of its own for 2..10 rows) 896 x 896 4.65 / 3.34, 2560 x 4096 8.80 / 6.2, 2560 x 9728 14.4 / 12.7.
#include "fk_host.hpp"
#include "gemv_kernel.hpp"

namespace fk {

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
// 16 bytes of an operand, which need not lie on their own alignment (a row of a larger tensor, a matrix inside a file): the
// vector memory unit takes any address, and the type keeps the compiler from assuming more.  The same instructions.
typedef uint32_t u32x4_any_t __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x2_any_t __attribute__((ext_vector_type(2), aligned(2)));

constexpr uint32_t kRowsMax = 64;   // activation rows: four tiles of 16

struct QgemmRowsArgs {
    const uint4* w[3];   // the matrix, the gate / up pair, or up to three matrices served side by side
    const uint16_t* sc[3];
    const uint16_t* bi[3];
    const uint16_t* bias[3];
    uint16_t* y[3];
    uint32_t n[3], blk0[3];   // rows of matrix i, its first block
    uint32_t y_stride[3];     // elements between the rows of y[i]
    const uint16_t* x;        // M rows of K values, x_stride apart
    const uint16_t* res;      // like y[0], or null (single matrix)
    const uint16_t* norm_w;   // the rows enter as T(w * T(x * r)), r = 1 / rms of the row; null: as they are
    // sums of squares of the rows, as the launch that wrote them left them (or null: formed here, in one more pass over
    // the rows): ssq_in[row * ssq_n + i], i < ssq_n; and where this launch leaves those of its outputs (single matrix)
    const float* ssq_in;
    float* ssq_out;
    uint32_t ssq_n;
    float eps;
    uint32_t M, K, n_seg, x_stride;
    uint32_t gshift;          // 64-code groups per scale: 0 (group 64), 1 (group 128)
    int variant;
};

constexpr uint32_t kRowsLine = 9;   // uint4 per staged 128-byte line (8 used: the ninth spreads the banks)
// groups of 64 columns per 128-byte line of a weight row
__host__ __device__ constexpr uint32_t rows_slab_groups(uint32_t bits) { return bits == 4 ? 4u : (bits == 8 ? 2u : 1u); }
// One wave: activation lines of a group, weight lines of a slab, (scale, bias) pairs of a slab (ONE: scales, then biases, of four
// groups, and four groups of the norm weights).
__host__ __device__ constexpr uint32_t rows_wave_lds(uint32_t mt, uint32_t nt) { return (mt + nt) * 16u * kRowsLine * 16u + nt * 16u * 4u * 4u + 4u * 128u; }
__host__ __device__ constexpr uint32_t rows_lds_bytes(uint32_t mt, uint32_t nt, uint32_t waves) {
    const uint32_t stage = waves * (rows_wave_lds(mt, nt) + mt * 16u * 4u), meet = waves * mt * nt * 256u * 4u;   // one after the other
    return stage > meet ? stage : meet;
}

// Eight codes of a row, in order, as the eight bf16 values of a B fragment.
template <WKind KIND>
__device__ __forceinline__ uint4 rows_unpack(uint32_t w0, uint32_t w1) {
    uint4 b;
    if constexpr (KIND == W_Q4) {
        const uint32_t even = w0 & 0x0F0F0F0Fu, odd = (w0 >> 4) & 0x0F0F0F0Fu;
        const uint32_t lo = __builtin_amdgcn_perm(odd, even, 0x05010400u), hi = __builtin_amdgcn_perm(odd, even, 0x07030602u);
        b.x = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, false));
        b.y = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, true));
        b.z = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, false));
        b.w = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, true));
    } else {
        b.x = pack_bf16((float)(w0 & 0xffu), (float)((w0 >> 8) & 0xffu));   // integers up to 255 are exact in bf16
        b.y = pack_bf16((float)((w0 >> 16) & 0xffu), (float)(w0 >> 24));
        b.z = pack_bf16((float)(w1 & 0xffu), (float)((w1 >> 8) & 0xffu));
        b.w = pack_bf16((float)((w1 >> 16) & 0xffu), (float)(w1 >> 24));
    }
    return b;
}

// MT tiles of 16 activation rows, NT tiles of 16 weight rows (PAIR: NT / 2 of the gate matrix and as many of the up matrix).
// ONE: no wave has more than one slab of K (quantised; K up to 1024 int4 columns with four waves, 2048 with eight).  Everything
// is then asked for exactly once, in straight line -- the loop below asks two slabs and two groups past its range, two thirds of
// all requests at K = 896, and a CU issues one per 16 .. 20 cycles --, the four groups' scales and biases with one request for
// all tiles, the norm weights with one.  Both forms ask for what the epilogue adds together with the first slab, not after the
// waves have met.  The loop with its operands late / now, 37 rows of int4 with a residual, one call in a chain: 896 x 896 3.70 /
// 3.42 us, 4864 x 896 7.48 / 6.98 (pair 8.98 / 8.61), 1024 x 2048 4.93 / 4.54, 2560 x 2048 7.56 / 6.84; the loop itself with
// its operands early: 896 x 4864 7.55 / 7.14, 2560 x 4096 10.48 / 10.10.  The same sums in the same order.
template <WKind KIND, bool PAIR, int NT, int MT, int WAVES, bool ONE>
__global__ __launch_bounds__(WAVES* kWave, 2) void qgemm_rows_kernel(const QgemmRowsArgs a) {
    constexpr int CT = PAIR ? NT / 2 : NT;                                      // output tiles of a block
    constexpr uint32_t BITS = KIND == W_Q4 ? 4u : (KIND == W_Q8 ? 8u : 16u);
    constexpr uint32_t SG = rows_slab_groups(BITS);
    extern __shared__ uint4 lds_raw[];
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t c16 = lane & 15u, kq = lane >> 4, l8 = lane & 7u, r8 = lane >> 3;
    uint32_t seg = 0;
    if constexpr (!PAIR) {
        if (a.n_seg > 1 && blockIdx.x >= a.blk0[1]) seg = 1;
        if (a.n_seg > 2 && blockIdx.x >= a.blk0[2]) seg = 2;
    }
    const uint32_t m0 = blockIdx.y * (MT * 16u), M = a.M - m0 < MT * 16u ? a.M - m0 : MT * 16u;   // this block's activation rows
    const uint32_t blk = blockIdx.x - a.blk0[seg], N = a.n[seg], K = a.K, G = K >> 6, gpr = G >> a.gshift;
    const uint32_t g0 = wave * G / WAVES, g1 = (wave + 1u) * G / WAVES;
    u32x4_t* xs = reinterpret_cast<u32x4_t*>(reinterpret_cast<char*>(lds_raw) + wave * rows_wave_lds(MT, NT));   // [MT * 16][kRowsLine]
    u32x4_t* wl = xs + MT * 16 * kRowsLine;                                                                    // [NT * 16][kRowsLine]
    uint32_t* ml = reinterpret_cast<uint32_t*>(wl + NT * 16 * kRowsLine);                                    // [NT * 16][4]
    [[maybe_unused]] uint16_t* sl = reinterpret_cast<uint16_t*>(ml);                                         // ONE: [NT][2][16][4]
    [[maybe_unused]] u32x4_t* nl = reinterpret_cast<u32x4_t*>(ml + NT * 64);                                 // ONE: [4][8]

    // request roles: line `r8 + 8 h` of a tile, its piece l8; scale and bias of row lane / 4, group lane % 4
    // (uniform bases and 32-bit lane offsets: full pointers cost the registers that let a second wave share the SIMD)
    const unsigned char *wbase[NT], *sbase[NT], *bbase[NT];
    uint32_t woff[NT][2], soff[NT], xoff[MT][2];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const uint32_t mat = PAIR ? (uint32_t)(t / CT) : seg, n0 = (blk * CT + (uint32_t)(t % CT)) * 16u;
        const uint32_t first = n0 < N ? n0 : N - 1, row_bytes = K / 8u * BITS;
        auto row = [&](uint32_t r) { return n0 + r < N ? n0 + r - first : N - 1 - first; };   // (past the end: the last row, not stored)
        wbase[t] = reinterpret_cast<const unsigned char*>(a.w[mat]) + (size_t)first * row_bytes;
        sbase[t] = reinterpret_cast<const unsigned char*>(a.sc[mat]) + (KIND == W_BF16 ? 0u : (size_t)first * gpr * 2u);
        bbase[t] = reinterpret_cast<const unsigned char*>(a.bi[mat]) + (KIND == W_BF16 ? 0u : (size_t)first * gpr * 2u);
#pragma unroll
        for (int h = 0; h < 2; ++h) woff[t][h] = row(r8 + 8u * (uint32_t)h) * row_bytes;
        soff[t] = row(lane >> 2) * gpr * 2u;
    }
    const unsigned char* xbase = reinterpret_cast<const unsigned char*>(a.x + (size_t)m0 * a.x_stride);
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t m = (uint32_t)t * 16u + r8 + 8u * (uint32_t)h;
            xoff[t][h] = ((m < M ? m : M - 1) * a.x_stride + l8 * 8u) * 2u;
        }
    const bool normed = a.norm_w != nullptr;                        // block-uniform
    const unsigned char* nbase = normed ? reinterpret_cast<const unsigned char*>(a.norm_w) : xbase;   // (without a norm: unused)

    f32x4_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    struct Slab {
        u32x4_t w[NT][2];   // (native vectors: copied as structures they stay in scratch)
        uint32_t sc[NT], bi[NT];
    };
    struct Acts {
        u32x4_t x[MT][2], nw;
    };
    // ONE: four entries of each row's scales and biases, from the wave's first group or, at a row's end, the row's last four
    [[maybe_unused]] const uint32_t e_first = ONE ? ((g0 >> a.gshift) + 4u <= gpr ? g0 >> a.gshift : gpr - 4u) : 0u;
    // What the epilogue's first outputs of this thread add (a null operand reads the activations instead and is not used: asked for
    // under a condition 37 rows of 6144 x 2560 are at 12.4 us instead of 11.9).
    constexpr uint32_t OUT = 16u * CT;
    constexpr int EARLY = MT * NT > 6 ? 0 : 2;   // (beyond, no registers are left for them: 64 rows of 6144 x 2560 at 16.7 us instead of 14.9)
    const uint32_t yst = a.y_stride[seg];
    const uint16_t* res = a.res ? a.res + (size_t)m0 * yst : nullptr;
    const uint16_t* bias = a.bias[seg];
    [[maybe_unused]] uint32_t e_bias[EARLY + 1] = {}, e_res[EARLY + 1] = {};
    auto fetch_epilogue = [&]() __attribute__((always_inline)) {
        if constexpr (!PAIR) {
#pragma unroll
            for (int k = 0; k < EARLY; ++k) {
                const uint32_t e = (uint32_t)k * (WAVES * kWave) + threadIdx.x, m = e / OUT, n = blk * OUT + e % OUT;
                const uint32_t mc = m < M ? m : M - 1u, nc = n < N ? n : N - 1u;
                e_bias[k] = *(bias ? bias + nc : a.x);
                e_res[k] = *(res ? res + (size_t)mc * yst + nc : a.x);
            }
        }
    };
    // Straight-line requests: what lies past the wave's range (or the row) is clamped to its last piece and never used.
    const uint32_t gl = g1 > g0 ? g1 - 1u : (g0 < G ? g0 : G - 1u);
    auto fetch_w = [&](uint32_t g, Slab& s) __attribute__((always_inline)) {   // groups g .. g + SG - 1
        constexpr uint32_t PPG = 8u / SG;        // 16-byte pieces per group
        const uint32_t gp = g + l8 / PPG, gc = gp < gl ? gp : gl;
        const uint32_t at = (gc * PPG + l8 % PPG) * 16u;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
#pragma unroll
            for (int h = 0; h < 2; ++h) s.w[t][h] = *reinterpret_cast<const u32x4_any_t*>(wbase[t] + (woff[t][h] + at));
            if constexpr (KIND != W_BF16 && !ONE) {
                const uint32_t gm = g + (lane & 3u), gmc = (gm < gl ? gm : gl) >> a.gshift;
                s.sc[t] = *reinterpret_cast<const uint16_t*>(sbase[t] + (soff[t] + gmc * 2u));
                s.bi[t] = *reinterpret_cast<const uint16_t*>(bbase[t] + (soff[t] + gmc * 2u));
            }
        }
    };
    auto fetch_x = [&](uint32_t g, Acts& s) __attribute__((always_inline)) {
        const uint32_t gc = g < gl ? g : gl;
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h) s.x[t][h] = *reinterpret_cast<const u32x4_any_t*>(xbase + (xoff[t][h] + gc * 128u));
        if constexpr (!ONE) s.nw = *reinterpret_cast<const u32x4_any_t*>(nbase + (l8 * 16u + gc * 128u));
    };
    const uint4 ones4 = make_uint4(0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u);
    const bf16x8_t ones = __builtin_bit_cast(bf16x8_t, ones4);
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    auto consume = [&](uint32_t u) __attribute__((always_inline)) {   // group u of the parked slab
        bf16x8_t xa[MT][2];
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) xa[i][j] = __builtin_bit_cast(bf16x8_t, xs[((uint32_t)i * 16u + c16) * kRowsLine + kq * 2u + (uint32_t)j]);
        if constexpr (KIND == W_BF16) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const bf16x8_t bw = __builtin_bit_cast(bf16x8_t, wl[((uint32_t)t * 16u + c16) * kRowsLine + kq * 2u + (uint32_t)j]);
#pragma unroll
                    for (int i = 0; i < MT; ++i) acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[i][j], bw, acc[i][t], 0, 0, 0);
                }
        } else {
            f32x4_t sx[MT];
#pragma unroll
            for (int i = 0; i < MT; ++i) sx[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[i][0], ones, zero, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < MT; ++i) sx[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[i][1], ones, sx[i], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const u32x4_t* line = wl + ((uint32_t)t * 16u + c16) * kRowsLine;
                uint4 b0, b1;
                if constexpr (KIND == W_Q4) {
                    const uint2 v = reinterpret_cast<const uint2*>(line)[u * 4u + kq];
                    b0 = rows_unpack<KIND>(v.x, 0u);
                    b1 = rows_unpack<KIND>(v.y, 0u);
                } else {
                    const u32x4_t v = line[u * 4u + kq];
                    b0 = rows_unpack<KIND>(v.x, v.y);
                    b1 = rows_unpack<KIND>(v.z, v.w);
                }
                float sf, bf;
                if constexpr (ONE) {
                    const uint16_t* at = sl + (uint32_t)t * 128u + c16 * 4u + (((g0 + u) >> a.gshift) - e_first);
                    sf = bf16_bits_to_f32(at[0]);
                    bf = bf16_bits_to_f32(at[64]);
                } else {
                    const uint32_t sb = ml[((uint32_t)t * 16u + c16) * 4u + u];
                    sf = bf16_lo(sb);
                    bf = bf16_hi(sb);
                }
                f32x4_t c[MT];
#pragma unroll
                for (int i = 0; i < MT; ++i) c[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[i][0], __builtin_bit_cast(bf16x8_t, b0), zero, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < MT; ++i) c[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[i][1], __builtin_bit_cast(bf16x8_t, b1), c[i], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[i][t][r] += fmaf(sf, c[i][r], bf * sx[i][r]);
            }
        }
    };
    Slab w0;
    [[maybe_unused]] Slab w1;
    Acts x0, x1;
    // One slab and one tile of rows: all four of the slab's groups of activations are in flight, not two, a trip to the L2 less.  Two / four,
    // us: 37 rows of 896 x 896 3.70 / 3.59, 8 rows of 3072 x 2048 4.85 / 4.73, of 2048 x 2048 4.60 / 4.43, 16 of the 4864 x 896 pair 5.53 /
    // 5.38.  More tiles and several slabs keep two: 37 rows of that pair 8.54 / 8.83, 24 rows of 3072 x 2048 5.80 / 6.02 (registers), 8
    // rows of 2560 x 4096 6.36 / 6.75 (what is asked for past a wave's range).
    constexpr bool ALL_X = ONE && MT == 1 && SG == 4u;
    [[maybe_unused]] Acts x2, x3;
    [[maybe_unused]] u32x2_any_t meta;
    [[maybe_unused]] u32x4_t norms;
    if constexpr (ONE) {
        // lane: tile lane / 32, scales or biases, row lane % 16 (one tile: its upper half repeats it)
        const uint32_t t = NT > 1 ? lane >> 5 : 0u;
        const unsigned char *sfrom = NT > 1 && t ? sbase[NT - 1] : sbase[0], *bfrom = NT > 1 && t ? bbase[NT - 1] : bbase[0];
        const unsigned char* from = lane & 16u ? bfrom : sfrom;
        const uint32_t n0 = (blk * CT + (PAIR ? 0u : t)) * 16u, first = n0 < N ? n0 : N - 1u, r = first + c16 < N ? c16 : N - 1u - first;
        meta = *reinterpret_cast<const u32x2_any_t*>(from + (r * gpr + e_first) * 2u);
        const uint32_t gn = g0 + (r8 & 3u);
        norms = *reinterpret_cast<const u32x4_any_t*>(nbase + (l8 * 16u + (gn < gl ? gn : gl) * 128u));
    }
    fetch_w(g0, w0);
    fetch_x(g0, x0);
    fetch_x(g0 + 1u, x1);
    if constexpr (ALL_X) {
        fetch_x(g0 + 2u, x2);
        fetch_x(g0 + 3u, x3);
    }
    if constexpr (!ONE) fetch_w(g0 + SG, w1);
    fetch_epilogue();
    float rr[MT][2];   // 1 / rms of the rows this lane parks
#pragma unroll
    for (int i = 0; i < MT; ++i) rr[i][0] = rr[i][1] = 1.f;
    if (normed && a.ssq_in) {
        float* tot = reinterpret_cast<float*>(reinterpret_cast<char*>(lds_raw) + WAVES * rows_wave_lds(MT, NT));   // [MT * 16]
        // sixteen lanes a row, four rows a wave and step, every step's requests made before the first is used
        constexpr int STEPS = (MT * 16 + 4 * WAVES - 1) / (4 * WAVES);
        float v[STEPS];
#pragma unroll
        for (int i = 0; i < STEPS; ++i) v[i] = 0.f;
        for (uint32_t c = lane & 15u; c < a.ssq_n / 4u; c += 16u)
#pragma unroll
            for (int i = 0; i < STEPS; ++i) {
                const uint32_t m = ((uint32_t)i * WAVES + wave) * 4u + kq;
                const float4 p = reinterpret_cast<const float4*>(a.ssq_in + (size_t)(m0 + (m < M ? m : M - 1)) * a.ssq_n)[c];
                v[i] += (p.x + p.y) + (p.z + p.w);
            }
#pragma unroll
        for (int i = 0; i < STEPS; ++i) {
            const uint32_t m = ((uint32_t)i * WAVES + wave) * 4u + kq;
            const float t = group_sum(v[i], 16);
            if (c16 == 0 && m < MT * 16u) tot[m] = 1.0f / sqrtf(t / (float)K + a.eps);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint32_t m = (uint32_t)i * 16u + r8 + 8u * (uint32_t)h;
                rr[i][h] = tot[m];
            }
    } else if (normed) {
        // the squares of the wave's own columns, the first weights on their way meanwhile; the waves add them up in LDS
        float ss[MT][2];
#pragma unroll
        for (int i = 0; i < MT; ++i) ss[i][0] = ss[i][1] = 0.f;
        auto squares = [&](const Acts& x) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int e = 0; e < 4; ++e) ss[i][h] = dot2_bf16(x.x[i][h][e], x.x[i][h][e], ss[i][h]);
        };
        if constexpr (ALL_X) {
            squares(x0);
            if (g0 + 1u < g1) squares(x1);
            if (g0 + 2u < g1) squares(x2);
            if (g0 + 3u < g1) squares(x3);
        } else {
            for (uint32_t g = g0; g < g1; g += 2u) {
                squares(x0);
                fetch_x(g + 2u < g1 ? g + 2u : g0, x0);
                if (g + 1u < g1) squares(x1);
                fetch_x(g + 3u < g1 ? g + 3u : g0 + 1u, x1);
            }
        }
        float* part = reinterpret_cast<float*>(reinterpret_cast<char*>(lds_raw) + WAVES * rows_wave_lds(MT, NT));   // [WAVES][MT * 16]
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float v = group_sum(ss[i][h], 8);
                if (l8 == 0) part[wave * (MT * 16u) + (uint32_t)i * 16u + r8 + 8u * (uint32_t)h] = v;
            }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float v = 0.f;
#pragma unroll
                for (int w = 0; w < WAVES; ++w) v += part[(uint32_t)w * (MT * 16u) + (uint32_t)i * 16u + r8 + 8u * (uint32_t)h];
                rr[i][h] = 1.0f / sqrtf(v / (float)K + a.eps);
            }
    }
    auto step = [&](uint32_t g, uint32_t u, Acts& x) __attribute__((always_inline)) {
        if constexpr (ONE) {
            if (normed) x.nw = nl[u * 8u + l8];
        }
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                u32x4_t v = x.x[i][h];
                if (normed) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t xv = v[e], wv = x.nw[e], t = pack_bf16(bf16_lo(xv) * rr[i][h], bf16_hi(xv) * rr[i][h]);
                        v[e] = pack_bf16(bf16_lo(wv) * bf16_lo(t), bf16_hi(wv) * bf16_hi(t));
                    }
                }
                xs[((uint32_t)i * 16u + r8 + 8u * (uint32_t)h) * kRowsLine + l8] = v;
            }
        if (!ONE || (!ALL_X && u + 2u < SG)) fetch_x(g + u + 2u, x);
        __builtin_amdgcn_wave_barrier();
        if (g + u < g1) consume(u);   // wave-uniform
        __builtin_amdgcn_wave_barrier();
    };
    auto slab = [&](uint32_t g, Slab& s, Acts& xa, Acts& xb) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
#pragma unroll
            for (int h = 0; h < 2; ++h) wl[((uint32_t)t * 16u + r8 + 8u * (uint32_t)h) * kRowsLine + l8] = s.w[t][h];
            if constexpr (KIND != W_BF16 && !ONE) ml[(uint32_t)t * 64u + lane] = s.sc[t] | (s.bi[t] << 16);
        }
        if constexpr (ONE) {
            if (NT > 1 || lane < 32u) *reinterpret_cast<u32x2_any_t*>(sl + (NT > 1 ? lane : lane & 31u) * 4u) = meta;
            if (normed && r8 < 4u) nl[lane] = norms;
        } else {
            fetch_w(g + 2u * SG, s);
        }
        step(g, 0u, xa);
        if constexpr (SG > 1) step(g, 1u, xb);
        if constexpr (ALL_X) {
            step(g, 2u, x2);
            step(g, 3u, x3);
        } else if constexpr (SG > 2) {
            step(g, 2u, xa);
            step(g, 3u, xb);
        }
    };
    if constexpr (ONE) {
        slab(g0, w0, x0, x1);
    } else {
        for (uint32_t g = g0; g < g1; g += 2u * SG) {
            slab(g, w0, x0, x1);
            if (g + SG < g1) {
                if constexpr (SG & 1u)
                    slab(g + SG, w1, x1, x0);
                else
                    slab(g + SG, w1, x0, x1);
            }
        }
    }
    __syncthreads();   // every wave is through with its staging area

    // The waves meet: [wave][activation row][weight row of the block]; register r of a lane is activation row 4 kq + r.
    float* meet = reinterpret_cast<float*>(lds_raw);
    constexpr uint32_t COLS = 16u * NT, PER_WAVE = 16u * MT * COLS;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                meet[wave * PER_WAVE + ((uint32_t)i * 16u + kq * 4u + (uint32_t)r) * COLS + (uint32_t)t * 16u + c16] = acc[i][t][r];
    __syncthreads();
    uint16_t* yo = a.y[seg] + (size_t)m0 * yst;
    // One round of outputs; EARLY ones have their operands already.
    auto outputs = [&](uint32_t e0, auto early, uint32_t bias_bits, uint32_t res_bits) __attribute__((always_inline)) {
        const uint32_t e = e0 + threadIdx.x, m = e / OUT, col = e % OUT, n = blk * OUT + col;
        const bool live = m < M && n < N;
        uint32_t o = 0;
        if (live) {
            const float* at = meet + m * COLS + col;
            float s0 = 0.f, s1 = 0.f;
#pragma unroll
            for (int w = 0; w < WAVES; ++w) {
                s0 += at[(uint32_t)w * PER_WAVE];
                if constexpr (PAIR) s1 += at[(uint32_t)w * PER_WAVE + OUT];
            }
            if constexpr (PAIR) {
                o = swiglu_bits(s0, s1, a.variant, 1.0f);
            } else {
                if (bias) s0 += bf16_bits_to_f32(decltype(early)::value ? bias_bits : (uint32_t)bias[n]);
                if (res) s0 += bf16_bits_to_f32(decltype(early)::value ? res_bits : (uint32_t)res[(size_t)m * yst + n]);
                o = f32_to_bf16_bits(s0);
            }
            yo[(size_t)m * yst + n] = (uint16_t)o;
        }
        if constexpr (!PAIR) {
            if (a.ssq_out) {   // block-uniform; the 16 lanes of a tile's row are neighbours (columns past N: zero)
                const float v = bf16_bits_to_f32(o), t = group_sum(v * v, 16);
                if (m < M && (col & 15u) == 0) a.ssq_out[(size_t)(m0 + m) * a.ssq_n + blk * CT + (col >> 4)] = t;
            }
        }
    };
    constexpr uint32_t ROUND = WAVES * kWave;
    if constexpr (PAIR) {
        for (uint32_t e0 = 0; e0 < M * OUT; e0 += ROUND) outputs(e0, std::false_type{}, 0u, 0u);
    } else {
#pragma unroll
        for (int k = 0; k < EARLY; ++k)
            if ((uint32_t)k * ROUND < M * OUT) outputs((uint32_t)k * ROUND, std::true_type{}, e_bias[k], e_res[k]);
        for (uint32_t e0 = EARLY * ROUND; e0 < M * OUT; e0 += ROUND) outputs(e0, std::false_type{}, 0u, 0u);
    }
}

template <WKind KIND, bool PAIR, int NT, bool ONE>
const void* rows_func(uint32_t mt, uint32_t waves) {
#define FK_ROWS_CASE(MT)                                                                               \
    return waves == 8 ? reinterpret_cast<const void*>(&qgemm_rows_kernel<KIND, PAIR, NT, MT, 8, ONE>)   \
                      : reinterpret_cast<const void*>(&qgemm_rows_kernel<KIND, PAIR, NT, MT, 4, ONE>)
    switch (mt) {
        case 1: FK_ROWS_CASE(1);
        case 2: FK_ROWS_CASE(2);
        case 3: FK_ROWS_CASE(3);
        default: FK_ROWS_CASE(4);
    }
#undef FK_ROWS_CASE
}
template <WKind KIND, bool ONE>
const void* rows_func(bool pair, bool two, uint32_t mt, uint32_t waves) {
    if (pair) return rows_func<KIND, true, 2, ONE>(mt, waves);
    return two ? rows_func<KIND, false, 2, ONE>(mt, waves) : rows_func<KIND, false, 1, ONE>(mt, waves);
}

}  // namespace

bool qgemm_takes_rows(uint32_t M, uint32_t bits, uint32_t group, uint32_t K) {
    return M >= 1 && M <= kRowsMax && K >= 64u && K % 64u == 0 && K < (1u << 24) &&   // (32-bit offsets)
           (bits == 16 || ((bits == 4 || bits == 8) && (group == 64 || (group == 128 && K % 128u == 0))));
}

fk_status plan_qgemm_rows(const RowsRequest& rq, Launch* out) {
    const DeviceFacts* dev;
    FK_TRY(device_facts(&dev));
    if (rq.n_mats < 1 || rq.n_mats > 3 || (rq.pair && rq.n_mats != 2)) return set_error(FK_ERR_INVALID, "qgemm (rows): one to three matrices");
    const fk_weight* W0 = rq.W[0];
    if (!W0 || !rq.x) return set_error(FK_ERR_INVALID, "qgemm (rows): null weight or activations");
    const uint32_t M = rq.M, K = W0->k, x_stride = rq.x_stride ? rq.x_stride : K;
    if (!qgemm_takes_rows(M, W0->bits, W0->group, K)) return set_error(FK_ERR_UNSUPPORTED, "qgemm (rows): 1..64 rows, whole groups of 64 columns");
    if (x_stride >= (1u << 24)) return set_error(FK_ERR_UNSUPPORTED, "qgemm (rows): rows too far apart");
    if (x_stride < K) return set_error(FK_ERR_INVALID, "qgemm (rows): row stride below K");
    // (normalised or strided rows: the entry points for those have always asked for it)
    if ((rq.norm_w || rq.x_stride) && (x_stride % 8u || (((uintptr_t)rq.x | (uintptr_t)rq.norm_w) & 15u)))
        return set_error(FK_ERR_INVALID, "qgemm (rows): rows and norm weights must be 16-byte aligned");
    QgemmRowsArgs a;
    memset(&a, 0, sizeof(a));
    uint32_t b16 = 0;
    for (uint32_t i = 0; i < rq.n_mats; ++i) {
        const fk_weight* W = rq.W[i];
        if (!W || !W->w || W->n == 0 || (W->bits != 16 && (!W->scales || !W->biases))) return set_error(FK_ERR_INVALID, "qgemm (rows): null weight");
        if (W->k != K || W->bits != W0->bits || (W->bits != 16 && W->group != W0->group) || (rq.pair && W->n != W0->n))
            return set_error(FK_ERR_INVALID, "qgemm (rows): the matrices must share K, bits and group size (a pair: N too)");
        a.w[i] = reinterpret_cast<const uint4*>(W->w);
        a.sc[i] = W->scales;
        a.bi[i] = W->biases;
        a.n[i] = W->n;
        if (rq.pair && i) continue;
        if (!rq.y[i]) return set_error(FK_ERR_INVALID, "qgemm (rows): null output");
        a.bias[i] = rq.bias[i];
        a.y[i] = rq.y[i];
        a.y_stride[i] = rq.y_stride[i] ? rq.y_stride[i] : W->n;
        if (a.y_stride[i] < W->n) return set_error(FK_ERR_INVALID, "qgemm (rows): output row stride below the matrix's rows");
        b16 += (W->n + 15u) / 16u;
    }
    if (rq.ssq_out && (rq.pair || rq.n_mats != 1)) return set_error(FK_ERR_INVALID, "qgemm (rows): sums of squares come from a single matrix");
    a.x = rq.x; a.res = rq.res; a.norm_w = rq.norm_w; a.eps = rq.eps;
    a.ssq_in = rq.ssq_in; a.ssq_out = rq.ssq_out;
    a.ssq_n = rq.ssq_out ? rows_ssq_parts(W0->n) : rows_ssq_parts(K);
    a.M = M; a.K = K; a.x_stride = x_stride; a.variant = rq.variant;
    a.n_seg = rq.pair ? 1u : rq.n_mats;
    a.gshift = W0->bits != 16 && W0->group == 128 ? 1u : 0u;
    const uint32_t cus = (uint32_t)dev->cus, tiles = (M + 15u) / 16u;
    // Eight waves per block where the blocks do not fill the chip and K is deep enough for them; else four, of which two
    // blocks share a CU and cover each other's start (37 rows of int4, eight / four waves: 896 x 4864 12.1 / 13.3 us,
    // 2560 x 4096 11.1 / 12.1, 896 x 896 5.7 / 5.2, 4864 x 896 pair 14.0 / 9.7, 6144 x 2560 17.6 / 14.0).
    const uint32_t waves = b16 <= cus && K >= 2048u ? 8u : 4u;
    // Two tiles of weight rows per block -- half the blocks, each of which reads all activation rows -- once three or four
    // tiles of those make that traffic count (9728 x 2560: 37 rows 20.3 / 18.2 us with one / two, 12 rows 11.1 / 11.7; 64
    // rows of 6144 x 2560 17.0 / 15.5, but of 9728 x 2560 25.1 / 27.8: registers).  A pair has two tiles as it is.
    auto two_of = [&](uint32_t mt) { return !rq.pair && b16 > cus && (mt == 3u || (mt == 4u && b16 <= 2u * cus)); };
    auto blocks_of = [&](bool two) {
        uint32_t n = 0;
        for (uint32_t i = 0; i < a.n_seg; ++i) n += (a.n[i] + (two ? 31u : 15u)) / (two ? 32u : 16u);
        return n;
    };
    // How many of the tiles of 16 activation rows a block takes (the other tiles' blocks read the weights again, from the L2): least work of
    // the fullest CU, its blocks times a block's products and what its start takes of one (bf16 weights, which are not unpacked, as long as
    // one; int4 something under half), and another half for each further reading of weights that the L2s do not hold.  All tiles in one
    // block / this, us, int4: 37 rows of 896 x 4864 11.4 / 7.0, of 2560 x 9728 19.6 / 17.3, of 2560 x 4096 10.3 / 9.5, of the 4864 x 896 pair
    // 8.6 / 6.9, 64 rows of it 10.1 / 7.7, of the 9728 x 2560 pair 29.4 / 25.8, of 6144 x 2560 16.6 / 13.8; int8, 64 rows of 6144 x 2560 19.1 /
    // 14.1, 32 13.1 / 12.3 (17, the same tiles, 11.7 / 12.2), 37 of the 4864 x 896 pair 9.9 / 9.4.  On the line's other side, one block / more:
    // 24 rows of the 9728 x 2560 pair 18.4 / 19.9, 37 of the 2816 x 2048 pair 8.7 / 9.3, 24 of 2560 x 4096 8.3 / 9.2; int8, 64 of 3072 x 2048
    // 9.1 / 9.3; bf16, 64 of 3072 x 2048 8.6 / 9.2, 17 of 6144 x 2560 9.7 / 10.7.
    const uint64_t weight_bytes = (uint64_t)b16 * 16u * (rq.pair ? 2u : 1u) * K / 8u * W0->bits;
    const float reread = weight_bytes > (16ull << 20) ? 0.5f : 0.f, start = W0->bits == 4 ? 0.45f : (W0->bits == 8 ? 0.52f : 1.0f);
    uint32_t mt = tiles, m_blocks = 1u;
    float least = 1e30f;
    for (uint32_t t = tiles; t >= 1u; --t) {
        const uint32_t mb = (tiles + t - 1u) / t;   // (every block has rows)
        const bool tw = two_of(t);
        const float per_cu = (float)((blocks_of(tw) * mb + cus - 1u) / cus);
        const float work = per_cu * ((float)(t * (tw ? 2u : 1u)) + start) + (float)(mb - 1u) * reread;
        if (work < least) {
            least = work;
            mt = t;
            m_blocks = mb;
        }
    }
    const bool two = two_of(mt);
    uint32_t blocks = 0;
    for (uint32_t i = 0; i < a.n_seg; ++i) {
        a.blk0[i] = blocks;
        blocks += (a.n[i] + (two ? 31u : 15u)) / (two ? 32u : 16u);
    }
    // one slab a wave, and rows of at least the four scales that its one request takes
    const uint32_t groups = K / 64u;
    const bool one = W0->bits != 16 && (groups + waves - 1u) / waves <= rows_slab_groups(W0->bits) && (groups >> a.gshift) >= 4u;
    if (W0->bits == 4)
        out->func = one ? rows_func<W_Q4, true>(rq.pair, two, mt, waves) : rows_func<W_Q4, false>(rq.pair, two, mt, waves);
    else if (W0->bits == 8)
        out->func = one ? rows_func<W_Q8, true>(rq.pair, two, mt, waves) : rows_func<W_Q8, false>(rq.pair, two, mt, waves);
    else
        out->func = rows_func<W_BF16, false>(rq.pair, two, mt, waves);
    out->grid = dim3(blocks, m_blocks, 1);
    out->block = dim3(waves * kWave, 1, 1);
    out->shmem = rows_lds_bytes(mt, rq.pair || two ? 2u : 1u, waves);
    out->set_args(a);
    return raise_dynamic_lds(out->func, out->shmem);
}

}  // namespace fk
