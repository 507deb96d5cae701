// Routed projections (mixture of experts) of several tokens: each expert's weights are read ONCE and multiplied by the
// activation rows of all the routes that name the expert -- one route at a time (routed.hip), an expert chosen by n rows is
// streamed n times.  The counterpart of the reference's routed kernels (src/codegen/kernels/routed_qmv_swiglu.rs:99-446,
// routed_qmv_reduce.rs:110-322) for more than a few rows.
//
// Bound by the bytes of the chosen experts from some 24 rows on, below that by how early they are asked for.  A launch is a
// fixed set of workgroups: each sorts the routes by expert in LDS (the list is a few KB, one trip to memory), which names the
// work that there is -- an expert with routes, a tile of its rows -- and takes every grid-th piece of it, so that experts that
// nobody chose cost nothing.  Inside a piece the scheme is that of qgemm_rows.hip: four waves split K, a wave's weight and
// activation lines pass through its own piece of LDS, v_mfma_f32_16x16x32_bf16 with the codes as exact integers, a group's
// product folded into the sums with its scale and bias, the waves meet in LDS.  Two slabs of weights are always in flight, those of the NEXT
// piece while this one is finished.
#include "fk_host.hpp"
#include "gemv_kernel.hpp"
#include "routed_rule.hpp"

#include "fk_probe.hpp"
FK_PROBE_DEFINE(routed, 1024, 8)
#define FK_RT_STAMP(i) FK_PROBE_STAMP(routed, 1024, 8, blockIdx.x, threadIdx.x == 0, i)

namespace fk {

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_any_t __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t u32x4_any_t __attribute__((ext_vector_type(4), aligned(2)));   // 16 bytes of an operand at any of its addresses

constexpr uint32_t kRtThreads = kRtWaves * kWave, kRtMaxRoutes = 1024, kRtMaxExperts = 256, kRtLine = 9;

struct QgemmRoutedArgs {
    const unsigned char* w[2];   // stacks of n_experts matrices: one, or gate and up
    const unsigned char* sc[2];
    const unsigned char* bi[2];
    uint16_t* y;                  // [n_routes, N]
    const uint16_t* x;            // [n_x_rows, K]
    const uint32_t* expert_idx;   // [n_routes]
    const uint32_t* row_idx;      // activation row of a route, or null: the route itself
    const uint16_t* route_weight; // bf16, or null (pair: multiplies the SwiGLU product before its rounding)
    uint32_t N, K, gshift;        // gshift: 64-code groups per scale: 0 (group 64), 1 (group 128)
    uint32_t n_routes, n_experts, n_x_rows;
    uint32_t tiles;               // pieces of one expert
    uint32_t cus;
};

// The sorted list: row << 16 | route by expert; routes of an expert (then their first place); the pieces' experts, first
// places and counts.
struct RtList {
    uint32_t route[kRtMaxRoutes];
    uint32_t count[kRtMaxExperts];
    uint32_t chunk_expert[kRtMaxExperts + kRtMaxRoutes / kRtRows], chunk_at[kRtMaxExperts + kRtMaxRoutes / kRtRows];
    uint32_t chunks, several;   // several: an expert has more than one chunk
};
constexpr uint32_t kRtMeta = 12u;   // (scale, bias) pairs of a row in LDS: eight, behind three at most that a clamped request begins early
constexpr uint32_t kRtWaveLds = 2u * 16u * kRtLine * 16u + 2u * 16u * kRtMeta * 4u;   // weight lines, (scale, bias) pairs
constexpr uint32_t kRtMeetLds = kRtWaves * 2u * 256u * 4u;
constexpr uint32_t kRtLds = kRtWaves * kRtWaveLds + kRtMeetLds + (uint32_t)((sizeof(RtList) + 15u) & ~15u);

// Eight codes of a row, in order, as the eight bf16 values of a B fragment (qgemm_rows.hip).
template <WKind KIND>
__device__ __forceinline__ bf16x8_t rt_unpack(uint32_t w0, uint32_t w1) {
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
    return __builtin_bit_cast(bf16x8_t, b);
}

// Sorts the routes by expert and cuts each expert's into chunks of kRtRows.  Places within an expert first follow the order of
// the LDS additions, which differs from workgroup to workgroup and which no result depends on (a row of the product is formed
// for itself) -- but which of an expert's routes make up a chunk has to be the same in all of them, so where an expert has
// more than one its routes are put in order.  Whole block.
__device__ __forceinline__ void rt_sort(const QgemmRoutedArgs& a, RtList& L) {
    constexpr uint32_t rows = kRtRows;
    const uint32_t tid = threadIdx.x;
    uint32_t e[kRtMaxRoutes / kRtThreads], r[kRtMaxRoutes / kRtThreads], at[kRtMaxRoutes / kRtThreads];
#pragma unroll
    for (uint32_t j = 0; j < kRtMaxRoutes / kRtThreads; ++j) {
        if (j * kRtThreads >= a.n_routes) break;   // uniform
        const uint32_t i = j * kRtThreads + tid, ic = i < a.n_routes ? i : 0u;
        e[j] = a.expert_idx[ic];
        r[j] = *(a.row_idx ? a.row_idx + ic : a.expert_idx + ic);
    }
    L.count[tid] = 0;   // kRtMaxExperts == kRtThreads
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kRtMaxRoutes / kRtThreads; ++j) {
        if (j * kRtThreads >= a.n_routes) break;
        const uint32_t i = j * kRtThreads + tid;
        e[j] = e[j] < a.n_experts ? e[j] : a.n_experts - 1u;   // routed_qmv_swiglu.rs:138
        if (i < a.n_routes) at[j] = atomicAdd(&L.count[e[j]], 1u);
    }
    __syncthreads();
    if (tid < (uint32_t)kWave) {   // first places and chunks, 64 experts a step
        uint32_t routes = 0, chunks = 0, several = 0;
        for (uint32_t base = 0; base < a.n_experts; base += kWave) {
            const uint32_t ex = base + tid, n = ex < a.n_experts ? L.count[ex] : 0u, c = (n + rows - 1u) / rows;
            several |= __any((int)(c > 1u)) ? 1u : 0u;
            uint32_t sum_n = n, sum_c = c;   // inclusive sums over the lanes
#pragma unroll
            for (uint32_t d = 1; d < (uint32_t)kWave; d <<= 1) {
                const uint32_t vn = __shfl_up(sum_n, d, kWave), vc = __shfl_up(sum_c, d, kWave);
                if (tid >= d) sum_n += vn, sum_c += vc;
            }
            const uint32_t first = routes + sum_n - n;
            for (uint32_t k = 0; k < c; ++k) {
                const uint32_t left = n - k * rows;
                L.chunk_expert[chunks + sum_c - c + k] = ex;
                L.chunk_at[chunks + sum_c - c + k] = ((first + k * rows) << 16) | (left < rows ? left : rows);
            }
            L.count[ex] = first;   // (ex < kRtMaxExperts: 64 experts a step)
            routes += (uint32_t)__builtin_amdgcn_readlane((int)sum_n, kWave - 1);
            chunks += (uint32_t)__builtin_amdgcn_readlane((int)sum_c, kWave - 1);
        }
        if (tid == 0) {
            L.chunks = chunks;
            L.several = several;
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kRtMaxRoutes / kRtThreads; ++j) {
        if (j * kRtThreads >= a.n_routes) break;
        const uint32_t i = j * kRtThreads + tid;
        if (i >= a.n_routes) break;
        const uint32_t row = a.row_idx ? r[j] : i;
        r[j] = ((row < a.n_x_rows ? row : a.n_x_rows - 1u) << 16) | i;
        L.route[L.count[e[j]] + at[j]] = r[j];
    }
    __syncthreads();
    if (!L.several) return;
#pragma unroll
    for (uint32_t j = 0; j < kRtMaxRoutes / kRtThreads; ++j) {
        if (j * kRtThreads >= a.n_routes) break;
        const uint32_t i = j * kRtThreads + tid;
        if (i >= a.n_routes) break;
        const uint32_t first = L.count[e[j]], end = e[j] + 1u < a.n_experts ? L.count[e[j] + 1u] : a.n_routes;
        at[j] = first;
        for (uint32_t k = first; k < end; ++k) at[j] += (L.route[k] & 0xffffu) < i ? 1u : 0u;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kRtMaxRoutes / kRtThreads; ++j) {
        if (j * kRtThreads >= a.n_routes) break;
        if (j * kRtThreads + tid < a.n_routes) L.route[at[j]] = r[j];
    }
    __syncthreads();
}

// Two tiles of 16 weight rows (PAIR: one of the gate matrix and the same one of the up matrix) against up to 16 activation rows.
// (Two tiles of those for the experts with more routes were slower at every count: 576 / 768 / 960 routes of 64 experts, a layer
// of the model 318 / 351 / 414 us against 303 / 348 / 410.)
template <WKind KIND, bool PAIR>
__global__ __launch_bounds__(kRtThreads, 2) void qgemm_routed_kernel(const QgemmRoutedArgs a) {
    constexpr int NT = 2, CT = PAIR ? 1 : 2;
    constexpr uint32_t BITS = KIND == W_Q4 ? 4u : 8u, SG = rt_slab_groups(BITS), PPG = 8u / SG;   // 16-byte pieces per group
    extern __shared__ uint4 lds_raw[];
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t c16 = lane & 15u, kq = lane >> 4, l8 = lane & 7u, r8 = lane >> 3;
    char* lds = reinterpret_cast<char*>(lds_raw);
    u32x4_t* wl = reinterpret_cast<u32x4_t*>(lds + wave * kRtWaveLds);                      // [NT * 16][kRtLine]
    uint32_t* ml = reinterpret_cast<uint32_t*>(wl + NT * 16 * kRtLine);                        // [NT * 16][kRtMeta]
    float* meet = reinterpret_cast<float*>(lds + kRtWaves * kRtWaveLds);                  // [waves][16][NT * 16]
    RtList& L = *reinterpret_cast<RtList*>(lds + kRtWaves * kRtWaveLds + kRtMeetLds);
    FK_RT_STAMP(0);
    kernarg_warm<(int)sizeof(QgemmRoutedArgs)>();
    rt_sort(a, L);
    FK_RT_STAMP(1);
    const uint32_t N = a.N, K = a.K, G = K >> 6, gpr = G >> a.gshift, row_bytes = K / 8u * BITS;
    const uint32_t pieces = L.chunks * a.tiles;
    if (blockIdx.x >= pieces) return;
    const uint32_t g0 = wave * G / kRtWaves, g1 = (wave + 1u) * G / kRtWaves;
    const uint32_t gl = g1 > g0 ? g1 - 1u : (g0 < G ? g0 : G - 1u);
    const uint32_t slabs = rt_slabs(K, BITS);

    // A piece: uniform bases, 32-bit lane offsets (rows past the matrix repeat its last one and are not stored).
    struct Piece {
        const unsigned char *w[NT], *s, *b;   // s, b: of this lane's tile
        uint32_t woff[NT][2], xoff, n0, first, count;
        int soff, slast;
    };
    auto open = [&](uint32_t p, Piece& q) __attribute__((always_inline)) {
        const uint32_t chunk = p / a.tiles, tile = p - chunk * a.tiles, at = L.chunk_at[chunk];
        const uint32_t ex = __builtin_amdgcn_readfirstlane(L.chunk_expert[chunk]);
        q.first = __builtin_amdgcn_readfirstlane(at >> 16);
        q.count = __builtin_amdgcn_readfirstlane(at & 0xffffu);
        q.n0 = tile * CT * 16u;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const uint32_t mat = PAIR ? (uint32_t)t : 0u, n0 = q.n0 + (PAIR ? 0u : (uint32_t)t * 16u), f = n0 < N ? n0 : N - 1u;
            const size_t row = (size_t)ex * N + f;
            q.w[t] = a.w[mat] + row * row_bytes;
            auto clamp = [&](uint32_t r) { return f + r < N ? r : N - 1u - f; };
#pragma unroll
            for (int h = 0; h < 2; ++h) q.woff[t][h] = clamp(r8 + 8u * (uint32_t)h) * row_bytes;
            if (t == 0 || lane >= 32u) {   // scales and biases: tile lane / 32, row lane / 2 % 16
                q.s = a.sc[mat] + row * gpr * 2u;
                q.b = a.bi[mat] + row * gpr * 2u;
                q.soff = (int)(clamp((lane >> 1) & 15u) * gpr);
                const int64_t last = (int64_t)((size_t)a.n_experts * N - row) * gpr - 4;   // where the stack's last four begin
                q.slast = last < 0x3fffffff ? (int)last : 0x3fffffff;
            }
        }
        q.xoff = ((L.route[q.first + (c16 < q.count ? c16 : q.count - 1u)] >> 16) * K + kq * 16u) * 2u;
    };
    struct Slab {
        u32x4_t w[NT][2];
    };
    // Scales and biases of two slabs with one request each: lane 2 r + h of a tile's 32 holds four of row r's from the 4 h-th on (or the
    // stack's last four), at + i the i-th one's place in the row's line.  Two bytes a lane and tile, four requests a slab, they were a
    // quarter of all requests and a CU issues one in 16 .. 20 cycles: 64 experts, pair of 1408 x 2048 int4, 48 routes 32.2 / 31.6 us, 96
    // 43.8 / 42.7, 192 52.3 / 50.4, 576 64.1 / 60.9.
    struct Meta {
        u32x2_any_t s, b;
        uint32_t at;
    };
    struct Acts {   // sixteen of the row's values, straight from memory: the rows are few and stay in the caches
        u32x4_t x[2];
    };
    const unsigned char* xbase = reinterpret_cast<const unsigned char*>(a.x);
    // Straight-line requests: what lies past the wave's range is clamped to its last piece and never used.
    auto fetch_w = [&](const Piece& q, uint32_t slab, Slab& s) __attribute__((always_inline)) {
        const uint32_t g = g0 + slab * SG, gp = g + l8 / PPG, gc = gp < gl ? gp : gl, at = (gc * PPG + l8 % PPG) * 16u;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
#pragma unroll
            for (int h = 0; h < 2; ++h) s.w[t][h] = *reinterpret_cast<const u32x4_any_t*>(q.w[t] + (q.woff[t][h] + at));
        }
    };
    auto first_meta = [&](uint32_t slab) { return (g0 + slab * SG < gl ? g0 + slab * SG : gl) >> a.gshift; };   // of the two slabs from `slab` on
    auto fetch_m = [&](const Piece& q, uint32_t slab, Meta& m) __attribute__((always_inline)) {
        const int from = q.soff + (int)first_meta(slab), want = from + 4 * (int)(lane & 1u), at = want < q.slast ? want : q.slast;
        m.s = *reinterpret_cast<const u32x2_any_t*>(q.s + at * 2);
        m.b = *reinterpret_cast<const u32x2_any_t*>(q.b + at * 2);
        m.at = (uint32_t)(4 + at - from);
    };
    auto fetch_x = [&](const Piece& q, uint32_t u, Acts& s) __attribute__((always_inline)) {   // the wave's u-th group
        const uint32_t g = g0 + u, gc = g < gl ? g : gl;
#pragma unroll
        for (int h = 0; h < 2; ++h) s.x[h] = *reinterpret_cast<const u32x4_any_t*>(xbase + (q.xoff + gc * 128u + 16u * (uint32_t)h));
    };
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    f32x4_t acc[NT];
    // A group's product is formed about the codes' middle: the matrix instructions start from -MID * Sx and the fold adds
    // s * (dot - MID * Sx) + (b + MID * s) * Sx.  Formed as s * dot + b * Sx the two terms cancel to a fraction of either, and
    // with activations whose mean is not zero what is lost there is more than the route-by-route form loses, whose terms have
    // half the length.  Outputs rounded to the wrong side, of a million, route by route / uncentred / this: 64 experts of
    // 1408 x 2048 int4, activations of mean 0 104 / 136 / 82, mean 1 281 / 514 / 148, mean 4 27 / 529 / 21; 16 of 1024 x 2048, 8
    // bits, 117 / 160 / 85, 206 / 795 / 146, 90 / 627 / 111.  Uncentred / this, us: pair of 1408 x 2048 int4, 48 routes 28.6 / 29.2, 96
    // 42.6 / 43.9, 576 60.9 / 61.3; 8 bits, 96 routes 65.7 / 66.2.
    // HALVES: each half of a group starts from its own Sx.  8-bit codes need it: from the whole group's, what the first half has
    // not yet made up for is 128 times the other half's sum (309 of a million at mean 1).
    constexpr float MID = KIND == W_Q4 ? 8.f : 128.f;
    constexpr uint32_t MID2 = KIND == W_Q4 ? 0xC100C100u : 0xC300C300u;   // -MID as two bf16 values
    constexpr bool HALVES = KIND == W_Q8;
    const bf16x8_t mids = __builtin_bit_cast(bf16x8_t, make_uint4(MID2, MID2, MID2, MID2));
    auto consume = [&](uint32_t u, uint32_t entry, const Acts& x) __attribute__((always_inline)) {   // group u of the parked slab, its pair
        const bf16x8_t xa0 = __builtin_bit_cast(bf16x8_t, x.x[0]), xa1 = __builtin_bit_cast(bf16x8_t, x.x[1]);
        // -MID * Sx, as the instructions take it (a power of two: exactly MID times what Sx would be)
        const f32x4_t m0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa0, mids, zero, 0, 0, 0);
        const f32x4_t m1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa1, mids, HALVES ? zero : m0, 0, 0, 0);
        f32x4_t mx = m1;
        if constexpr (HALVES) {
#pragma unroll
            for (int r = 0; r < 4; ++r) mx[r] += m0[r];
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const u32x4_t* line = wl + ((uint32_t)t * 16u + c16) * kRtLine;
            bf16x8_t b0, b1;
            if constexpr (KIND == W_Q4) {
                const uint2 v = reinterpret_cast<const uint2*>(line)[u * 4u + kq];
                b0 = rt_unpack<KIND>(v.x, 0u);
                b1 = rt_unpack<KIND>(v.y, 0u);
            } else {
                const u32x4_t v = line[u * 4u + kq];
                b0 = rt_unpack<KIND>(v.x, v.y);
                b1 = rt_unpack<KIND>(v.z, v.w);
            }
            const uint32_t sb = ml[((uint32_t)t * 16u + c16) * kRtMeta + entry];
            const float sf = bf16_lo(sb), bm = fmaf(bf16_hi(sb), -1.f / MID, -sf);   // (b + MID s) / -MID
            f32x4_t c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa0, b0, HALVES ? m0 : mx, 0, 0, 0);
            const f32x4_t c1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa1, b1, HALVES ? m1 : c, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[t][r] += fmaf(sf, HALVES ? c[r] + c1[r] : c1[r], bm * mx[r]);
        }
    };

    Piece now, next;
    Slab w0, w1;
    Acts x0, x1;
    Meta meta;
    uint32_t p = blockIdx.x;
    open(p, now);
    fetch_m(now, 0u, meta);
    fetch_w(now, 0u, w0);
    fetch_x(now, 0u, x0);
    fetch_x(now, 1u, x1);
    fetch_w(now, 1u, w1);
    // The waves of a CU's three workgroups (the grid deals one to each CU before the next) go first in turn, a piece each: left to their age
    // the third one's first piece was done 5 us after the first one's and its last so much later, the others' memory idle meanwhile (64
    // experts, pair of 1408 x 2048 int4, runs differ by 0.1: 48 routes 30.1 / 29.9 us, 96 40.0 / 39.6, 192 48.4 / 47.8, 576 58.1 / 57.3).
    uint32_t turn = blockIdx.x < a.cus ? 0u : (blockIdx.x < 2u * a.cus ? 1u : 2u);
    while (true) {
        switch (turn++ % 3u) {   // uniform
            case 0: __builtin_amdgcn_s_setprio(0); break;
            case 1: __builtin_amdgcn_s_setprio(1); break;
            default: __builtin_amdgcn_s_setprio(2);
        }
        const uint32_t pn = p + gridDim.x;
        const bool more = pn < pieces;   // uniform
        open(more ? pn : p, next);       // (the last piece asks for its own first slabs again)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = zero;
        // Slab s of this piece into the product; the slab two further on, or of the next piece, asked for meanwhile (LAST: this
        // is one of the piece's last two), and likewise the activations two groups ahead.
        auto slab = [&](uint32_t s, Slab& w, auto last, auto second) __attribute__((always_inline)) {
            constexpr bool LAST = decltype(last)::value, SECOND = decltype(second)::value;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
#pragma unroll
                for (int h = 0; h < 2; ++h) wl[((uint32_t)t * 16u + r8 + 8u * (uint32_t)h) * kRtLine + l8] = w.w[t][h];
            }
            if constexpr (!SECOND) {
                uint32_t* line = ml + (lane >> 1) * kRtMeta + meta.at;
                line[0] = __builtin_amdgcn_perm(meta.b[0], meta.s[0], 0x05040100u);
                line[1] = __builtin_amdgcn_perm(meta.b[0], meta.s[0], 0x07060302u);
                line[2] = __builtin_amdgcn_perm(meta.b[1], meta.s[1], 0x05040100u);
                line[3] = __builtin_amdgcn_perm(meta.b[1], meta.s[1], 0x07060302u);
                if constexpr (LAST)
                    fetch_m(next, 0u, meta);
                else
                    fetch_m(now, s + 2u, meta);
            }
            if constexpr (LAST)
                fetch_w(next, SECOND ? 1u : 0u, w);
            else
                fetch_w(now, s + 2u, w);
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (uint32_t j = 0; j < SG; ++j) {
                const uint32_t u = s * SG + j;
                Acts& x = j & 1u ? x1 : x0;
                if (g0 + u < g1) consume(j, 4u + ((g0 + u) >> a.gshift) - first_meta(SECOND ? s - 1u : s), x);   // wave-uniform
                if (LAST && SECOND && j + 2u >= SG)
                    fetch_x(next, j + 2u - SG, x);
                else
                    fetch_x(now, u + 2u, x);
            }
            __builtin_amdgcn_wave_barrier();
        };
        using std::false_type;
        using std::true_type;
        for (uint32_t s = 0; s + 2u < slabs; s += 2u) {
            slab(s, w0, false_type{}, false_type{});
            slab(s + 1u, w1, false_type{}, true_type{});
        }
        slab(slabs - 2u, w0, true_type{}, false_type{});
        slab(slabs - 1u, w1, true_type{}, true_type{});
        FK_RT_STAMP(2);
        // The waves meet: [wave][activation row][weight row]; register r of a lane is activation row 4 kq + r.
        constexpr uint32_t COLS = 16u * NT, PER_WAVE = kRtRows * COLS, OUT = 16u * CT;
        __syncthreads();   // the sums of the piece before have been read
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) meet[wave * PER_WAVE + (kq * 4u + (uint32_t)r) * COLS + (uint32_t)t * 16u + c16] = acc[t][r];
        __syncthreads();
        for (uint32_t e = threadIdx.x; e < now.count * OUT; e += kRtThreads) {
            const uint32_t m = e / OUT, col = e % OUT, n = now.n0 + col;
            if (n >= N) continue;
            const float* at = meet + m * COLS + col;
            float s0 = 0.f, s1 = 0.f;
#pragma unroll
            for (uint32_t w = 0; w < kRtWaves; ++w) {
                s0 += at[w * PER_WAVE];
                if constexpr (PAIR) s1 += at[w * PER_WAVE + OUT];
            }
            const uint32_t route = L.route[now.first + m] & 0xffffu;
            uint32_t o;
            if constexpr (PAIR)
                o = swiglu_bits(s0, s1, 1, a.route_weight ? bf16_bits_to_f32(a.route_weight[route]) : 1.0f);
            else
                o = f32_to_bf16_bits(s0);
            a.y[(size_t)route * N + n] = (uint16_t)o;
        }
        FK_RT_STAMP(3);
        if (p == blockIdx.x) FK_RT_STAMP(4);
        if (!more) return;
        p = pn;
        now = next;
    }
}

template <WKind KIND>
const void* routed_func(bool pair) {
    return pair ? reinterpret_cast<const void*>(&qgemm_routed_kernel<KIND, true>) : reinterpret_cast<const void*>(&qgemm_routed_kernel<KIND, false>);
}

}  // namespace

bool qgemm_takes_routed(const fk_weight* W, bool pair, uint32_t n_experts, uint32_t n_x_rows, uint32_t n_routes) {
    if (n_x_rows < 2 || n_x_rows > 0xffffu || n_routes > kRtMaxRoutes || n_experts > kRtMaxExperts) return false;
    if ((W->bits != 4 && W->bits != 8) || (W->group != 64 && !(W->group == 128 && W->k % 128u == 0)) || W->k < 64u || W->k % 64u) return false;
    // 32-bit offsets: into the activations, into a tile's rows
    if ((uint64_t)n_x_rows * W->k * 2u > 0xffffffffull || (uint64_t)32u * W->k > 0xffffffffull || (uint64_t)n_experts * W->n > 0x7fffffffull) return false;
    if ((uint64_t)n_experts * W->n * (W->k / W->group) < 4u) return false;   // four scales are asked for at a time
    const DeviceFacts* dev;
    return device_facts(&dev) == FK_OK && routes_served_together(n_experts, n_routes, W->n, W->k, W->bits, pair, (uint32_t)dev->cus);
}

fk_status plan_qgemm_routed(const uint16_t* x, uint32_t n_x_rows, const fk_weight* Wa, const fk_weight* Wb, uint32_t n_experts,
                            const uint32_t* row_idx, const uint32_t* expert_idx, const uint16_t* route_weight, uint32_t n_routes,
                            uint16_t* y, Launch* out) {
    const DeviceFacts* dev;
    FK_TRY(device_facts(&dev));
    QgemmRoutedArgs a;
    memset(&a, 0, sizeof(a));
    const bool pair = Wb != nullptr;
    for (uint32_t i = 0; i < (pair ? 2u : 1u); ++i) {
        const fk_weight* W = i ? Wb : Wa;
        if (!W->w || W->n == 0 || !W->scales || !W->biases) return set_error(FK_ERR_INVALID, "routed: null weight, scales or biases");
        if (W->k != Wa->k || W->n != Wa->n || W->bits != Wa->bits || W->group != Wa->group)
            return set_error(FK_ERR_INVALID, "routed: gate and up must share their shape, bits and group size");
        a.w[i] = static_cast<const unsigned char*>(W->w);
        a.sc[i] = reinterpret_cast<const unsigned char*>(W->scales);
        a.bi[i] = reinterpret_cast<const unsigned char*>(W->biases);
    }
    if (!x || !y) return set_error(FK_ERR_INVALID, "routed: null activations or output");
    a.y = y;
    a.x = x;
    a.N = Wa->n;
    a.K = Wa->k;
    a.gshift = Wa->group == 128 ? 1u : 0u;
    a.expert_idx = expert_idx;
    a.row_idx = row_idx;
    a.route_weight = route_weight;
    a.n_routes = n_routes;
    a.n_experts = n_experts;
    a.n_x_rows = n_x_rows;
    a.tiles = rt_pieces_of_an_expert(a.N, pair);
    a.cus = (uint32_t)dev->cus;
    const uint64_t most = (uint64_t)(n_routes < n_experts ? n_routes : n_experts + n_routes / kRtRows) * a.tiles;
    const uint32_t resident = 3u * (uint32_t)dev->cus;   // by LDS four; two were 1 %, four 0 .. 1 % slower
    out->func = Wa->bits == 4 ? routed_func<W_Q4>(pair) : routed_func<W_Q8>(pair);
    out->grid = dim3((uint32_t)(most < resident ? most : resident), 1, 1);
    out->block = dim3(kRtThreads, 1, 1);
    out->shmem = kRtLds;
    out->set_args(a);
    return raise_dynamic_lds(out->func, out->shmem);
}

}  // namespace fk
