// One-tile GEMV: the flat stream of gemv_kernel.hpp for the projections of a decode step (0.2 .. 60 MB).  A block owns ONE tile of R
// rows and asks for its activations, scales, biases, epilogue operands and first chunks of weights before it waits for anything; the
// other chunks follow when the activations are staged.  A launch of more blocks than are resident starts blocks over
// (gemv_tile_choice says where that is worth it).
//
// What bounds these launches is not the bytes but the chain a block runs through: its arguments, the activations, the
// weights, the row sums, the epilogue's operands -- a memory trip each where they are not overlapped -- and the vector
// memory instructions in front of it, which a CU issues one per 16 .. 20 cycles whatever their width.  So
//   * a quantised tile's scales and biases are one contiguous run of each array: four groups a lane and request, parked in
//     LDS as (scale | bias << 16), instead of two 2-byte requests for every 16-byte chunk of weights;
//   * the activations are asked for as often as the row is long, the norm weight only where there is one;
//   * projection bias and residual are asked for in front of the weights' use, not behind the row sums;
//   * the tile height follows the launch: a few chunks a thread on as many CUs as there are (gemv_tile_choice in gemv_tiling.hpp).
// int4, launch to launch in a captured chain over cold weights, gemv_stream_kernel -> this, with a residual: 896 x 896 4.3 -> 2.95 us, 4864 x
// 896 4.8 -> 3.7, 2560 x 4096 5.8 -> 4.3, 2560 x 9728 7.9 -> 6.2; gate / up pairs: 4864 x 896 5.9 -> 4.7, 9728 x 2560 10.4 -> 8.9, 14336 x 4096
// 17.8 -> 15.3.
// Every partial, the order in which a row's partials are added and the epilogue are those of gemv_run, bit for bit.
#pragma once
#include "gemv_kernel.hpp"

namespace fk {

typedef uint32_t u32x2_any_t __attribute__((ext_vector_type(2), aligned(2)));  // four 16-bit entries at any of their addresses

// NL: 16-byte chunks of each matrix per thread.  AHEAD of them go out in front of the staging (a wave cannot stage before it
// has issued what stands in front of it; pair of 9728 x 2560, 12 a thread: 1 / 2 / 4 / 6 ahead 9.5 / 9.3 / 9.1 / 9.6 us; 6144 x 2560, 3 a
// thread: 1 / 2 / all 5.36 / 5.33 / 5.5; 896 -> 4864 pair, 4 a thread: 1 / 2 / all 4.84 / 4.66 / 4.76).
template <WKind KIND, int NSEG, int NL>
__global__ __launch_bounds__(kGemvBlock) void gemv_tile_kernel(const uint16_t* x, const uint16_t* norm_w, uint32_t K, const GemvArgs a) {
    extern __shared__ uint4 lds_raw[];
    constexpr int PIECES = ChunkTraits<KIND>::kPieces;
    constexpr int TOTAL = NSEG * NL, AHEAD = TOTAL < 2 ? TOTAL : (TOTAL < 12 ? 2 : 4);
    const uint32_t tid = threadIdx.x;

    // Activations first: they return first.  Uniform branches around the requests of the longer rows are harmless here, in
    // front of everything else that is in flight.
    uint4 xr[kStageRegs], wr[kStageRegs];
    {
        const uint32_t n8 = K >> 3;
        const uint4 *x8 = reinterpret_cast<const uint4*>(x), *w8 = reinterpret_cast<const uint4*>(norm_w);
#pragma unroll
        for (int i = 0; i < kStageRegs; ++i) {
            if (i && (uint32_t)i * kGemvBlock >= n8) break;
            const uint32_t t = tid + i * kGemvBlock;
            xr[i] = x8[t < n8 ? t : 0u];
        }
        if (norm_w) {
#pragma unroll
            for (int i = 0; i < kStageRegs; ++i) {
                if (i && (uint32_t)i * kGemvBlock >= n8) break;
                const uint32_t t = tid + i * kGemvBlock;
                wr[i] = w8[t < n8 ? t : 0u];
            }
        }
    }
    kernarg_warm<24 + (int)sizeof(GemvArgs)>();

    const uint32_t cpr = a.cpr, R = a.R, lr = a.lr;
    const GemvTile<NSEG> t = gemv_tile<KIND, NSEG, GemvArgs>(a, blockIdx.x);
    const uint32_t valid_chunks = t.valid * cpr;
    uint4* xs = lds_raw;
    float* sx = reinterpret_cast<float*>(xs + PIECES * cpr);
    float* part = sx + cpr;                                                  // [NSEG][NL * 256]
    uint32_t* meta = reinterpret_cast<uint32_t*>(part + NSEG * NL * kGemvBlock);  // [NSEG][gemv_tile_meta]
    const uint32_t gpr = KIND == W_BF16 ? 0u : cpr >> a.gshift, n_meta = KIND == W_BF16 ? 0u : gemv_tile_meta(R, gpr);
    float* scratch = reinterpret_cast<float*>(meta + NSEG * n_meta);

    // A lane's run of four groups; the last run of the tile is moved back so that it ends with the tile (the planner
    // promises four groups a row), and rewrites what its neighbour wrote.
    u32x2_any_t ms[NSEG], mb[NSEG];
    const uint32_t groups = t.valid * gpr;
    const uint32_t g0 = KIND == W_BF16 ? 0u : (4u * tid < groups - 4u ? 4u * tid : groups - 4u);
    if constexpr (KIND != W_BF16) {
#pragma unroll
        for (int sg = 0; sg < NSEG; ++sg) {
            ms[sg] = *reinterpret_cast<const u32x2_any_t*>(t.sc[sg] + 2u * g0);
            mb[sg] = *reinterpret_cast<const u32x2_any_t*>(t.bi[sg] + 2u * g0);
        }
    }
    uint4 wv[TOTAL];  // slot j: chunk j / NSEG of matrix j % NSEG
    auto request = [&](auto from, auto to) {
#pragma unroll
        for (int j = decltype(from)::value; j < decltype(to)::value; ++j) {
            const uint32_t pos = (uint32_t)(j / NSEG) * kGemvBlock + tid;
            wv[j] = *reinterpret_cast<const uint4*>(t.w[j % NSEG] + ((pos < valid_chunks ? pos : 0u) << 4));
        }
    };
    request(std::integral_constant<int, 0>{}, std::integral_constant<int, AHEAD>{});

    // What the epilogue of this thread's row adds (a null operand reads the activations instead and is not used).
    const uint32_t rr = tid / lr, lane = tid & (lr - 1), row = t.row0 + (rr < t.valid ? rr : t.valid - 1u);
    uint32_t e_bias = 0, e_res = 0;
    if constexpr (NSEG == 1) {
        const uint16_t *pb = a.bias[t.m], *pr = t.m == 0 ? a.res : nullptr;
        e_bias = *(pb ? pb + row : x);
        e_res = *(pr ? pr + row : x);
    }

    auto store_meta = [&]() {
        if constexpr (KIND != W_BF16) {
            if (4u * tid < groups) {
#pragma unroll
                for (int sg = 0; sg < NSEG; ++sg) {
                    uint32_t* d = meta + sg * n_meta + g0;
                    d[0] = __builtin_amdgcn_perm(mb[sg].x, ms[sg].x, 0x05040100u);
                    d[1] = __builtin_amdgcn_perm(mb[sg].x, ms[sg].x, 0x07060302u);
                    d[2] = __builtin_amdgcn_perm(mb[sg].y, ms[sg].y, 0x05040100u);
                    d[3] = __builtin_amdgcn_perm(mb[sg].y, ms[sg].y, 0x07060302u);
                }
            }
        }
    };
    stage_activations<KIND, GemvArgs>(a, xs, sx, scratch, xr, wr, store_meta);
    request(std::integral_constant<int, AHEAD>{}, std::integral_constant<int, TOTAL>{});

#pragma unroll
    for (int j = 0; j < TOTAL; ++j) {
        const uint32_t pos = (uint32_t)(j / NSEG) * kGemvBlock + tid;
        const uint32_t col = pos - (uint32_t)(((float)pos + 0.5f) * a.inv_cpr) * cpr;
        uint32_t m = 0;
        if constexpr (KIND != W_BF16) m = meta[(j % NSEG) * n_meta + (pos < valid_chunks ? pos >> a.gshift : 0u)];
        const float p = chunk_partial<KIND>(wv[j], m & 0xffffu, m >> 16, xs, sx, col, cpr);
        part[(j % NSEG) * NL * kGemvBlock + pos] = p;
        __builtin_amdgcn_sched_barrier(0);  // as in gemv_run: keeps every chunk's LDS reads from being hoisted to the top
    }
    __syncthreads();

    // Row sums: lr lanes a row, each adds its partials in order (eight read in one trip to the LDS), then a butterfly.
    if (rr < R) {
        float s0 = 0.f, s1 = 0.f;
        const float *p0 = part + rr * cpr, *p1 = p0 + (NSEG - 1) * NL * kGemvBlock;
        for (uint32_t i = lane; i < cpr; i += 8u * lr) {
            float v0[8], v1[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const uint32_t c = i + (uint32_t)k * lr, cc = c < cpr ? c : 0u;
                v0[k] = p0[cc];
                if constexpr (NSEG == 2) v1[k] = p1[cc];
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const bool in = i + (uint32_t)k * lr < cpr;
                s0 += in ? v0[k] : 0.f;
                if constexpr (NSEG == 2) s1 += in ? v1[k] : 0.f;
            }
        }
        s0 = group_sum(s0, lr);
        if constexpr (NSEG == 2) s1 = group_sum(s1, lr);
        if (lane == 0 && rr < t.valid) {
            const uint32_t n = t.row0 + rr, m = t.m;
            if constexpr (NSEG == 2) {
                a.y[0][n] = (uint16_t)swiglu_bits(s0, s1, a.swiglu_variant, a.y_scale);
            } else {
                float v = s0;
                if (a.bias[m]) v += bf16_bits_to_f32(e_bias);
                if (m == 0 && a.res) v += bf16_bits_to_f32(e_res);
                uint32_t o = f32_to_bf16_bits(v);
                if (m == 0 && a.res2) o = f32_to_bf16_bits(bf16_bits_to_f32(o) + bf16_bits_to_f32(a.res2[n]));
                a.y[m][n] = (uint16_t)o;
            }
        }
    }
}

}  // namespace fk
