// Which routed projections serve an expert's routes together (qgemm_routed.hip), and which route by route (routed.hip).  Host code in
// plain C++.
#pragma once
#include <math.h>
#include <stdint.h>

namespace fk {

constexpr uint32_t kRtWaves = 4, kRtRows = 16;   // waves that split K; routes of an expert served together: one tile
constexpr uint32_t kRtPieceRows = 32;            // weight rows of a piece: two tiles of 16 (a pair: one of either matrix)
constexpr uint32_t rt_slab_groups(uint32_t bits) { return bits == 4 ? 4u : 2u; }
// Slabs of a piece, the same for every wave and even: the next piece's first slab takes the first set of registers again.
constexpr uint32_t rt_slabs(uint32_t K, uint32_t bits) {
    const uint32_t per_wave = (K / 64u + kRtWaves - 1u) / kRtWaves, sg = rt_slab_groups(bits);
    return ((per_wave + sg - 1u) / sg + 1u) & ~1u;
}
constexpr uint32_t rt_pieces_of_an_expert(uint32_t N, bool pair) { return pair ? (N + 15u) / 16u : (N + 31u) / 32u; }

// Together when that asks for no more of the weights.  Route by route every route asks for its expert's K x N; together every
// expert that has routes (of uniform ones E (1 - e^(-routes / E)); skewed ones have fewer) asks for its pieces, K rounded up to the
// waves' slabs: K = 768 int4 counts as 2048, and 512, 1024.  Fewer pieces than four a CU take as long as four: each is a chain of its
// slabs and a meeting of its waves.  And from three quarters of a route per expert at the least: below that the list and its sort
// are paid for hardly any expert that is named twice.  us, route by route / together, uniform routes, a captured chain over cold
// weights (single matrices with the launch that adds the routes up):
//   64 experts, pair 1408 x 2048 int4: 36 routes 26.7 / 25.5, 48 33.9 / 31.6, 96 57.4 / 42.4, 576 291 / 61; int8 48 routes 52 / 42
//   64 experts, 2048 x 1408 int4:      48 routes 21.3 / 21.6, 60 25.1 / 24.5, 72 29.1 / 27.4, 96 33.4 / 29.2; int8 48 routes 32.5 / 34.7
//   128 experts, 2048 x 768 int4:      128 routes 25.7 / 29.8, 192 35.4 / 36.5, 384 61.4 / 48.4;  int8, 96 routes 32.8 / 33.9
//   256 experts, 2048 x 512 int4:      192 routes 28.3 / 42.9, 384 46.4 / 62.8
//   32 experts, pair 1024 x 1024 int4: 24 routes 9.3 / 10.6, 48 16.0 / 13.9, 96 24.2 / 16.0
//   8 experts, 2048 x 3584 int4:       6 routes 11.7 / 12.2, 12 15.3 / 15.1, 16 16.5 / 15.3, 32 23.0 / 16.2
//   2 experts, pair 512 x 512 int4:    2 .. 8 routes 5.5 .. 5.6 / 6.0 .. 6.3
// Over 424 such points (2 .. 256 experts, K 256 .. 4096, both widths) the rule's choice was 0.6 % behind the better of the two on
// average, 9 % at the worst that it sends together and 19 % (17 us) at the worst that it leaves; three quarters of a route per expert
// alone: 4 % and 54 %.  (Timed before the products were centred, qgemm_routed.hip, which costs the form
// 0 .. 3 % near the line, and before its scales came with fewer requests, which gives it 2 .. 6 %.)
inline bool routes_served_together(uint32_t n_experts, uint32_t n_routes, uint32_t N, uint32_t K, uint32_t bits, bool pair, uint32_t cus) {
    if (4u * (uint64_t)n_routes < 3u * (uint64_t)n_experts) return false;
    const double touched = n_experts * (1.0 - exp(-(double)n_routes / n_experts));
    const double pieces = touched * rt_pieces_of_an_expert(N, pair), least = 4.0 * cus;
    const double columns = (double)rt_slabs(K, bits) * rt_slab_groups(bits) * 64u * kRtWaves;
    return (double)n_routes * N * (pair ? 2.0 : 1.0) * K >= (pieces > least ? pieces : least) * kRtPieceRows * columns;
}

}  // namespace fk
