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
// are paid for hardly any expert that is named twice.  us, route by route / together, uniform routes over cold weights:
//   64 experts, pair 1408 x 2048 int4: 36 routes 29.9 / 28.5, 48 37.1 / 33.6, 96 60.5 / 42.3, 576 311 / 66; int8 48 routes 57 / 48
//   64 experts, 2048 x 1408 int4:      48 routes 26.9 / 27.8, 60 30.2 / 29.4, 72 34.4 / 33.0, 96 37.6 / 34.1; int8 48 routes 37.4 / 37.7
//   128 experts, 2048 x 768 int4:      128 routes 31.3 / 38.8, 192 40.5 / 44.3, 384 65.0 / 52.4;  int8, 96 routes 38.4 / 36.8
//   256 experts, 2048 x 512 int4:      192 routes 34.1 / 51.7, 384 51.6 / 69.2
//   32 experts, pair 1024 x 1024 int4: 24 routes 9.8 / 11.9, 48 15.9 / 14.6, 96 24.4 / 16.9
//   8 experts, 2048 x 3584 int4:       6 routes 12.4 / 13.4, 12 16.6 / 17.2, 16 18.6 / 17.5, 32 25.1 / 18.5
//   2 experts, pair 512 x 512 int4:    2 .. 8 routes 4.7 .. 4.8 / 5.2 .. 5.5
// Over 424 such points (2 .. 256 experts, K 256 .. 4096, both widths) the rule's choice is 0.6 % behind the better of the two on
// average, 9 % at the worst that it sends together and 19 % (17 us) at the worst that it leaves; three quarters of a route per expert
// alone: 4 % and 54 %.
inline bool routes_served_together(uint32_t n_experts, uint32_t n_routes, uint32_t N, uint32_t K, uint32_t bits, bool pair, uint32_t cus) {
    if (4u * (uint64_t)n_routes < 3u * (uint64_t)n_experts) return false;
    const double touched = n_experts * (1.0 - exp(-(double)n_routes / n_experts));
    const double pieces = touched * rt_pieces_of_an_expert(N, pair), least = 4.0 * cus;
    const double columns = (double)rt_slabs(K, bits) * rt_slab_groups(bits) * 64u * kRtWaves;
    return (double)n_routes * N * (pair ? 2.0 : 1.0) * K >= (pieces > least ? pieces : least) * kRtPieceRows * columns;
}

}  // namespace fk
