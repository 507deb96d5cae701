// How a GEMV launch of the flat stream is cut into tiles, and the table that keeps a thread's last cuts.  Host code in plain C++, with
// the constants that kernels and planner share.
#pragma once
#include <stdint.h>

namespace fk {

enum WKind : int { W_Q4 = 0, W_Q8 = 1, W_BF16 = 2 };

constexpr int kGemvBlock = 256;
constexpr int kGemvUnroll = 4;  // 16-byte loads in flight per lane and batch
constexpr int kMaxMats = 3;
constexpr uint32_t kTileGroups = 4u * kGemvBlock;  // quantisation groups of a tile and matrix in the one-tile form: four a thread

template <WKind KIND>
struct ChunkTraits;
template <>
struct ChunkTraits<W_Q4> {
    static constexpr int kValues = 32, kPieces = 4;
};
template <>
struct ChunkTraits<W_Q8> {
    static constexpr int kValues = 16, kPieces = 4;
};
template <>
struct ChunkTraits<W_BF16> {
    static constexpr int kValues = 8, kPieces = 1;
};

// LDS bytes the flat form needs: staged activations + per-chunk sums + partials + scratch.
template <WKind KIND>
constexpr uint32_t gemv_lds_bytes(uint32_t cpr, uint32_t seg_chunks, uint32_t nseg) {
    const uint32_t pos = kGemvBlock * (kGemvUnroll / nseg);
    const uint32_t seg_pad = (seg_chunks + pos - 1) / pos * pos;
    return ChunkTraits<KIND>::kPieces * cpr * 16u + cpr * 4u + nseg * seg_pad * 4u + 64u;
}

// Entries of a matrix's scale / bias words in LDS (one-tile form), and the LDS bytes of that form.
constexpr uint32_t gemv_tile_meta(uint32_t rows, uint32_t gpr) { return (rows * gpr + 3u) & ~3u; }
template <WKind KIND>
constexpr uint32_t gemv_tile_lds_bytes(uint32_t cpr, uint32_t rows, uint32_t gpr, uint32_t nl, uint32_t nseg) {
    return ChunkTraits<KIND>::kPieces * cpr * 16u + cpr * 4u + nseg * nl * kGemvBlock * 4u +
           (KIND == W_BF16 ? 0u : nseg * gemv_tile_meta(rows, gpr) * 4u) + 64u;
}

// A launch as its tiles see it.  The search below has nothing else to go by (but the device), so two launches that are alike here
// may share what it found, and no others may.
struct GemvShape {
    WKind kind = W_BF16;
    uint32_t nseg = 1;  // 2: a gate / up pair
    uint32_t n_mats = 1, n[kMaxMats] = {0, 0, 0}, K = 0;
    uint32_t group = 0;  // codes per scale; bf16: 0
    uint32_t rows_per_tile = 0, grid_blocks = 0, grid_override = 0;

    bool operator==(const GemvShape& o) const {
        return kind == o.kind && nseg == o.nseg && n_mats == o.n_mats && n[0] == o.n[0] && n[1] == o.n[1] && n[2] == o.n[2] && K == o.K &&
               group == o.group && rows_per_tile == o.rows_per_tile && grid_blocks == o.grid_blocks && grid_override == o.grid_override;
    }
    uint32_t cpr() const { return K / (kind == W_Q4 ? 32u : (kind == W_Q8 ? 16u : 8u)); }  // 16-byte chunks a row
    uint32_t gpr() const { return kind == W_BF16 ? 0u : K / group; }                       // quantisation groups a row
    uint64_t tiles(uint32_t r) const {
        if (nseg == 2) return (n[0] + r - 1) / r;
        uint64_t t = 0;
        for (uint32_t m = 0; m < n_mats; ++m) t += (n[m] + r - 1) / r;
        return t;
    }
    uint32_t flat_lds(uint32_t r) const {
        switch (kind) {
            case W_Q4: return gemv_lds_bytes<W_Q4>(cpr(), r * cpr(), nseg);
            case W_Q8: return gemv_lds_bytes<W_Q8>(cpr(), r * cpr(), nseg);
            default: return gemv_lds_bytes<W_BF16>(cpr(), r * cpr(), nseg);
        }
    }
    uint32_t tile_lds(uint32_t r, uint32_t nl) const {
        switch (kind) {
            case W_Q4: return gemv_tile_lds_bytes<W_Q4>(cpr(), r, gpr(), nl, nseg);
            case W_Q8: return gemv_tile_lds_bytes<W_Q8>(cpr(), r, gpr(), nl, nseg);
            default: return gemv_tile_lds_bytes<W_BF16>(cpr(), r, gpr(), nl, nseg);
        }
    }
};

// rows: of a tile (and matrix of a pair); lr: lanes of a row's sum; chunks: 16-byte chunks a thread (one-tile form), 0: the flat form.
struct GemvTiling {
    uint32_t rows = 0, blocks = 0, lr = 0, chunks = 0;
};

// A thread's last tilings: 32 sets of four, the oldest of a set makes room (no lock, no growth).  With one place per hash two
// shapes of a model that fall on the same one are searched for on every call, some 1.5 us each.
class GemvTilings {
public:
    const GemvTiling* find(const GemvShape& s) {
        for (Kept& k : sets_[set_of(s)].way)
            if (k.shape == s) return &k.tiling;  // (an empty place has K = 0, as no launch has)
        return nullptr;
    }
    const GemvTiling* keep(const GemvShape& s, const GemvTiling& t) {
        Set& set = sets_[set_of(s)];
        Kept& k = set.way[set.next];
        set.next = (set.next + 1u) & 3u;
        k.shape = s;
        k.tiling = t;
        return &k.tiling;
    }

private:
    struct Kept {
        GemvShape shape;
        GemvTiling tiling;
    };
    struct Set {
        Kept way[4];
        uint32_t next = 0;
    };
    static uint32_t set_of(const GemvShape& s) {
        uint64_t h = (uint64_t)s.kind * 2u + s.nseg;
        for (uint32_t v : {s.n[0], s.n[1], s.n[2], s.K, s.group}) h = (h ^ v) * 0x9E3779B97F4A7C15ull;
        return (uint32_t)(h >> 59);
    }
    Set sets_[32];
};

// The one-tile form (gemv_tile.hpp) of a launch: chunks of each matrix per thread and rows per tile; chunks = 0: the flat form.
//
// The time goes by what the busiest CU runs: its blocks times (one block's fixed part, in units of a chunk's arithmetic: some
// three and one more for every 2048 activations it stages, + its chunks), and by the chunks that a thread works through one
// after the other once they have arrived.  Measured in a chain over cold weights, us, int4, chunks x rows (flat form before):
//   2560 -> 9728 pair  6 x 19 9.2, 4 x 12 10.5, 3 x 9 10.5 (10.9)     9728 -> 2560  6 x 5 6.15, 4 x 3 7.1, 8 x 6 6.6 (8.0)
//   4096 -> 2560       3 x 6 4.15, 2 x 4 4.2, 4 x 8 4.4 (5.5)         896 -> 896    1 x 9 2.74, 2 x 18 2.86, 4 x 36 3.24 (3.8)
//   896 -> 4864 pair   3 x 24 4.65, 1 x 9 4.70 (5.9)                  4864 -> 896   3 x 5 3.7, 1 x 1 4.2 (4.5)
// Blocks past what is resident start over (stage the activations again).  That is harmless while a block's rows are many
// next to its staging (14336 rows x 4096 pair, 8 bits, 4 rows of each, 14 blocks a CU: 26.3 us, flat form 28.9) and costs more than
// it gains where a long row leaves few (quantised, us, this form / flat: 9728 -> 2560 8 bits, 3 rows 10.2 / 9.9; 10944 -> 2944 8
// bits, 2 rows 15.9 / 13.3; 20352 -> 4096 int4, 3 rows 21.5 / 16.7; 4 rows, 14336 -> 4096 int4: 13.4 / 13.5.  bf16, whose staging is a
// copy: one row 14336 -> 4096 29.6 / 26.0, 12736 -> 2432 18.9 / 17.5, with 5 blocks a CU 6528 -> 1181 5.9 / 6.9; two rows 8128 -> 2048
// 9.1 / 9.4).  So a tile of few rows takes this form only while hardly any block starts over.
struct TileChoice {
    uint32_t chunks, rows;
};
inline TileChoice gemv_tile_choice(const GemvShape& s, uint32_t lr, uint32_t cus) {
    const uint32_t K = s.K, cpr = s.cpr(), gpr = s.gpr(), nseg = s.nseg;
    TileChoice best{0, 0};
    uint64_t best_cost = ~0ull, best_per_cu = 0;
    // a tile's scales are fetched in whole runs of four, and as whole groups a row (K = 576 with groups of 128 has 4.5)
    if (s.kind != W_BF16 && (gpr < 4 || K % s.group != 0)) return best;
    for (uint32_t nl : {1u, 2u, 3u, 4u, 6u, 8u}) {
        uint32_t r = nl * kGemvBlock / cpr;
        if (r > kGemvBlock / lr) r = kGemvBlock / lr;
        if (gpr && r > kTileGroups / gpr) r = kTileGroups / gpr;
        if (r == 0) continue;
        const uint64_t per_cu = (s.tiles(r) + cus - 1) / cus;
        const uint64_t cost = per_cu * (2 + (K + 2047) / 2048 + nl * nseg) + 2 * nl * nseg;
        if (cost < best_cost) {
            best_cost = cost;
            best_per_cu = per_cu;
            best = TileChoice{nl, r};
        }
    }
    const uint32_t few = s.kind == W_BF16 ? 2u : 5u, starts = s.kind == W_BF16 ? 5u : 3u;
    if (best.rows * nseg < few && best_per_cu > starts) best.chunks = 0;
    return best;
}

// Blocks that can be resident at once (registers and LDS decide): the flat form's grid never
// exceeds it, so no block waits for a slot and then pays the whole start-up chain
// (stage x, first loads) a second time; surplus tiles go to the persistent loop,
// whose next batch is already in flight while the current one is consumed.
//
// Rows per tile.  A batch (4 x 16-byte loads per lane) costs the same whether its
// lanes are full or not, and the blocks resident on a CU share its issue slots, so
// the first figure of merit is the number of batches the busiest CU runs,
// ceil(blocks / CUs) x tiles per block x batches per tile; ties go to the least
// total work, batches over all tiles plus one unit per block for its start-up
// (argument fetch, activation staging).  Measured on the 4B-class gate/up pair
// (2 x 9728 x 2560): 19 rows per tile = 512 blocks of three 97 %-full batches runs
// 10.4 us where one-batch tiles of 6 rows on 1280 blocks ran 12.2 us.
//
// per_cu_for(lds bytes): blocks of the flat form's kernel one CU holds.  False: no tile fits the LDS.
template <typename PER_CU>
bool gemv_tiling(const GemvShape& s, uint32_t cus, uint32_t max_lds, PER_CU&& per_cu_for, GemvTiling* out) {
    const uint32_t cpr = s.cpr(), pos = kGemvBlock * (kGemvUnroll / s.nseg);
    auto cap_for = [&](uint32_t lds_bytes) -> uint64_t {
        return s.grid_override ? s.grid_override : (s.grid_blocks ? s.grid_blocks : per_cu_for(lds_bytes) * cus);
    };
    uint32_t r_max = 8 * pos / cpr;  // up to eight batches per tile
    if (r_max < 1) r_max = 1;
    if (r_max > (uint32_t)kGemvBlock) r_max = kGemvBlock;
    uint32_t best_r = 1, best_blocks = 1;
    uint64_t best_cost = ~0ull, best_waste = ~0ull;
    for (uint32_t r = 1; r <= r_max; ++r) {
        const uint32_t lds_r = s.flat_lds(r);
        if (lds_r > max_lds) continue;
        const uint64_t tiles = s.tiles(r), cap = cap_for(lds_r);
        const uint64_t blocks = tiles < cap ? tiles : cap;
        const uint64_t per_block = (tiles + blocks - 1) / blocks;
        const uint64_t batches = ((uint64_t)r * cpr + pos - 1) / pos;
        // fewer than two blocks (eight waves) on a CU cannot hide the load latency:
        // such a choice is priced as if it ran two
        uint64_t per_cu = (blocks + cus - 1) / cus;
        if (per_cu < 512 / kGemvBlock) per_cu = 512 / kGemvBlock;
        const uint64_t cost = per_cu * per_block * batches;
        const uint64_t waste = tiles * batches + blocks;
        if (cost < best_cost || (cost == best_cost && waste < best_waste)) {
            best_cost = cost;
            best_waste = waste;
            best_r = r;
            best_blocks = (uint32_t)blocks;
        }
    }
    if (best_cost == ~0ull) return false;
    if (s.rows_per_tile) {
        best_r = s.rows_per_tile;
        const uint64_t tiles = s.tiles(best_r), cap = cap_for(s.flat_lds(best_r));
        best_blocks = (uint32_t)(tiles < cap ? tiles : cap);
    }
    if (s.flat_lds(best_r) > max_lds) return false;
    out->rows = best_r;
    out->blocks = best_blocks;
    // lanes of a row's sum: they fix the order of its additions, so the one-tile form takes the flat form's
    uint32_t lr = 64;
    while (lr > 1 && best_r > kGemvBlock / lr) lr >>= 1;
    while (lr > 1 && lr > cpr) lr >>= 1;
    out->lr = lr;
    out->chunks = 0;
    if (!s.rows_per_tile && !s.grid_blocks && !s.grid_override) {  // (those ask for the persistent form's tiles)
        const TileChoice c = gemv_tile_choice(s, lr, cus);
        if (c.chunks && s.tile_lds(c.rows, c.chunks) <= max_lds) {
            out->rows = c.rows;
            out->blocks = (uint32_t)s.tiles(c.rows);
            out->chunks = c.chunks;
        }
    }
    return true;
}

}  // namespace fk
