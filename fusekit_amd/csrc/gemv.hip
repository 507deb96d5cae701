// Launch planner and template instances of the flat-stream GEMV.
#include <stdlib.h>

#include <map>
#include <mutex>

#include "fk_host.hpp"

#include "fk_probe.hpp"
FK_PROBE_DEFINE(gemv, 2048, 8)
#define FK_GEMV_STAMP(i) FK_PROBE_STAMP(gemv, 2048, 8, blockIdx.x, threadIdx.x == 0, i)
#include "gemv_kernel.hpp"
#include "gemv_rows.hpp"
#include "gemv_tile.hpp"

namespace fk {

GemvPolicy g_gemv_policy = [] {
    GemvPolicy p;
    const char* e = getenv("FUSEKIT_GEMV_FLAT_ONLY");  // "1": never pick the row-group form (measurements, tests)
    p.flat_only = e && e[0] == '1';
    return p;
}();
thread_local uint32_t t_gemv_grid_override = 0;

namespace {

template <WKind KIND, int NSEG>
const void* gemv_func() {
    return reinterpret_cast<const void*>(&gemv_stream_kernel<KIND, NSEG>);
}

const void* select_gemv(WKind kind, bool swiglu) {
    switch (kind) {
        case W_Q4: return swiglu ? gemv_func<W_Q4, 2>() : gemv_func<W_Q4, 1>();
        case W_Q8: return swiglu ? gemv_func<W_Q8, 2>() : gemv_func<W_Q8, 1>();
        default: return swiglu ? gemv_func<W_BF16, 2>() : gemv_func<W_BF16, 1>();
    }
}

template <WKind KIND, int NSEG>
const void* tile_func(uint32_t nl) {
    switch (nl) {
        case 1: return reinterpret_cast<const void*>(&gemv_tile_kernel<KIND, NSEG, 1>);
        case 2: return reinterpret_cast<const void*>(&gemv_tile_kernel<KIND, NSEG, 2>);
        case 3: return reinterpret_cast<const void*>(&gemv_tile_kernel<KIND, NSEG, 3>);
        case 4: return reinterpret_cast<const void*>(&gemv_tile_kernel<KIND, NSEG, 4>);
        case 6: return reinterpret_cast<const void*>(&gemv_tile_kernel<KIND, NSEG, 6>);
        default: return reinterpret_cast<const void*>(&gemv_tile_kernel<KIND, NSEG, 8>);
    }
}
const void* tile_func(WKind kind, bool swiglu, uint32_t nl) {
    switch (kind) {
        case W_Q4: return swiglu ? tile_func<W_Q4, 2>(nl) : tile_func<W_Q4, 1>(nl);
        case W_Q8: return swiglu ? tile_func<W_Q8, 2>(nl) : tile_func<W_Q8, 1>(nl);
        default: return swiglu ? tile_func<W_BF16, 2>(nl) : tile_func<W_BF16, 1>(nl);
    }
}

template <WKind KIND, bool TAIL, bool ARGMAX>
const void* rows_func(uint32_t nb) {
    switch (nb) {
        case 3: return reinterpret_cast<const void*>(&gemv_rows_kernel<KIND, 3, TAIL, ARGMAX>);
        case 4: return reinterpret_cast<const void*>(&gemv_rows_kernel<KIND, 4, TAIL, ARGMAX>);
        default: return reinterpret_cast<const void*>(&gemv_rows_kernel<KIND, 5, TAIL, ARGMAX>);
    }
}
template <WKind KIND>
const void* rows_func(uint32_t nb, bool tail, bool argmax) {
    if (argmax) return tail ? rows_func<KIND, true, true>(nb) : rows_func<KIND, false, true>(nb);
    return tail ? rows_func<KIND, true, false>(nb) : rows_func<KIND, false, false>(nb);
}
const void* rows_func(WKind kind, uint32_t nb, bool tail, bool argmax) {
    switch (kind) {
        case W_Q4: return rows_func<W_Q4>(nb, tail, argmax);
        case W_Q8: return rows_func<W_Q8>(nb, tail, argmax);
        default: return rows_func<W_BF16>(nb, tail, argmax);
    }
}

// Blocks of `func` one CU holds at once (registers and LDS decide); cached per (kernel, LDS bytes).
uint32_t blocks_per_cu(const void* func, uint32_t lds_bytes) {
    static std::mutex mu;
    static std::map<std::pair<const void*, uint32_t>, int> cache;
    std::lock_guard<std::mutex> lk(mu);
    auto key = std::make_pair(func, lds_bytes);
    auto it = cache.find(key);
    if (it == cache.end()) {
        (void)raise_dynamic_lds(func, lds_bytes);
        int per_cu = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, func, kGemvBlock, lds_bytes) != hipSuccess || per_cu < 1)
            per_cu = 1;
        it = cache.emplace(key, per_cu).first;
    }
    return (uint32_t)it->second;
}

// The tile height and grid of a flat-stream launch, by everything they depend on.
struct GemvTiling {
    const void* func;
    uint32_t n[kMaxMats], cpr;
    uint32_t rows_per_tile, grid_blocks, grid_override;
    uint32_t rows, blocks, lr, chunks;  // the result; chunks: 16-byte chunks a thread (one-tile form), 0: the flat form
    bool same_request(const GemvTiling& o) const {
        return func == o.func && n[0] == o.n[0] && n[1] == o.n[1] && n[2] == o.n[2] && cpr == o.cpr &&
               rows_per_tile == o.rows_per_tile && grid_blocks == o.grid_blocks && grid_override == o.grid_override;
    }
};

// A thread's last tilings: 32 sets of four, the oldest of a set makes room (no lock, no growth).  With one place per hash two
// shapes of a model that fall on the same one are searched for on every call, some 1.5 us each.
GemvTiling* gemv_tiling_lookup(const GemvTiling& key, bool* found) {
    struct Set {
        GemvTiling way[4];  // func null: empty
        uint32_t next;
    };
    static thread_local Set sets[32];
    uint64_t h = (uint64_t)(uintptr_t)key.func;
    for (uint32_t v : {key.n[0], key.n[1], key.n[2], key.cpr}) h = (h ^ v) * 0x9E3779B97F4A7C15ull;
    Set& set = sets[h >> 59];
    for (GemvTiling& t : set.way)
        if (t.same_request(key)) {
            *found = true;
            return &t;
        }
    *found = false;
    GemvTiling* t = &set.way[set.next];
    set.next = (set.next + 1u) & 3u;
    t->func = nullptr;  // until the search has filled it in
    return t;
}

uint32_t ilog2(uint32_t v) {
    uint32_t r = 0;
    while ((1u << (r + 1)) <= v) ++r;
    return r;
}

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
template <typename TILES>
TileChoice gemv_tile_choice(WKind kind, uint32_t nseg, uint32_t K, uint32_t cpr, uint32_t gpr, uint32_t lr, uint32_t cus, TILES tiles_for) {
    TileChoice best{0, 0};
    uint64_t best_cost = ~0ull, best_per_cu = 0;
    if (kind != W_BF16 && gpr < 4) return best;  // a tile's scales are fetched in whole runs of four
    for (uint32_t nl : {1u, 2u, 3u, 4u, 6u, 8u}) {
        uint32_t r = nl * kGemvBlock / cpr;
        if (r > kGemvBlock / lr) r = kGemvBlock / lr;
        if (gpr && r > kTileGroups / gpr) r = kTileGroups / gpr;
        if (r == 0) continue;
        const uint64_t per_cu = (tiles_for(r) + cus - 1) / cus;
        const uint64_t cost = per_cu * (2 + (K + 2047) / 2048 + nl * nseg) + 2 * nl * nseg;
        if (cost < best_cost) {
            best_cost = cost;
            best_per_cu = per_cu;
            best = TileChoice{nl, r};
        }
    }
    const uint32_t few = kind == W_BF16 ? 2u : 5u, starts = kind == W_BF16 ? 5u : 3u;
    if (best.rows * nseg < few && best_per_cu > starts) best.chunks = 0;
    return best;
}

}  // namespace

// Shapes of the row-group form: rows of whole 256-byte blocks that the staging registers cover, group size 64,
// 32-bit byte offsets into the matrix, and enough rows that every CU gets at least two blocks of four-row passes.
// Batches of 5, 4 or 3 column blocks, whichever leaves the fewest unused slots in a row's last batch (at most 7 %).
uint32_t gemv_rows_batch(uint32_t n, uint32_t k, uint32_t bits, uint32_t group) {
    if (g_gemv_policy.flat_only || (bits != 4 && bits != 8 && bits != 16) || (bits != 16 && group != 64)) return 0;
    const uint32_t values = bits == 4 ? 32u : (bits == 8 ? 16u : 8u);
    if (k == 0 || k % values != 0) return 0;
    const uint32_t cpr = k / values;
    if (cpr % kRowLanes != 0 || k > (uint32_t)kStageRegs * kGemvBlock * 8u) return 0;
    const DeviceFacts* dev;
    if (device_facts(&dev) != FK_OK) return 0;
    const uint64_t passes = ((uint64_t)n + kPassRows - 1) / kPassRows;
    if (passes < 2ull * kBlockWaves * dev->cus || (uint64_t)n * cpr * 16ull > 0xffffffffull) return 0;
    const uint32_t cpl = cpr / kRowLanes;
    uint32_t nb = 0, best_slots = ~0u;
    for (uint32_t c : {5u, 4u, 3u}) {
        const uint32_t slots = (cpl + c - 1) / c * c;
        if (slots < best_slots) best_slots = slots, nb = c;
    }
    return best_slots * 100u <= cpl * 107u ? nb : 0u;
}

fk_status plan_gemv(const GemvRequest& rq, Launch* out) {
    const DeviceFacts* dev;
    FK_TRY(device_facts(&dev));
    const int nm = rq.swiglu ? 2 : rq.n_mats;
    if (nm < 1 || nm > kMaxMats) return set_error(FK_ERR_INVALID, "gemv: 1..3 matrices");
    const fk_weight* w0 = rq.mats[0];
    if (!w0 || !rq.x) return set_error(FK_ERR_INVALID, "gemv: null weight or activation pointer");
    const uint32_t K = w0->k, bits = w0->bits;
    if (bits != 4 && bits != 8 && bits != 16) return set_error(FK_ERR_UNSUPPORTED, "gemv: bits must be 4, 8 or 16");
    if (K == 0 || K % 64 != 0) return set_error(FK_ERR_UNSUPPORTED, "gemv: K must be a positive multiple of 64");
    uint32_t group = w0->group;
    if (bits != 16 && group != 32 && group != 64 && group != 128)
        return set_error(FK_ERR_UNSUPPORTED, "gemv: group size must be 32, 64 or 128");
    for (int m = 0; m < nm; ++m) {
        const fk_weight* w = rq.mats[m];
        if (!w || !w->w) return set_error(FK_ERR_INVALID, "gemv: null weight");
        if (w->k != K || w->bits != bits || (bits != 16 && w->group != group))
            return set_error(FK_ERR_INVALID, "gemv: fused matrices must share K, bits and group size");
        if (bits != 16 && (!w->scales || !w->biases)) return set_error(FK_ERR_INVALID, "gemv: null scales/biases");
        if (w->n == 0) return set_error(FK_ERR_INVALID, "gemv: matrix with zero rows");
        if (!rq.swiglu && !rq.y[m]) return set_error(FK_ERR_INVALID, "gemv: null output");
    }
    if (rq.swiglu) {
        if (rq.mats[0]->n != rq.mats[1]->n) return set_error(FK_ERR_INVALID, "gemv: gate and up need equal rows");
        if (!rq.y[0]) return set_error(FK_ERR_INVALID, "gemv: null output");
    }
    if (rq.argmax && (!rq.argmax->next_token || !rq.argmax->workspace))
        return set_error(FK_ERR_INVALID, "gemv: head argmax needs a token slot and a workspace");
    const WKind kind = bits == 4 ? W_Q4 : (bits == 8 ? W_Q8 : W_BF16);
    const uint32_t values = bits == 4 ? 32u : (bits == 8 ? 16u : 8u);
    const uint32_t cpr = K / values;
    const uint32_t nseg = rq.swiglu ? 2u : 1u;

    // Row-group form (gemv_rows.hpp): see gemv_rows_batch for the shapes.
    const uint32_t rows_nb = (!rq.swiglu && nm == 1 && !t_gemv_grid_override && !g_gemv_policy.rows_per_tile && !rq.res &&
                              !rq.res2 && !rq.bias[0])
                                 ? gemv_rows_batch(rq.mats[0]->n, K, bits, bits == 16 ? 64 : group)
                                 : 0u;
    if (rows_nb) {
        const uint32_t cpl = cpr / kRowLanes, nb = rows_nb;
        const uint32_t mb = bits == 4 ? 16u : 8u;
        bool ok = true;
        const uint64_t passes = (rq.mats[0]->n + kPassRows - 1) / kPassRows;
        if (bits != 16 && (((uintptr_t)rq.mats[0]->scales | (uintptr_t)rq.mats[0]->biases) & (mb - 1)) != 0) ok = false;
        if (((uintptr_t)rq.mats[0]->w & 15u) != 0) ok = false;
        const uint32_t lds = kind == W_Q4 ? gemv_rows_lds_bytes<W_Q4>(cpr)
                             : (kind == W_Q8 ? gemv_rows_lds_bytes<W_Q8>(cpr) : gemv_rows_lds_bytes<W_BF16>(cpr));
        if (ok && (int)lds <= dev->max_dyn_lds) {
            const void* f = rows_func(kind, nb, cpl % nb != 0, rq.argmax != nullptr);
            // whole rounds: every wave of the grid gets the same number of passes (to within one)
            const uint64_t cap = g_gemv_policy.grid_blocks ? g_gemv_policy.grid_blocks : (uint64_t)blocks_per_cu(f, lds) * dev->cus;
            const uint64_t block_passes = (passes + kBlockWaves - 1) / kBlockWaves;
            const uint64_t rounds = (block_passes + cap - 1) / cap;
            const uint64_t blocks = (block_passes + rounds - 1) / rounds;
            if (rq.argmax && blocks > kHeadArgmaxMaxBlocks)
                return set_error(FK_ERR_UNSUPPORTED, "gemv: head argmax over more blocks than its workspace holds");
            GemvArgmaxArgs a;
            memset(&a, 0, sizeof(a));
            if (rq.argmax) {
                a.tail.next_token = rq.argmax->next_token;
                a.tail.history = rq.argmax->history;
                a.tail.hist_counter = rq.argmax->hist_counter;
                a.tail.hist_capacity = rq.argmax->hist_capacity;
                a.tail.counter = reinterpret_cast<uint32_t*>(rq.argmax->workspace);
                a.tail.partial = reinterpret_cast<uint64_t*>(reinterpret_cast<char*>(rq.argmax->workspace) + 8);
            }
            uint32_t t0 = 0;
            for (int m = 0; m < nm; ++m) {
                a.w[m] = reinterpret_cast<const uint4*>(rq.mats[m]->w);
                a.sc[m] = rq.mats[m]->scales;
                a.bi[m] = rq.mats[m]->biases;
                a.bias[m] = rq.bias[m];
                a.y[m] = rq.y[m];
                a.n[m] = rq.mats[m]->n;
                a.tile_start[m] = t0;
                t0 += (rq.mats[m]->n + kPassRows - 1) / kPassRows;
            }
            a.tile_start[nm] = t0;
            a.n_mats = nm;
            a.K = K;
            a.cpr = cpr;
            a.gshift = bits == 16 ? 0 : ilog2(group / values);
            a.R = kPassRows;
            a.n_tiles = (uint32_t)passes;
            a.lr = kRowLanes;
            a.inv_cpr = 1.0f / (float)cpr;
            a.x = rq.x;
            a.norm_w = rq.norm_w;
            a.eps = rq.eps;
            a.res = rq.res;
            a.res2 = rq.res2;
            a.y_scale = 1.0f;
            out->func = f;
            out->grid = dim3((uint32_t)blocks, 1, 1);
            out->block = dim3(kGemvBlock, 1, 1);
            out->shmem = lds;
            if (rq.argmax)
                out->set_args(a);
            else
                out->set_args(static_cast<const GemvArgs&>(a));
            out->n_lead = 0;
            out->add_lead(a.x);
            out->add_lead(a.norm_w);
            out->add_lead(a.K);
            return raise_dynamic_lds(out->func, lds);
        }
    }
    if (rq.argmax) return set_error(FK_ERR_UNSUPPORTED, "gemv: head argmax needs a shape the row-group form takes");
    const void* func = select_gemv(kind, rq.swiglu);
    auto tiles_for = [&](uint32_t r) {
        uint64_t t = 0;
        if (rq.swiglu) return (uint64_t)((rq.mats[0]->n + r - 1) / r);
        for (int m = 0; m < nm; ++m) t += (rq.mats[m]->n + r - 1) / r;
        return t;
    };
    auto lds_for = [&](uint32_t r) {
        switch (kind) {
            case W_Q4: return gemv_lds_bytes<W_Q4>(cpr, r * cpr, nseg);
            case W_Q8: return gemv_lds_bytes<W_Q8>(cpr, r * cpr, nseg);
            default: return gemv_lds_bytes<W_BF16>(cpr, r * cpr, nseg);
        }
    };
    auto tile_lds = [&](uint32_t r, uint32_t nl) {
        const uint32_t gpr = bits == 16 ? 0u : K / group;
        switch (kind) {
            case W_Q4: return gemv_tile_lds_bytes<W_Q4>(cpr, r, gpr, nl, nseg);
            case W_Q8: return gemv_tile_lds_bytes<W_Q8>(cpr, r, gpr, nl, nseg);
            default: return gemv_tile_lds_bytes<W_BF16>(cpr, r, gpr, nl, nseg);
        }
    };
    // Blocks that can be resident at once (registers and LDS decide): the grid never
    // exceeds it, so no block waits for a slot and then pays the whole start-up chain
    // (stage x, first loads) a second time; surplus tiles go to the persistent loop,
    // whose next batch is already in flight while the current one is consumed.
    auto resident_for = [&](uint32_t lds_bytes) -> uint32_t { return blocks_per_cu(func, lds_bytes) * (uint32_t)dev->cus; };

    // Rows per tile.  A batch (4 x 16-byte loads per lane) costs the same whether its
    // lanes are full or not, and the blocks resident on a CU share its issue slots, so
    // the first figure of merit is the number of batches the busiest CU runs,
    // ceil(blocks / CUs) x tiles per block x batches per tile; ties go to the least
    // total work, batches over all tiles plus one unit per block for its start-up
    // (argument fetch, activation staging).  Measured on the 4B-class gate/up pair
    // (2 x 9728 x 2560): 19 rows per tile = 512 blocks of three 97 %-full batches runs
    // 10.4 us where one-batch tiles of 6 rows on 1280 blocks ran 12.2 us.
    // The search tries up to a few hundred tile heights, several microseconds on the host: more than a small launch
    // takes on the GPU.  What it finds depends on the shape alone, so a direct call looks it up (4864 x 896 int4, called
    // back to back: 6.9 us of host time per call with the search, 4.0 us without, as long as the runtime takes for an empty kernel).
    GemvTiling key;
    memset(&key, 0, sizeof(key));
    key.func = func;
    for (int m = 0; m < nm; ++m) key.n[m] = rq.mats[m]->n;
    key.cpr = cpr;
    key.rows_per_tile = g_gemv_policy.rows_per_tile;
    key.grid_blocks = g_gemv_policy.grid_blocks;
    key.grid_override = t_gemv_grid_override;
    bool found;
    GemvTiling& tiling = *gemv_tiling_lookup(key, &found);
    if (!found) {
        const uint32_t pos = kGemvBlock * (kGemvUnroll / nseg);
        uint32_t r_max = 8 * pos / cpr;  // up to eight batches per tile
        if (r_max < 1) r_max = 1;
        if (r_max > kGemvBlock) r_max = kGemvBlock;
        uint32_t best_r = 1, best_blocks = 1;
        uint64_t best_cost = ~0ull, best_waste = ~0ull;
        for (uint32_t r = 1; r <= r_max; ++r) {
            const uint32_t lds_r = lds_for(r);
            if ((int)lds_r > dev->max_dyn_lds) continue;
            const uint64_t tiles = tiles_for(r);
            uint64_t cap = t_gemv_grid_override ? t_gemv_grid_override
                           : (g_gemv_policy.grid_blocks ? g_gemv_policy.grid_blocks : resident_for(lds_r));
            const uint64_t blocks = tiles < cap ? tiles : cap;
            const uint64_t per_block = (tiles + blocks - 1) / blocks;
            const uint64_t batches = ((uint64_t)r * cpr + pos - 1) / pos;
            // fewer than two blocks (eight waves) on a CU cannot hide the load latency:
            // such a choice is priced as if it ran two
            uint64_t per_cu = (blocks + dev->cus - 1) / dev->cus;
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
        if (best_cost == ~0ull) return set_error(FK_ERR_UNSUPPORTED, "gemv: K too large for LDS staging");
        if (g_gemv_policy.rows_per_tile) {
            best_r = g_gemv_policy.rows_per_tile;
            const uint64_t tiles = tiles_for(best_r);
            const uint64_t cap = t_gemv_grid_override ? t_gemv_grid_override
                                 : (g_gemv_policy.grid_blocks ? g_gemv_policy.grid_blocks : resident_for(lds_for(best_r)));
            best_blocks = (uint32_t)(tiles < cap ? tiles : cap);
        }
        if ((int)lds_for(best_r) > dev->max_dyn_lds) return set_error(FK_ERR_UNSUPPORTED, "gemv: K too large for LDS staging");
        tiling = key;
        tiling.rows = best_r;
        tiling.blocks = best_blocks;
        // lanes of a row's sum: they fix the order of its additions, so the one-tile form takes the flat form's
        uint32_t lr = 1u << ilog2(kGemvBlock / best_r ? kGemvBlock / best_r : 1);
        if (lr > 64) lr = 64;
        while (lr > 1 && lr > cpr) lr >>= 1;
        tiling.lr = lr;
        tiling.chunks = 0;
        if (!key.rows_per_tile && !key.grid_blocks && !key.grid_override) {  // (those ask for the persistent form's tiles)
            const TileChoice c = gemv_tile_choice(kind, nseg, K, cpr, bits == 16 ? 0u : K / group, lr, (uint32_t)dev->cus, tiles_for);
            if (c.chunks && (int)tile_lds(c.rows, c.chunks) <= dev->max_dyn_lds) {
                tiling.rows = c.rows;
                tiling.blocks = (uint32_t)tiles_for(c.rows);
                tiling.chunks = c.chunks;
            }
        }
    }
    if (tiling.chunks) func = tile_func(kind, rq.swiglu, tiling.chunks);
    const uint32_t R = tiling.rows;
    const uint64_t tiles = tiles_for(R);
    if (tiles > 0x7fffffffull) return set_error(FK_ERR_UNSUPPORTED, "gemv: too many tiles");

    GemvArgs a;
    memset(&a, 0, sizeof(a));
    uint32_t t0 = 0;
    for (int m = 0; m < nm; ++m) {
        a.w[m] = reinterpret_cast<const uint4*>(rq.mats[m]->w);
        a.sc[m] = rq.mats[m]->scales;
        a.bi[m] = rq.mats[m]->biases;
        a.bias[m] = rq.bias[m];
        a.y[m] = rq.y[m];
        a.n[m] = rq.mats[m]->n;
        a.tile_start[m] = t0;
        t0 += (rq.mats[m]->n + R - 1) / R;
    }
    a.tile_start[nm] = t0;
    a.n_mats = nm;
    a.K = K;
    a.cpr = cpr;
    a.gshift = bits == 16 ? 0 : ilog2(group / values);
    a.R = R;
    a.n_tiles = (uint32_t)tiles;
    a.lr = tiling.lr;
    a.inv_cpr = 1.0f / (float)cpr;
    a.x = rq.x;
    a.norm_w = rq.norm_w;
    a.eps = rq.eps;
    a.res = rq.res;
    a.res2 = rq.res2;
    a.swiglu_variant = rq.swiglu_variant;
    a.y_scale = 1.0f;

    const uint32_t lds = tiling.chunks ? tile_lds(R, tiling.chunks) : lds_for(R);
    out->func = func;
    out->grid = dim3(tiling.blocks, 1, 1);
    out->block = dim3(kGemvBlock, 1, 1);
    out->shmem = lds;
    out->set_args(a);
    out->n_lead = 0;
    out->add_lead(a.x);
    out->add_lead(a.norm_w);
    out->add_lead(a.K);
    return raise_dynamic_lds(func, lds);
}

}  // namespace fk
