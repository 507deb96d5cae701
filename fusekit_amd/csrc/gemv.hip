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

uint32_t ilog2(uint32_t v) {
    uint32_t r = 0;
    while ((1u << (r + 1)) <= v) ++r;
    return r;
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
    // The search tries up to a few hundred tile heights, several microseconds on the host: more than a small launch
    // takes on the GPU.  What it finds depends on the shape alone, so a direct call looks it up (4864 x 896 int4, called
    // back to back: 6.9 us of host time per call with the search, 4.0 us without, as long as the runtime takes for an empty kernel).
    GemvShape shape;
    shape.kind = kind;
    shape.nseg = nseg;
    shape.n_mats = (uint32_t)nm;
    for (int m = 0; m < nm; ++m) shape.n[m] = rq.mats[m]->n;
    shape.K = K;
    shape.group = bits == 16 ? 0u : group;
    shape.rows_per_tile = g_gemv_policy.rows_per_tile;
    shape.grid_blocks = g_gemv_policy.grid_blocks;
    shape.grid_override = t_gemv_grid_override;
    static thread_local GemvTilings kept;
    const GemvTiling* known = kept.find(shape);
    if (!known) {
        GemvTiling found;
        if (!gemv_tiling(shape, (uint32_t)dev->cus, (uint32_t)dev->max_dyn_lds, [&](uint32_t lds_bytes) { return blocks_per_cu(func, lds_bytes); }, &found))
            return set_error(FK_ERR_UNSUPPORTED, "gemv: K too large for LDS staging");
        known = kept.keep(shape, found);
    }
    const GemvTiling& tiling = *known;
    if (tiling.chunks) func = tile_func(kind, rq.swiglu, tiling.chunks);
    const uint32_t R = tiling.rows;
    const uint64_t tiles = shape.tiles(R);
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

    const uint32_t lds = tiling.chunks ? shape.tile_lds(R, tiling.chunks) : shape.flat_lds(R);
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
