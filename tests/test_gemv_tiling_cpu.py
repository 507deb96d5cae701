"""How the GEMV cuts a launch into tiles: what a thread keeps of its searches is only ever given to the same launch again, and no
tile of the one-tile form asks for more than its kernel fetches."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "fusekit_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <initializer_list>
#include "gemv_tiling.hpp"
using namespace fk;

static const uint32_t kCus = 256, kMaxLds = 160 * 1024;
static unsigned per_cu(uint32_t lds) { const unsigned n = kMaxLds / (lds ? lds : 1u); return n < 1 ? 1 : (n > 8 ? 8 : n); }
static bool search(const GemvShape& s, GemvTiling* t) { return gemv_tiling(s, kCus, kMaxLds, per_cu, t); }
static GemvTilings kept;

// as a call does: looked up, else searched for and kept
static int call(const GemvShape& s) {
    GemvTiling fresh;
    if (!search(s, &fresh)) return 0;
    const GemvTiling* t = kept.find(s);
    if (!t) t = kept.keep(s, fresh);
    const uint32_t cpr = s.cpr(), gpr = s.gpr();
    const bool same = t->rows == fresh.rows && t->blocks == fresh.blocks && t->lr == fresh.lr && t->chunks == fresh.chunks;
    const bool fits = !t->chunks || (t->rows >= 1 && t->rows * cpr <= t->chunks * kGemvBlock && t->rows * t->lr <= (uint32_t)kGemvBlock &&
                                     t->blocks == s.tiles(t->rows) && s.tile_lds(t->rows, t->chunks) <= kMaxLds &&
                                     (s.kind == W_BF16 || (gpr >= 4 && s.K % s.group == 0 && t->rows * gpr <= kTileGroups)));
    if (same && fits) return 0;
    printf("kind %d nseg %u n %u K %u group %u: rows %u (%u groups) chunks %u%s\n", s.kind, s.nseg, s.n[0], s.K, s.group, t->rows,
           t->rows * gpr, t->chunks, same ? "" : ", another launch's");
    return 1;
}

static GemvShape shape(WKind kind, uint32_t nseg, uint32_t n, uint32_t K, uint32_t group) {
    GemvShape s;
    s.kind = kind;
    s.nseg = nseg;
    s.n_mats = nseg;
    s.n[0] = n;
    s.n[1] = nseg == 2 ? n : 0;
    s.K = K;
    s.group = group;
    return s;
}

int main() {
    int bad = 0;
    for (uint32_t n : {1u, 2u, 7u, 129u, 896u, 1181u, 2560u, 4864u, 9728u, 14336u, 65537u})
        for (uint32_t K = 64; K <= 16384; K += K < 1024 ? 64 : 512)
            for (uint32_t nseg : {1u, 2u})
                for (WKind kind : {W_Q4, W_Q8, W_BF16})
                    for (uint32_t group : {64u, 32u, 128u, 64u, 128u, 32u})
                        bad += call(shape(kind, nseg, n, K, kind == W_BF16 ? 0 : group));
    // a fan-out of the same first matrix, and a policy, are other launches too
    GemvShape s = shape(W_Q4, 1, 2560, 2560, 64);
    bad += call(s);
    s.n_mats = 3, s.n[1] = s.n[2] = 512;
    bad += call(s);
    s.rows_per_tile = 3;
    bad += call(s);
    s.grid_override = 128;
    bad += call(s);
    return bad ? 1 : 0;
}
"""


def test_a_kept_tiling_is_its_own_launchs(tmp_path):
    src, exe = tmp_path / "tiling.cpp", tmp_path / "tiling"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-fsanitize=address,undefined", "-I", CSRC, str(src), "-o", str(exe)])
    done = subprocess.run([str(exe)], timeout=120, stdout=subprocess.PIPE, text=True)
    assert done.returncode == 0, done.stdout[-2000:]
