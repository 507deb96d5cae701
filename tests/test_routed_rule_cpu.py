"""Which routed projections serve an expert's routes together: the rule at the sizes it was measured at, and for those that the GPU
tests of that form run."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "fusekit_amd", "csrc")

# (experts, outputs, K, tokens, top-k, bits, group): outputs no multiple of 16; K of 11 and of 3 groups (waves with more and fewer, and
# with none); eight bits with groups of 64 and 128; more experts than a wave; 1024 routes, the most
TOGETHER = [(8, 2005, 704, 24, 2, 4, 64), (4, 2189, 192, 40, 4, 4, 64), (16, 731, 256, 30, 6, 8, 64), (16, 1720, 384, 17, 3, 8, 128),
            (100, 330, 128, 250, 4, 8, 64), (5, 1030, 64, 512, 2, 4, 64)]

# experts, routes, outputs, K, bits, pair, together: both sides of the line
MEASURED = [(64, 36, 1408, 2048, 4, 1, 0), (64, 48, 1408, 2048, 4, 1, 1), (64, 48, 1408, 2048, 8, 1, 1), (64, 48, 2048, 1408, 4, 0, 0),
            (64, 60, 2048, 1408, 4, 0, 1), (64, 576, 2048, 1408, 4, 0, 1), (128, 192, 2048, 768, 4, 0, 0), (128, 384, 2048, 768, 4, 0, 1),
            (128, 96, 2048, 768, 8, 0, 1), (256, 384, 2048, 512, 4, 0, 0), (32, 24, 1024, 1024, 4, 1, 0), (32, 96, 1024, 1024, 4, 1, 1),
            (16, 128, 1024, 2048, 4, 0, 1), (16, 128, 1024, 2048, 8, 0, 1), (2, 8, 512, 512, 4, 1, 0), (8, 6, 2048, 3584, 4, 0, 0), (8, 32, 2048, 3584, 4, 0, 1)]

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "routed_rule.hpp"
using namespace fk;

int main(int argc, char** argv) {
    int bad = 0;
    for (int i = 1; i + 6 < argc; i += 7) {
        unsigned v[7];
        for (int j = 0; j < 7; ++j) v[j] = (unsigned)atoi(argv[i + j]);
        if (routes_served_together(v[0], v[1], v[2], v[3], v[4], v[5] != 0, 256) != (v[6] != 0)) {
            printf("%u experts %u routes %u x %u, %u bits, pair %u: not %u\n", v[0], v[1], v[2], v[3], v[4], v[5], v[6]);
            ++bad;
        }
    }
    // more routes never leave the form again; a wave's slabs cover its share of K, two at the least
    const unsigned e[] = {2, 5, 8, 64, 100, 256}, n[] = {16, 333, 1408, 4096}, bits[] = {4, 8};
    for (unsigned E : e)
        for (unsigned N : n)
            for (unsigned K = 64; K <= 4096; K += 64)
                for (unsigned b : bits) {
                    const unsigned slabs = rt_slabs(K, b), share = (K / 64 + kRtWaves - 1) / kRtWaves;
                    if (slabs < 2 || slabs % 2 || slabs * rt_slab_groups(b) < share) ++bad;
                    for (int pair = 0; pair < 2; ++pair) {
                        bool was = false;
                        for (unsigned R = 2; R <= 1024; ++R) {
                            const bool is = routes_served_together(E, R, N, K, b, pair != 0, 256);
                            if (was && !is) ++bad;
                            was = is;
                        }
                    }
                }
    return bad ? 1 : 0;
}
"""


def test_the_rule_on_both_sides_of_its_line(tmp_path):
    src, exe = tmp_path / "rule.cpp", tmp_path / "rule"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-I", CSRC, str(src), "-o", str(exe)])
    points = MEASURED + [(e, t * k, o, K, b, pair, 1) for e, o, K, t, k, b, _ in TOGETHER for pair in (0, 1)]
    done = subprocess.run([str(exe)] + [str(v) for p in points for v in p], timeout=120, stdout=subprocess.PIPE, text=True)
    assert done.returncode == 0, done.stdout[-2000:]
