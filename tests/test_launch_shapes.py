"""Launch shapes and block orders (diso_amd/csrc/diso_launch.h), compiled with g++ and checked on the CPU
at every size up to the largest grid the engine accepts (2^32 segments): no dimension reaches 2^32
threads, every block is launched, and the block orders are permutations."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <stdio.h>
#include <stdlib.h>
#include <vector>
#include "diso_launch.h"
using namespace diso_launch;

#define CHECK(c) do { if (!(c)) { printf("FAIL line %d: %s (blocks %lld)\n", __LINE__, #c, (long long)nb); return 1; } } while (0)

static int shape(int64_t nb, int threads) {
    const Shape s = shape_of(nb, threads);
    CHECK((int64_t)s.x * threads < (1ll << 32) && s.y >= 1 && s.y < 65536);
    CHECK((int64_t)s.x * s.y >= nb && (int64_t)s.x * s.y < nb + 8ll * s.y + 8);
    CHECK(s.y == 1 || s.x % 8 == 0);  // block i on XCD i % 8
    CHECK(s.y == 1 ? (int64_t)s.x == nb : nb * threads > (1ll << 32) - 8ll * threads);
    return 0;
}

int main() {
    int64_t nb = 0;
    for (int threads : {64, 256})
        for (nb = 1; nb < (1ll << 37); nb = nb + 1 + nb / 7)
            for (int64_t d = -2; d <= 2; ++d)
                if (nb + d > 0 && shape(nb + d, threads)) return 1;
    for (int threads : {64, 256})  // around the limit
        for (int64_t d = -20; d <= 20; ++d)
            if (shape((1ll << 32) / threads + d, threads)) return 1;
    // the gather of a grid of 2^32 segments, 65 blocks for every 32
    if (shape(stripe_blocks((1ll << 32) / 32 * 65), 64)) return 1;

    // every block number of the shape takes one block, or none
    for (nb = 1; nb < 3000; nb += 1 + nb / 9) {
        std::vector<int> a(nb, 0), b(nb, 0);
        for (int64_t i = 0; i < stripe_blocks(nb) + 40; ++i) {  // (40: a shape's own padding)
            const int64_t k = xcd_stripe(i, nb);
            CHECK(k >= 0);
            if (k < nb) ++a[k];
        }
        for (int64_t i = 0; i < nb; ++i) {
            const int64_t k = xcd_block(i, nb);
            CHECK(k >= 0 && k < nb);
            ++b[k];
        }
        for (int64_t k = 0; k < nb; ++k) CHECK(a[k] == 1 && b[k] == 1);
    }
    // large: the stripes' inverse, at sampled blocks
    nb = 67600000 + 13;
    const int64_t c = stripe_len(nb);
    for (int64_t k = 0; k < nb; k += 99991) {
        const int64_t t = k / c, i = (t / 8 * c + k % c) * 8 + t % 8;
        CHECK(i < stripe_blocks(nb) && xcd_stripe(i, nb) == k);
    }
    printf("ok\n");
    return 0;
}
"""


def test_launch_shapes(tmp_path):
    src, exe = tmp_path / "launch.cpp", tmp_path / "launch"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I" + os.path.join(ROOT, "diso_amd", "csrc"), "-o", str(exe), str(src)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "ok" in r.stdout, r.stdout[-500:]
