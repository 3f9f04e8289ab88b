"""The bit-plane classification of the count pass (diso_amd/csrc/diso_bits.h), compiled with g++ and
compared on the CPU with the per-cell rule: code from the eight corners, triangle and patch counts
and the ambiguity direction from the case tables, and the face neighbour's inversion evaluated cell
by cell. Every position of random grids of odd sizes, sparse and dense, is checked: row tails, rows
and chunks at the grid's border, and chunk boundaries that the ambiguity rule crosses."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <stdio.h>
#include <stdlib.h>
#include <vector>
#include "diso_bits.h"
using namespace diso_bits;

#define CHECK(c) do { if (!(c)) { printf("FAIL line %d: %s (grid %d %d %d, at %d %d %d)\n", __LINE__, #c, G0, G1, G2, X, Y, Z); return 1; } } while (0)

static int G0, G1, G2, X, Y, Z;
static std::vector<unsigned char> in;
static int bit(int x, int y, int z) { return in[((size_t)x * G1 + y) * G2 + z]; }

static int mc_code(int x, int y, int z) {
    static const int c[8][3] = {{0,0,0},{1,0,0},{1,1,0},{0,1,0},{0,0,1},{1,0,1},{1,1,1},{0,1,1}};
    int code = 0;
    for (int i = 0; i < 8; ++i) code |= bit(x + c[i][0], y + c[i][1], z + c[i][2]) << i;
    return code;
}
static int dmc_raw(int x, int y, int z) {
    int code = 0;
    for (int i = 0; i < 8; ++i) code |= bit(x + (i & 1), y + ((i >> 1) & 1), z + (i >> 2)) << i;
    return code;
}
static int dmc_good(int x, int y, int z) {
    const int code = dmc_raw(x, y, z), dir = DISO_DMC_DIR(DISO_DMC_CASE[code]);
    if (dir == 7) return code;
    int n[3] = {x, y, z};
    const int lim[3] = {G0, G1, G2};
    n[dir >> 1] += (dir & 1) ? 1 : -1;
    if (n[dir >> 1] < 0 || n[dir >> 1] >= lim[dir >> 1] - 1) return code;
    return DISO_DMC_DIR(DISO_DMC_CASE[dmc_raw(n[0], n[1], n[2])]) != 7 ? code ^ 0xff : code;
}

template <bool DMC>
static int check_grid() {
    const int nchunk = (G2 + 63) / 64;
    std::vector<uint64_t> w((size_t)G0 * G1 * nchunk, 0);
    for (int x = 0; x < G0; ++x)
        for (int y = 0; y < G1; ++y)
            for (int z = 0; z < G2; ++z)
                w[((size_t)x * G1 + y) * nchunk + z / 64] |= (uint64_t)bit(x, y, z) << (z % 64);
    for (int x = 0; x < G0; ++x)
        for (int y = 0; y < G1; ++y)
            for (int c = 0; c < nchunk; ++c) {
                X = x, Y = y, Z = 64 * c;
                const Place p{x, y, c, G0, G1, G2, nchunk};
                bool outside = false;
                auto load = [&](int dx, int dy, int dc) -> uint64_t {
                    if (x + dx < 0 || x + dx >= G0 || y + dy < 0 || y + dy >= G1 || c + dc < 0 || c + dc >= nchunk) {
                        outside = true;
                        return 0;
                    }
                    return w[((size_t)(x + dx) * G1 + y + dy) * nchunk + c + dc];
                };
                uint64_t pX = 0, pY = 0, pZ = 0, pA = 0, m0 = 0, m1 = 0;
                uint32_t codes[2][8];
                int rf = 0;
                auto some = [](uint32_t b) { return b != 0; };
                classify<DMC>(p, true, load, some, [&](int h, const Classified &r) {
                    pX |= (uint64_t)r.X << (32 * h), pY |= (uint64_t)r.Y << (32 * h), pZ |= (uint64_t)r.Z << (32 * h);
                    pA |= (uint64_t)r.A << (32 * h), m0 |= (uint64_t)r.m0 << (32 * h), m1 |= (uint64_t)r.m1 << (32 * h);
                    codes_of(r.code, codes[h]);
                    rf += r.nf;
                });
                CHECK(!outside);
                bool none = true;
                classify<DMC>(p, false, load, some, [&](int, const Classified &r) {
                    none &= !r.X && !r.Y && !r.Z && !r.A && !r.m0 && !r.m1 && r.nf == 0;
                });
                CHECK(none && !outside);
                int nv = 0, nf = 0;
                for (int l = 0; l < 64; ++l) {
                    const int z = 64 * c + l;
                    Z = z;
                    const bool cell = x < G0 - 1 && y < G1 - 1 && z < G2 - 1;
                    const int ex = cell && bit(x, y, z) != bit(x + 1, y, z), ey = cell && bit(x, y, z) != bit(x, y + 1, z);
                    const int ez = cell && bit(x, y, z) != bit(x, y, z + 1);
                    CHECK((int)((pX >> l) & 1) == ex && (int)((pY >> l) & 1) == ey && (int)((pZ >> l) & 1) == ez);
                    nv += ex + ey + ez;
                    const int code = !cell ? 0 : (DMC ? dmc_good(x, y, z) : mc_code(x, y, z));
                    const bool active = code != 0 && code != 255;
                    CHECK(((pA >> l) & 1) == active);
                    if (!active) {
                        CHECK(!((m0 >> l) & 1) && !((m1 >> l) & 1));
                        continue;
                    }
                    CHECK((int)((codes[l / 32][l / 4 % 8] >> (8 * (l % 4))) & 0xff) == code);
                    if (DMC) {
                        const int np = DISO_DMC_NPATCH(DISO_DMC_CASE[code]);
                        CHECK((int)(1 + ((m0 >> l) & 1) + 2 * ((m1 >> l) & 1)) == np);
                        nf += np;
                    } else {
                        nf += DISO_MC_NTRI(DISO_MC_CASE[code]);
                    }
                }
                CHECK(popc64(pX) + popc64(pY) + popc64(pZ) == nv && rf == nf);
            }
    return 0;
}

int main(int argc, char **argv) {
    G0 = atoi(argv[1]), G1 = atoi(argv[2]), G2 = atoi(argv[3]);
    srand(atoi(argv[4]));
    const int per_mille = atoi(argv[5]);  // share of inside samples
    in.resize((size_t)G0 * G1 * G2);
    for (auto &v : in) v = rand() % 1000 < per_mille;
    if (check_grid<false>() || check_grid<true>()) return 1;
    // every code alone: a grid of one cell, all 256 configurations
    G0 = G1 = G2 = 2;
    in.resize(8);
    for (int code = 0; code < 256; ++code) {
        for (int i = 0; i < 8; ++i) in[((i & 1) * 2 + ((i >> 1) & 1)) * 2 + (i >> 2)] = (code >> i) & 1;
        if (check_grid<false>() || check_grid<true>()) return 1;
    }
    printf("ok\n");
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("bits")
    src, exe = d / "bits.cpp", d / "bits"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I" + os.path.join(ROOT, "diso_amd", "csrc"), "-o", str(exe), str(src)],
                   check=True)
    return str(exe)


@pytest.mark.parametrize("dims", [(2, 2, 2), (5, 4, 63), (4, 5, 64), (6, 3, 65), (4, 4, 66), (7, 6, 127), (5, 6, 130),
                                  (3, 9, 193), (9, 8, 11)])
@pytest.mark.parametrize("per_mille", [8, 500, 700])
def test_planes_equal_the_per_cell_rule(program, dims, per_mille):
    r = subprocess.run([program, *map(str, dims), "7", str(per_mille)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "ok" in r.stdout, r.stdout[-500:]
