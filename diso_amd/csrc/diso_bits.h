// diso_bits.h - classification of 64 cells at once, on bit planes.
//
// The count pass keeps one bit per grid position (sample >= iso) in 64-bit words, one word per
// segment of 64 consecutive z positions. A cell's corners are then bits of the words of its four
// rows and of those words shifted by one, and every per-cell table lookup (triangle count, patch
// count, ambiguity) is a Boolean function of eight planes. eval() evaluates such a function for 32
// cells at a time as the decision tree of its truth table, taken from the case tables at compile
// time: constant and equal subtrees vanish, and equal subtrees under different prefixes are the
// same expression, which the compiler evaluates once. Each remaining node is one bit select.
//
// Plain C++ (host and device), so the rules are testable on the CPU.
#pragma once

#include <stdint.h>

#include "diso_tables.h"

#if defined(__HIPCC__)
#define DISO_BITS_HD __host__ __device__ inline __attribute__((always_inline))
#else
#define DISO_BITS_HD inline
#endif

namespace diso_bits {

constexpr uint64_t kMcTable[256] = {DISO_MC_CASE_VALUES};
constexpr uint64_t kDmcTable[256] = {DISO_DMC_CASE_VALUES};

// Boolean functions of a cell code. MC codes: Bourke corner order; DMC codes: Morton order.
template <int K>
struct McTriBit {  // bit K of the triangle count
    static constexpr bool at(int code) { return (DISO_MC_NTRI(kMcTable[code]) >> K) & 1; }
};
struct DmcAmbiguous {
    static constexpr bool at(int code) { return DISO_DMC_DIR(kDmcTable[code]) != 7; }
};
template <int D>
struct DmcDirIs {
    static constexpr bool at(int code) { return DISO_DMC_DIR(kDmcTable[code]) == D; }
};
template <int K>
struct DmcMorePatches {  // bit K of the patch count minus one (0 for codes without a patch)
    static constexpr bool at(int code) {
        const int n = DISO_DMC_NPATCH(kDmcTable[code]);
        return n > 0 && (((n - 1) >> K) & 1);
    }
};

// Order in which the tree tests the corners (fewest nodes among the orders tried: MC triangle
// bits 96, ambiguity and its directions 96, patch bits under 90).
constexpr int kOrder[8] = {0, 1, 7, 6, 4, 3, 2, 5};

constexpr int full_code(int level, int prefix, int rest) {
    int code = 0;
    for (int l = 0; l < 8; ++l) {
        const int bit = l < level ? (prefix >> l) & 1 : (rest >> (l - level)) & 1;
        code |= bit << kOrder[l];
    }
    return code;
}
template <class F>
constexpr bool all_equal(int level, int prefix, bool v) {
    for (int r = 0; r < (1 << (8 - level)); ++r)
        if (F::at(full_code(level, prefix, r)) != v) return false;
    return true;
}
// whether the subtrees of prefix with the level's corner clear and set agree (flip: are opposite)
template <class F>
constexpr bool halves_agree(int level, int prefix, bool flip) {
    for (int r = 0; r < (1 << (7 - level)); ++r)
        if ((F::at(full_code(level + 1, prefix, r)) != F::at(full_code(level + 1, prefix | 1 << level, r))) != flip)
            return false;
    return true;
}

template <class F, int L = 0, int P = 0>
DISO_BITS_HD uint32_t eval(const uint32_t (&c)[8]) {
    if constexpr (all_equal<F>(L, P, false)) {
        return 0u;
    } else if constexpr (all_equal<F>(L, P, true)) {
        return ~0u;
    } else if constexpr (halves_agree<F>(L, P, false)) {
        return eval<F, L + 1, P>(c);
    } else if constexpr (halves_agree<F>(L, P, true)) {
        return c[kOrder[L]] ^ eval<F, L + 1, P>(c);
    } else {
        const uint32_t lo = eval<F, L + 1, P>(c), hi = eval<F, L + 1, (P | 1 << L)>(c), s = c[kOrder[L]];
        return (s & hi) | (~s & lo);
    }
}

// Keeps the compiler from overlapping the two 32-cell halves of a segment (their interleaved
// temporaries would double the registers of the count pass).
DISO_BITS_HD void half_done() {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_sched_barrier(0);
#endif
}

DISO_BITS_HD int popc32(uint32_t v) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __popc(v);
#else
    return __builtin_popcount(v);
#endif
}
DISO_BITS_HD int popc64(uint64_t v) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __popcll(v);
#else
    return __builtin_popcountll(v);
#endif
}

// Lowest n bits (n clamped to [0, 64]).
DISO_BITS_HD uint64_t low_bits(int n) { return n >= 64 ? ~0ull : (n <= 0 ? 0ull : ((1ull << n) - 1)); }

// 8 bytes b[i] (i = plane) of eight positions each, to 8 codes (byte j = position j, bit i = plane
// i): an 8 x 8 bit transpose in two 32-bit halves (planes 0-3, planes 4-7), by exchanging blocks of
// 1, 2 and 4 bits (H. S. Warren, Hacker's Delight, "Transposing a bit matrix").
DISO_BITS_HD void transpose8(uint32_t &lo, uint32_t &hi) {
    uint32_t t;
    t = (lo ^ (lo >> 7)) & 0x00AA00AAu;
    lo ^= t ^ (t << 7);
    t = (hi ^ (hi >> 7)) & 0x00AA00AAu;
    hi ^= t ^ (t << 7);
    t = (lo ^ (lo >> 14)) & 0x0000CCCCu;
    lo ^= t ^ (t << 14);
    t = (hi ^ (hi >> 14)) & 0x0000CCCCu;
    hi ^= t ^ (t << 14);
    t = (lo ^ (hi << 4)) & 0xF0F0F0F0u;
    lo ^= t;
    hi ^= t >> 4;
}

// Bytes g = 0..3 of four words to four words: out[g] = bytes g of w[0], w[1], w[2], w[3].
DISO_BITS_HD void byte_transpose4(const uint32_t *w, uint32_t *out) {
#if defined(__HIP_DEVICE_COMPILE__)
    const uint32_t a = __builtin_amdgcn_perm(w[1], w[0], 0x05010400u), b = __builtin_amdgcn_perm(w[3], w[2], 0x05010400u);
    const uint32_t c = __builtin_amdgcn_perm(w[1], w[0], 0x07030602u), d = __builtin_amdgcn_perm(w[3], w[2], 0x07030602u);
    out[0] = __builtin_amdgcn_perm(b, a, 0x05040100u);
    out[1] = __builtin_amdgcn_perm(b, a, 0x07060302u);
    out[2] = __builtin_amdgcn_perm(d, c, 0x05040100u);
    out[3] = __builtin_amdgcn_perm(d, c, 0x07060302u);
#else
    for (int g = 0; g < 4; ++g) {
        out[g] = 0;
        for (int i = 0; i < 4; ++i) out[g] |= ((w[i] >> (8 * g)) & 0xffu) << (8 * i);
    }
#endif
}

// The codes of the 32 positions of eight planes, as 8 words of four codes.
DISO_BITS_HD void codes_of(const uint32_t (&c)[8], uint32_t (&out)[8]) {
    uint32_t lo[4], hi[4];
    byte_transpose4(c, lo);
    byte_transpose4(c + 4, hi);
    for (int g = 0; g < 4; ++g) {
        transpose8(lo[g], hi[g]);
        out[2 * g] = lo[g];
        out[2 * g + 1] = hi[g];
    }
}

// A segment: row (px, py) and z chunk of a grid of dims (g0, g1, g2), nchunk chunks per row.
struct Place {
    int px, py, chunk, g0, g1, g2, nchunk;
};

// Classification of one half of a segment: 32 positions, bit l = position 32 h + l.
struct Classified {
    uint32_t X, Y, Z;    // crossing edges owned along each axis
    uint32_t A;          // active cells
    uint32_t m0, m1;     // DMC: patch count minus one of the active cells
    uint32_t code[8];    // code planes (DMC: after the face-neighbour rule), valid where A
    int nf;              // MC triangles / DMC patches
};

// Half h of a segment's plane `w` whose row continues with plane `next` and was preceded by `prev`,
// and the same moved by one or two positions.
DISO_BITS_HD uint32_t half(uint64_t w, int h) { return (uint32_t)(w >> (32 * h)); }
DISO_BITS_HD uint32_t half_up(uint64_t w, uint64_t next, int h, int by) {
    const uint32_t lo = half(w, h), hi = h ? (uint32_t)next : half(w, 1);
    return (lo >> by) | (hi << (32 - by));
}
DISO_BITS_HD uint32_t half_down(uint64_t w, uint64_t prev, int h) {
    return (half(w, h) << 1) | ((h ? half(w, 0) : half(prev, 1)) >> 31);
}
DISO_BITS_HD uint64_t up1(uint64_t w, uint64_t next) { return (w >> 1) | (next << 63); }
DISO_BITS_HD uint64_t down1(uint64_t w, uint64_t prev) { return (w << 1) | (prev >> 63); }

// Classifies the cells of a segment (nothing where !valid) and hands each half to sink(h, c). load(dx,
// dy, dc): the inside plane of the segment dx rows along x, dy along y and dc chunks along z away; it
// is only called for segments of the grid. any(bits): whether `bits` is nonzero here or in a lane
// that runs with this one (so a rare step is skipped by all lanes together).
template <bool DMC, class Load, class Any, class Sink>
DISO_BITS_HD void classify(const Place &p, bool valid, Load load, Any any, Sink sink) {
    const bool anchor = valid && p.px < p.g0 - 1 && p.py < p.g1 - 1;
    const int nz = p.g2 - 1 - 64 * p.chunk;  // positions of the segment that anchor a cell
    const bool more = p.chunk + 1 < p.nchunk;
    // rows (0,0), (1,0), (0,1), (1,1) and their next chunks; a lane without cells reads its own row
    const int o = anchor ? 1 : 0;
    uint64_t a[4], n[4];
    for (int i = 0; i < 4; ++i) {
        a[i] = load((i & 1) * o, (i >> 1) * o, 0);
        n[i] = more ? load((i & 1) * o, (i >> 1) * o, 1) : 0ull;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        Classified r;
        const uint32_t am = anchor ? (uint32_t)low_bits(nz - 32 * h) : 0u;
        uint32_t w[4], u[4];
        for (int i = 0; i < 4; ++i) {
            w[i] = half(a[i], h);
            u[i] = half_up(a[i], n[i], h, 1);
        }
        r.X = (w[0] ^ w[1]) & am;
        r.Y = (w[0] ^ w[2]) & am;
        r.Z = (w[0] ^ u[0]) & am;
        r.A = r.X | r.Y | r.Z | (((w[0] ^ w[3]) | (w[0] ^ u[1]) | (w[0] ^ u[2]) | (w[0] ^ u[3])) & am);
        r.m0 = r.m1 = 0;
        r.nf = 0;
        for (int i = 0; i < 4; ++i) {
            // MC: Bourke corner order (rows 0, 1, 3, 2); DMC: Morton corner order
            const int at = DMC ? i : (i ^ (i >> 1));
            r.code[at] = w[i];
            r.code[4 + at] = u[i];
        }
        if (any(r.A)) {
            if (!DMC) {
                r.nf = popc32(eval<McTriBit<0>>(r.code) & am) + 2 * popc32(eval<McTriBit<1>>(r.code) & am) +
                       4 * popc32(eval<McTriBit<2>>(r.code) & am);
            } else {
                // an ambiguous cell is inverted when its face neighbour in the tabulated direction
                // exists and is ambiguous too (src/cudualmc.cu:815-839)
                if (any(eval<DmcAmbiguous>(r.code) & am)) {
                    uint32_t flip = 0;
                    // the neighbour one row further (k = 1) or before (k = -1) along x or y: its rows
                    // on that side (`far`) and, on the other, the cell's own
                    auto along = [&](uint32_t d, bool exists, bool x, int k) {
                        d = exists && anchor ? d : 0u;
                        if (!any(d)) return;
                        const int far = d ? (k < 0 ? -1 : 2) : 0, one = d ? 1 : 0;
                        const int i0 = 0, i1 = x ? 2 : 1, j0 = x ? 1 : 2, j1 = 3;  // low and high side rows
                        const int dx0 = x ? far : 0, dy0 = x ? 0 : far, dx1 = x ? far : one, dy1 = x ? one : far;
                        const uint64_t f0 = load(dx0, dy0, 0), f1 = load(dx1, dy1, 0);
                        const uint64_t e0 = h && more ? load(dx0, dy0, 1) : 0ull, e1 = h && more ? load(dx1, dy1, 1) : 0ull;
                        const uint32_t w0 = half(f0, h), w1 = half(f1, h), g0 = half_up(f0, e0, h, 1), g1 = half_up(f1, e1, h, 1);
                        uint32_t q[8];
                        q[i0] = k < 0 ? w0 : w[j0], q[i1] = k < 0 ? w1 : w[j1];
                        q[j0] = k < 0 ? w[i0] : w0, q[j1] = k < 0 ? w[i1] : w1;
                        q[4 + i0] = k < 0 ? g0 : u[j0], q[4 + i1] = k < 0 ? g1 : u[j1];
                        q[4 + j0] = k < 0 ? u[i0] : g0, q[4 + j1] = k < 0 ? u[i1] : g1;
                        flip |= d & eval<DmcAmbiguous>(q);
                    };
                    along(eval<DmcDirIs<0>>(r.code) & am, p.px >= 1, true, -1);
                    along(eval<DmcDirIs<1>>(r.code) & am, p.px + 1 < p.g0 - 1, true, 1);
                    along(eval<DmcDirIs<2>>(r.code) & am, p.py >= 1, false, -1);
                    along(eval<DmcDirIs<3>>(r.code) & am, p.py + 1 < p.g1 - 1, false, 1);
                    const uint32_t d4 = eval<DmcDirIs<4>>(r.code) & am & (p.chunk == 0 && h == 0 ? ~1u : ~0u);
                    const uint32_t d5 = eval<DmcDirIs<5>>(r.code) & am & (uint32_t)low_bits(nz - 1 - 32 * h);
                    if (any(d4)) {
                        uint32_t q[8];
                        for (int i = 0; i < 4; ++i) {
                            const uint64_t before = !h && p.chunk > 0 ? load((i & 1) * o, (i >> 1) * o, -1) : 0ull;
                            q[i] = half_down(a[i], before, h);
                            q[4 + i] = w[i];
                        }
                        flip |= d4 & eval<DmcAmbiguous>(q);
                    }
                    if (any(d5)) {
                        uint32_t q[8];
                        for (int i = 0; i < 4; ++i) {
                            q[i] = u[i];
                            q[4 + i] = half_up(a[i], n[i], h, 2);
                        }
                        flip |= d5 & eval<DmcAmbiguous>(q);
                    }
                    for (int i = 0; i < 8; ++i) r.code[i] ^= flip;
                }
                r.m0 = eval<DmcMorePatches<0>>(r.code) & r.A;
                r.m1 = eval<DmcMorePatches<1>>(r.code) & r.A;
                r.nf = popc32(r.A) + popc32(r.m0) + 2 * popc32(r.m1);
            }
        }
        sink(h, r);
        half_done();
    }
}

}  // namespace diso_bits
