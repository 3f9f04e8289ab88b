// diso_hip.hip - DiffMC / DiffDMC engine for MI355X (gfx950), behind the C ABI of diso_hip.h.
//
// Work decomposition
//   The (virtually padded) grid G = [g0,g1,g2] is cut into "segments": one z-row (px,py) of the
//   grid, split into chunks of 64 consecutive z positions, bit l of a 64-bit plane standing for
//   position pz = 64*chunk + l. Segment order (px, py, chunk) is the grid's linear order
//   (x-major, z fastest), which is the order in which the reference emits its vertices and faces
//   (used cells in increasing linear cell id, src/cumc.cu:299-311,370-410,564-610). So the output
//   position of any cell's first vertex / face is
//       base(segment) + bits of the segment's planes below its position,
//   and only the per-segment bases are stored (16 bytes per 64 cells). The count pass also stores the
//   classification as bit planes and codes (struct Planes), which the later passes read instead of
//   re-classifying (the recompute-classification backward re-derives the crossings from the samples
//   instead), and deals the active cells into units of 64, the emission's work items: a surface
//   fills few positions of a segment, and a wave that took segments would run half empty.
//
// Kernels
//   mask_kernel           the samples' inside and below bits as planes, and their flags.
//   count_kernel          classify + count, a lane per segment, + single-pass decoupled look-back
//                         scan of segment counts (also over the segments of a batch of grids).
//   emit_mc_kernel        MC vertices and triangles (+ shift / normalise / int64 epilogue).
//   emit_dmc_kernel       DMC vertices (patch means) and quads.
//   dmc_edge_grad_kernel  DMC backward, first step: per crossing edge, the sum of its <= 4 quad
//                         corners' vertex gradients / patch sizes.
//   bwd_mc_kernel         MC gather backward (DMC: on those edge gradients): one lane per touched
//                         grid vertex sums its <= 6 incident edges, deterministic, no atomics.
//   split_*_kernel        DiffDMC's quad -> triangle split.
//   *_batch_kernel        the same passes over many grids in one launch.
//
// Floating point: forward results use only IEEE +, -, *, /, sqrt and compares, in the
// reference's operation order, built with -ffp-contract=off and correctly rounded division, so
// fp32 vertices equal an fp32 CPU evaluation of the same expressions bit for bit. The fp32
// backward uses one hardware reciprocal per edge (gradients are compared within a tolerance).
#include <hip/hip_runtime.h>

#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <mutex>
#include <vector>

#include "diso_hip.h"
#include "diso_bits.h"
#include "diso_host.h"
#include "diso_launch.h"
#include "diso_scan_word.h"
#include "diso_tables.h"

namespace {

constexpr int kWave = 64;
constexpr int kWavesPerBlock = 4;
constexpr int kBlock = kWave * kWavesPerBlock;
constexpr uint32_t kSpinLimit = 1u << 20;  // bounded look-back wait (well under a second); never expected
constexpr int kCtlHeader = 64;             // bytes

__constant__ uint64_t kMcCase[256] = {DISO_MC_CASE_VALUES};
__constant__ uint64_t kDmcCase[256] = {DISO_DMC_CASE_VALUES};

// ------------------------------------------------------------------------------------------
// Geometry and sampling

struct Geo {
    int g0, g1, g2;  // conceptual grid (padded dims when padding is virtual)
    int n0, n1, n2;  // stored grid dims
    int off;         // stored sample (i,j,k) sits at conceptual (i+off, j+off, k+off)
    int nchunk;      // ceil(g2 / 64)
    int64_t nseg;    // g0 * g1 * nchunk
    double rchunk, rg1;  // 1 / nchunk, 1 / g1 (seg_pos)
};

template <typename S>
struct In {
    const S *sdf;
    const S *deform;  // [n0,n1,n2,3] or nullptr
    S iso;
    S pad;            // value of samples outside the stored grid (iso + 1)
    Geo geo;
};

template <typename S>
struct V3 {
    S x, y, z;
};

// Stores of outputs that no later kernel reads (vertices, faces, dense gradients): non-temporal,
// so these streams do not evict from L2 the inputs that the gathers re-read.
template <typename T>
__device__ __forceinline__ void put(T *p, T v) {
    __builtin_nontemporal_store(v, p);
}

// (Bitwise &, not &&: no short-circuit branch, so loads guarded by it stay branch-free.)
template <typename S>
__device__ __forceinline__ bool in_data(const In<S> &in, int x, int y, int z) {
    return ((unsigned)(x - in.geo.off) < (unsigned)in.geo.n0) & ((unsigned)(y - in.geo.off) < (unsigned)in.geo.n1) &
           ((unsigned)(z - in.geo.off) < (unsigned)in.geo.n2);
}

template <typename S>
__device__ __forceinline__ int64_t data_index(const In<S> &in, int x, int y, int z) {
    return ((int64_t)(x - in.geo.off) * in.geo.n1 + (y - in.geo.off)) * in.geo.n2 + (z - in.geo.off);
}

// sdf sample at conceptual (x,y,z); samples outside the stored grid read as the pad value, so no
// coordinate can address memory outside the input.
// (Branch-free: a sample outside the stored grid loads element 0 and is replaced by the pad value,
// so no lane needs its own execution mask around the load.)
template <typename S>
__device__ __forceinline__ S sample(const In<S> &in, int x, int y, int z) {
    const bool ok = in_data(in, x, y, z);
    const S v = in.sdf[ok ? data_index(in, x, y, z) : 0];
    return ok ? v : in.pad;
}

// clamp(x, a, b) = min(max(a, x), b) as in src/cumc.cu:80-91.
template <typename S>
__device__ __forceinline__ S clamp01(S v) {
    S m = S(0) > v ? S(0) : v;
    return m < S(1) ? m : S(1);
}

template <typename S>
__device__ __forceinline__ S interp_t(S d0, S d1, S iso) {
    return (d1 != d0) ? clamp01<S>((iso - d0) / (d1 - d0)) : S(0.5);  // src/cumc.cu:356
}

// ------------------------------------------------------------------------------------------
// Wave primitives

__device__ __forceinline__ int lane_id() { return (int)__lane_id(); }

// Set bits of a wave-wide mask below the calling lane (v_mbcnt_lo / v_mbcnt_hi: two VALU
// instructions, where masking with a per-lane 64-bit shift and counting takes six).
__device__ __forceinline__ int lanes_below(uint64_t mask) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// Inclusive prefix over the wave of a 32-bit value: a scan within each row of 16 lanes (DPP row
// shifts by 1, 2, 4, 8; lanes before the row start read 0), then the last lane of row 0 added to
// rows 1 and 3 and the last lane of row 1 (by then the sum of rows 0 and 1) to rows 2 and 3 (DPP
// row broadcasts). Six adds. Several small counts can be scanned at once, each in a bit field wide
// enough for its wave total. Must be reached by all 64 lanes.
__device__ __forceinline__ uint32_t wave_incl_dpp(uint32_t v) {
    int x = (int)v;
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);   // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);   // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);   // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);   // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15 to rows 1, 3
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31 to rows 2, 3
    return (uint32_t)x;
}

__device__ __forceinline__ int64_t wave_sum64(int64_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    return v;
}

__device__ __forceinline__ uint32_t wave_or(uint32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v |= (uint32_t)__shfl_xor((int)v, o, kWave);
    return v;
}

using diso_launch::stripe_blocks;
using diso_launch::xcd_block;
using diso_launch::xcd_stripe;

// The block's number in a launch of diso_launch::shape_of.
__device__ __forceinline__ int64_t block_number() { return (int64_t)blockIdx.y * gridDim.x + blockIdx.x; }

struct SegBase {
    int64_t v;  // first vertex (MC) / first quad (DMC) of the segment
    int64_t f;  // first triangle (MC) / first DMC vertex (patch) of the segment
};

// Segment (px, py, chunk) is (px * g1 + py) * nchunk + chunk, so the ids step by nchunk from row
// (px, py) to (px, py + 1) and by xstride(g) to (px + 1, py): neighbour rows' segments come from
// additions, not products.
__device__ __forceinline__ int64_t xstride(const Geo &g) { return (int64_t)g.g1 * g.nchunk; }

// Classification of a grid's positions, one bit per position of a segment in 64-bit planes (bit l =
// lane l), written by the count pass after the segment bases and read by the later passes instead
// of the samples:
//   inside  the position's own sample is >= iso (pad samples included);
//   X, Y, Z the edge owned along that axis crosses the surface;
//   A       the cell anchored here is cut by the surface (active);
//   m0, m1  DMC: the cell's patch count minus one, in binary (0 unless active);
//   codes   per position, the code of the active cell anchored there (MC: Bourke corner order; DMC:
//           Morton corner order after the face-neighbour rule). Written only in segments that hold
//           an active cell, and only meaningful at active positions.
// Where no cell is anchored, X, Y, Z and A are 0.
//
// The active cells, in the grid's linear order, are dealt to the emission's waves in units of 64:
//   abase   active cells before the segment's first position, modulo 2^16;
//   unit    unit u's first cell (number 64 u) lies in segment unit[u];
//   nunits  the number of units (only where a grid can hold a cell: at least four segments).
struct Plane2 {
    uint64_t a, b;
};

struct Planes {
    Plane2 *xy, *za, *m;  // (X, Y), (Z, A), (m0, m1; DMC only), one entry per segment
    uint8_t *codes;       // 64 per segment
    uint64_t *inside;
    uint32_t *unit;
    uint32_t *nunits;
    uint8_t *flags;       // DISO_TOTAL_* flags of the samples of a run of segments, at its first
    uint16_t *abase;
};
constexpr int64_t kSegStateBytes = 128;  // per segment: 48 + 64 + 8 + 4 + 1 + 1 + 2

// The planes behind the bases of `n` segments (seg[n], seg[n + 1] are the totals).
__host__ __device__ inline Planes planes_at(void *after, int64_t n) {
    uint8_t *b = static_cast<uint8_t *>(after);
    Planes q;
    q.xy = reinterpret_cast<Plane2 *>(b);
    q.za = q.xy + n;
    q.m = q.za + n;
    q.codes = b + n * 48;
    q.inside = reinterpret_cast<uint64_t *>(b + n * 112);
    q.unit = reinterpret_cast<uint32_t *>(b + n * 120);
    q.nunits = reinterpret_cast<uint32_t *>(b + n * 124);
    q.flags = b + n * 125;
    q.abase = reinterpret_cast<uint16_t *>(b + n * 126);
    return q;
}
__host__ __device__ inline Planes planes_of(const SegBase *seg, int64_t nseg) {
    return planes_at(const_cast<SegBase *>(seg + nseg + 2), nseg);
}

// A grid's segments as the emission and backward passes see them: its bases (seg[s], s from 0;
// seg[nseg] is the base after its last segment), its classification planes, and the base values
// of its first segment (v0, f0), which are subtracted to index its own outputs. A grid extracted
// alone has v0 = f0 = 0; in a batch the scan runs over all grids' segments in order.
struct SegCtx {
    const SegBase *__restrict__ seg;
    const Plane2 *__restrict__ xy, *__restrict__ za;
    int64_t v0, f0;
};
__device__ __forceinline__ SegCtx seg_ctx(const SegBase *seg, const Planes &q) { return SegCtx{seg, q.xy, q.za, 0, 0}; }

// ------------------------------------------------------------------------------------------
// Edge geometry shared by the emission and backward kernels

// A segment's row (px, py) and chunk. The quotients come from double reciprocals: (n + 1/2) / d is at
// least 1 / (2 d) away from an integer, and for n < 2^32 the product is off by less than 2^-20 (and
// by less than 2^-40 where d is large enough for that to matter), so its integer part is n / d.
// Three instructions where an integer division takes about twenty.
struct SegPos {
    int px, py, chunk;
};
__device__ __forceinline__ uint32_t div_rcp(uint32_t n, double r) { return (uint32_t)(((double)n + 0.5) * r); }
__device__ __forceinline__ SegPos seg_pos(const Geo &g, int64_t s) {
    const uint32_t su = (uint32_t)s, row = div_rcp(su, g.rchunk), px = div_rcp(row, g.rg1);
    return SegPos{(int)px, (int)(row - px * (uint32_t)g.g1), (int)(su - row * (uint32_t)g.nchunk)};
}

// The position of segment lo + i, read from lane i of a lane-parallel seg_pos (i uniform).
__device__ __forceinline__ SegPos pos_of_lane(const SegPos &lp, int i) {
    return SegPos{__builtin_amdgcn_readlane(lp.px, i), __builtin_amdgcn_readlane(lp.py, i),
                  __builtin_amdgcn_readlane(lp.chunk, i)};
}

// A wave-uniform struct read from memory, kept in scalar registers.
template <typename T>
__device__ __forceinline__ T load_uniform(const T *p) {
    static_assert(sizeof(T) % 4 == 0, "dword-sized");
    int w[sizeof(T) / 4];
    __builtin_memcpy(w, p, sizeof(T));
#pragma unroll
    for (int i = 0; i < (int)(sizeof(T) / 4); ++i) w[i] = __builtin_amdgcn_readfirstlane(w[i]);
    T r;
    __builtin_memcpy(&r, w, sizeof(T));
    return r;
}

// Wave index within the block, as a scalar (wave-uniform) value.
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x / kWave); }

// Edge e of a cell (src/cumc.cu:109-122): starts at cell-relative corner (eox, eoy, eoz) and
// runs along axis eax. Bit masks of the edge table, so unrolled loops fold them to constants.
__device__ constexpr int eox(int e) { return (0x622 >> e) & 1; }
__device__ constexpr int eoy(int e) { return (0x0F0 >> e) & 1; }
__device__ constexpr int eoz(int e) { return (0xC44 >> e) & 1; }
__device__ constexpr int eax(int e) { return e >= 8 ? 1 : ((e & 1) ? 2 : 0); }

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename S>
__device__ __forceinline__ V3<S> add3(V3<S> a, V3<S> b) {
    return {a.x + b.x, a.y + b.y, a.z + b.z};
}

// computeMcVert from samples and deforms already in registers: p0 + (p1 - p0) * t with
// p = integer position + deform (src/cumc.cu:343-368).
template <typename S, bool DEF>
__device__ __forceinline__ V3<S> lerp_vertex(int x, int y, int z, int axis, S d0, S d1, V3<S> f0, V3<S> f1,
                                             S iso) {
    const S t = interp_t(d0, d1, iso);
    S p0x = S(x), p0y = S(y), p0z = S(z);
    S p1x = S(x + (axis == 0)), p1y = S(y + (axis == 1)), p1z = S(z + (axis == 2));
    if (DEF) {
        p0x += f0.x;
        p0y += f0.y;
        p0z += f0.z;
        p1x += f1.x;
        p1y += f1.y;
        p1z += f1.z;
    }
    V3<S> r;
    r.x = p0x + (p1x - p0x) * t;
    r.y = p0y + (p1y - p0y) * t;
    r.z = p0z + (p1z - p0z) * t;
    return r;
}

// Samples and deforms of both endpoints of the edge from (x,y,z) along `axis`, the pad value and a
// zero deform where an endpoint is not stored: the second endpoint's index is the first's plus the axis stride (one
// index product per edge instead of two).
template <typename S, bool DEF>
struct EdgeEnds {
    S d0, d1;
    V3<S> f0, f1;
};
template <typename S, bool DEF>
__device__ __forceinline__ EdgeEnds<S, DEF> edge_ends(const In<S> &in, int x, int y, int z, int axis) {
    const Geo &g = in.geo;
    const bool ok0 = in_data(in, x, y, z), ok1 = in_data(in, x + (axis == 0), y + (axis == 1), z + (axis == 2));
    const int64_t i0 = data_index(in, x, y, z);
    const int64_t i1 = i0 + (axis == 0 ? (int64_t)g.n1 * g.n2 : (axis == 1 ? (int64_t)g.n2 : 1));
    const int64_t j0 = ok0 ? i0 : 0, j1 = ok1 ? i1 : 0;
    EdgeEnds<S, DEF> e;
    const S a = in.sdf[j0], b = in.sdf[j1];
    e.d0 = ok0 ? a : in.pad;
    e.d1 = ok1 ? b : in.pad;
    e.f0 = e.f1 = V3<S>{S(0), S(0), S(0)};
    if (DEF) {
        const S *p0 = in.deform + 3 * j0, *p1 = in.deform + 3 * j1;
        const S u0 = p0[0], u1 = p0[1], u2 = p0[2], w0 = p1[0], w1 = p1[1], w2 = p1[2];
        e.f0 = V3<S>{ok0 ? u0 : S(0), ok0 ? u1 : S(0), ok0 ? u2 : S(0)};
        e.f1 = V3<S>{ok1 ? w0 : S(0), ok1 ? w1 : S(0), ok1 ? w2 : S(0)};
    }
    return e;
}

// MC vertex on the edge from (x,y,z) along `axis`: samples and deforms of both endpoints.
template <typename S, bool DEF>
__device__ __forceinline__ V3<S> edge_vertex(const In<S> &in, int x, int y, int z, int axis) {
    const EdgeEnds<S, DEF> e = edge_ends<S, DEF>(in, x, y, z, axis);
    return lerp_vertex<S, DEF>(x, y, z, axis, e.d0, e.d1, e.f0, e.f1, in.iso);
}

// x / c for a divisor c fixed per call, with r = RN(1/c): q = x*r is within an ulp of x/c and
// one FMA correction with the exact residual makes it the correctly rounded quotient
// (Markstein's theorem), i.e. bit-identical to IEEE x / c, in 3 instructions instead of the
// ~10 of a general correctly rounded division.
template <typename S>
__device__ __forceinline__ S div_by(S x, S c, S r) {
    if (c == S(0)) return x / c;  // uniform; keeps IEEE inf/nan for a length-1 axis
    const S q = x * r;
    return fma(fma(-q, c, x), r, q);
}

// Per-axis divisors (dims - 1) and their reciprocals, for the wrapper's normalisation.
template <typename S>
struct Norm {
    S c[3], r[3];
};

// ------------------------------------------------------------------------------------------
// Batch descriptors (every pass of a batch reads them)

template <typename S>
struct BatchGrid {
    In<S> in;
    Norm<S> nm;
    int algo, flags;
    int64_t seg_first;  // first segment in the batch's segment space
    int64_t nv, nf;     // vertex and face rows (from the count pass)
    S *verts;
    void *faces;
    uint8_t *vinfo;
    int64_t vcap, fcap;
    const S *adj;  // upstream vertex gradients [nv, 3]
    S *adj_sdf, *adj_deform;
    int64_t q_first;  // DMC: first row of its per-edge gradients in the batch scratch
    int tile;           // segments per gathering wave (bwd_tile_of the grid's size bucket)
};

// j such that rf[j] <= b < rf[j + 1] (rf ascending, rf[0] = 0, rf[m] = total).
__device__ __forceinline__ int find_group(const int64_t *__restrict__ rf, int m, int64_t b) {
    int lo = 0, hi = m;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (rf[mid] <= b)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// ------------------------------------------------------------------------------------------
// Pass 1: classify, count, scan
//
// mask_kernel streams the samples once and keeps one bit per position: whether the sample is >=
// iso. count_kernel then works on those bits, one lane per segment (diso_bits.h), and scans the
// segment counts in the same launch.
//
// The scan (single pass). The segments are split into G contiguous ranges, one per block. A block
// counts its segments (writing each segment's planes, and keeping its counts), publishes its
// aggregate as two 64-bit words, each with the call's tag, so that a reader takes them only when both
// are this call's, reads the aggregates of all its predecessors in parallel (a look-back over the whole
// window at once: no chain of inclusive prefixes, so the wait is one memory latency rather than one per
// predecessor), and finally scans its own segment counts into segment bases. Aggregate words are accessed with agent-scope
// atomics only, so they are coherent across the XCDs' L2s without fences. Two word buffers
// alternate between calls; each call clears the one the next call uses (up to the extent that
// was written), and the last block advances the epoch once every block has published (and so has
// read the epoch), so no initialisation launch is needed. Words are tagged with their call's
// epoch (diso_scan_word.h: tag, sample flags, face / patch count, vertex / quad count), so a word
// that a block of an earlier call wrote late never counts for a later call, and no reset is
// needed after a timeout. A predecessor that does not publish in time (it may not be running:
// other launches can fill the slots of the XCD it was dispatched to) is counted by the waiting
// block itself; only the last block waits for all, and every block it waits for ends in bounded
// time once dispatched.

struct CtlHeader {
    uint32_t epoch;     // calls completed on this block (diso_scan_word.h)
    uint32_t dirty[2];  // words written in each buffer since it was last cleared
    uint32_t nan;       // set by mask_kernel when it meets a NaN, cleared by the count's last block
    uint32_t pad[12];
};

// Where a waiting host reads a count's totals: in host memory that the device writes, `seq` last.
struct HostTotals {
    int64_t v, f, flags;
    uint64_t seq;
};

constexpr int kCountWaves = 8;
constexpr int kCountBlock = kCountWaves * kWave;
constexpr int64_t kMaxCountBlocks = 4096;  // two words each
constexpr int kCountBlocksPerCU = 4;
constexpr int64_t kCountLds = 6144;  // segments of a block whose counts stay in LDS (24 KiB)

__device__ __forceinline__ uint64_t ld_relaxed(const uint64_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_relaxed(uint64_t *p, uint64_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// What a count launch classifies: one grid (`in`, algorithm ALGO), or (BATCH) the concatenated
// segments of several grids, each with its own descriptor; then per-grid sample flags are
// or-ed into gflags[grid] (zero on entry) and the scan runs over all segments in order.

template <typename S>
struct CountSrc {
    In<S> in;
    uint32_t *gflags;
    int ngrids;
    uint32_t recount_spins;  // reads of an unpublished predecessor word before counting its range
    int64_t nseg;            // segments of the launch
};

// The grid that segment s of a batch belongs to.
template <typename S>
__device__ __forceinline__ int batch_grid_of(const BatchGrid<S> *__restrict__ grids, int n, int64_t s) {
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (grids[mid].seg_first <= s)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

__device__ __forceinline__ int64_t readlane64(int64_t v, int i) {
    return (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), i) << 32) |
                     (uint32_t)__builtin_amdgcn_readlane((int)v, i));
}

// Inside planes and sample flags of the segments [lo, lo + n) (n <= kMaskTile) of one grid, whose
// first segment is segment `first` of the launch. Stored samples are read in words of 64 from the
// row's first (chunk c's word: samples 64 c .. 64 c + 63), kMaskLoads samples per lane in flight;
// each compare's lane mask is the word's bits, kept in lane i + 1 for segment lo + i and in lane 0
// for the chunk before the tile's first segment. With the virtual pad a segment's plane is its word
// moved up by the pad sample, the bit below it from the previous chunk's word; so a last chunk that
// holds only pad and the last sample needs no load of its own.
// Small grids, whose tiles do not fill the SIMDs, take shorter ones, read in one round of loads: MC count
// of 16^3, 32^3, 48^3, 64^3, 96^3 noisy (both kernels) 11.5, 12.7, 14.4, 13.1, 16.0 us with 32 segments a
// tile, 10.4, 11.6, 12.1, 13.2, 14.3 with 12 (13.2 at 48^3 with 16: with the chunk before, 17 words).
constexpr int kMaskTile = 32, kMaskSmallTile = 12;
constexpr int kMaskLoads = 16;
template <typename S>
__device__ __forceinline__ void mask_tile(const In<S> &in, int64_t first, int64_t lo, int n, const Planes &out,
                                          uint32_t *nan, int lane) {
    const Geo &g = in.geo;
    const int64_t sg = lo - first + lane - 1;  // segment of this lane's word
    const SegPos sp = seg_pos(g, sg >= 0 ? sg : 0);
    const int x = sp.px - g.off, y = sp.py - g.off, z0 = sp.chunk * kWave;
    const bool row = (unsigned)x < (unsigned)g.n0 && (unsigned)y < (unsigned)g.n1;
    const int64_t ro = row ? ((int64_t)x * g.n1 + y) * g.n2 + z0 : 0;
    uint64_t todo = __ballot(row && z0 < g.n2 && sg >= 0 && lane <= n);
    uint32_t ilo = 0, ihi = 0, elo = 0, ehi = 0;
    while (todo) {  // wave-uniform
        S v[kMaskLoads];
        int at[kMaskLoads];
#pragma unroll
        for (int j = 0; j < kMaskLoads; ++j) {
            // (past the last word to do: that word again)
            at[j] = todo ? (int)__builtin_ctzll(todo) : at[j ? j - 1 : 0];
            todo &= todo - 1;
            const int left = g.n2 - 1 - __builtin_amdgcn_readlane(z0, at[j]);  // samples past the row: the last one
            v[j] = in.sdf[readlane64(ro, at[j]) + (lane < left ? lane : left)];
        }
#pragma unroll
        for (int j = 0; j < kMaskLoads; ++j) {
            const uint64_t inside = __ballot(v[j] >= in.iso);
            const uint64_t equal = __ballot(!(v[j] < in.iso || v[j] > in.iso));  // == iso, or NaN
            const bool mine = lane == at[j];
            ilo = mine ? (uint32_t)inside : ilo;
            ihi = mine ? (uint32_t)(inside >> 32) : ihi;
            elo = mine ? (uint32_t)equal : elo;
            ehi = mine ? (uint32_t)(equal >> 32) : ehi;
        }
    }
    const uint64_t have = row ? diso_bits::low_bits(g.n2 - z0) : 0ull;  // the word's stored samples
    const uint64_t I = ((uint64_t)ihi << 32 | ilo) & have, E = (uint64_t)ehi << 32 | elo;
    // flags of the tile's own words; a chunk beyond the stored samples has none
    const uint64_t own = lane >= 1 && lane <= n ? have : 0ull;
    uint32_t fl = ((~I & ~E & own) ? DISO_TOTAL_HAS_BELOW : 0u) | ((I & ~E & own) ? DISO_TOTAL_HAS_ABOVE : 0u) |
                  ((~I & E & own) ? DISO_TOTAL_HAS_NAN : 0u);
    if (in.iso != in.iso) {  // every compare fails: no sample is below or above, and E says nothing of NaN
        fl = 0u;
        const int end = own ? g.n2 - z0 : 0;
#pragma unroll 1
        for (int l = 0; l < kWave && l < end; ++l) {
            const S v = in.sdf[ro + l];
            fl |= v != v ? DISO_TOTAL_HAS_NAN : 0u;
        }
    }
    fl = wave_or(fl);
    if ((fl & DISO_TOTAL_HAS_NAN) && lane == 0) __hip_atomic_store(nan, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // the previous lane's top bit (its chunk precedes this one, unless this is the row's first)
    const uint32_t before = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(I >> 32), 0x138, 0xf, 0xf, false) >> 31;
    const uint64_t grid = diso_bits::low_bits(g.g2 - z0);
    uint64_t plane = I, stored = have;
    if (g.off) {  // uniform
        plane = (I << 1) | (sp.chunk > 0 ? (uint64_t)before : 0ull);
        stored = row ? diso_bits::low_bits(g.n2 + 1 - z0) & (sp.chunk > 0 ? ~0ull : ~1ull) : 0ull;
    }
    if (in.pad >= in.iso) plane |= grid & ~stored;
    if (lane >= 1 && lane <= n) {
        out.inside[lo + lane - 1] = plane;
        out.flags[lo + lane - 1] = lane == 1 ? (uint8_t)fl : (uint8_t)0;
    }
}

template <typename S, bool BATCH>
__global__ __launch_bounds__(kBlock) void mask_kernel(CountSrc<S> src, const BatchGrid<S> *__restrict__ grids,
                                                      Planes out, uint8_t *ctl, int tile) {
    const int lane = threadIdx.x % kWave;
    const int64_t lo = (block_number() * kWavesPerBlock + wave_id()) * tile;
    const int64_t hi = lo + tile < src.nseg ? lo + tile : src.nseg;
    uint32_t *nan = &reinterpret_cast<CtlHeader *>(ctl)->nan;
    if (lo >= hi) return;
    if constexpr (!BATCH) {
        mask_tile<S>(src.in, 0, lo, (int)(hi - lo), out, nan, lane);
    } else {
        int gi = batch_grid_of(grids, src.ngrids, lo);
        for (int64_t s = lo; s < hi; ++gi) {  // the tile may span several grids
            const In<S> in = load_uniform(&grids[gi].in);
            const int64_t first = grids[gi].seg_first;
            const int64_t end = first + in.geo.nseg < hi ? first + in.geo.nseg : hi;
            mask_tile<S>(in, first, s, (int)(end - s), out, nan, lane);
            s = end;
        }
    }
}

// An edge with a NaN end does not cross: takes such edges out of a segment's crossings (from the
// samples; only called when the launch holds a NaN). Each lane goes through its own segment's positions
// with a crossing; through all 64 in turn, a NaN cost a 256^3 count 230 us more on any surface.
template <typename S>
__device__ __forceinline__ void drop_nan_edges(const In<S> &in, const SegPos &sp, uint64_t &X, uint64_t &Y, uint64_t &Z) {
#pragma unroll 1
    for (uint64_t todo = X | Y | Z; todo; todo &= todo - 1) {
        const int l = (int)__builtin_ctzll(todo), z = sp.chunk * kWave + l;
        const S a = sample(in, sp.px, sp.py, z), x = sample(in, sp.px + 1, sp.py, z), y = sample(in, sp.px, sp.py + 1, z),
                u = sample(in, sp.px, sp.py, z + 1);
        X &= ~((uint64_t)(a != a || x != x) << l);
        Y &= ~((uint64_t)(a != a || y != y) << l);
        Z &= ~((uint64_t)(a != a || u != u) << l);
    }
}

// Counts the segments [lo, hi) of one grid whose first segment is segment `first` of the launch, one
// lane per segment, tiles of 64 segments dealt to the block's waves (the first to wave `turn`); adds
// each lane's totals to (wv, wf) and its sample flags to fl. WRITE: also records each segment's
// planes, codes and counts; without WRITE the range is only summed (a block recounting a
// predecessor's range, see the look-back).
template <typename S, bool DMC, bool WRITE>
__device__ __forceinline__ void count_tiles(const In<S> &in, int64_t first, int64_t lo, int64_t hi, int wave, int lane,
                                            bool has_nan, const Planes &P, SegBase *seg, int64_t &wv, int64_t &wf,
                                            int64_t &wa, uint32_t &fl, uint32_t *s_cnt, int64_t block_lo) {
    const Geo &g = in.geo;
    const int64_t sx = xstride(g), sy = g.nchunk;
    for (int64_t base = lo + (int64_t)wave * kWave; base < hi; base += kCountBlock) {  // wave-uniform
        const int64_t s = base + lane;
        const bool valid = s < hi;
        const int64_t sv = valid ? s : hi - 1;
        const SegPos sp = seg_pos(g, sv - first);
        const diso_bits::Place pl{sp.px, sp.py, sp.chunk, g.g0, g.g1, g.g2, g.nchunk};
        const uint64_t *ip = P.inside + sv;
        uint64_t X = 0, Y = 0, Z = 0, A = 0, m0 = 0, m1 = 0;
        int nf = 0;
        diso_bits::classify<DMC>(
            pl, valid, [&](int dx, int dy, int dc) { return ip[dx * sx + dy * sy + dc]; },
            [&](uint32_t b) { return __any(b != 0) != 0; },
            [&](int h, const diso_bits::Classified &c) {
                X |= (uint64_t)c.X << (32 * h);
                Y |= (uint64_t)c.Y << (32 * h);
                Z |= (uint64_t)c.Z << (32 * h);
                A |= (uint64_t)c.A << (32 * h);
                m0 |= (uint64_t)c.m0 << (32 * h);
                m1 |= (uint64_t)c.m1 << (32 * h);
                nf += c.nf;
                if constexpr (WRITE) {
                    if (c.A) {
                        uint32_t w[8];
                        diso_bits::codes_of(c.code, w);
                        uint4 *d = reinterpret_cast<uint4 *>(P.codes + s * kWave + 32 * h);
                        d[0] = uint4{w[0], w[1], w[2], w[3]};
                        d[1] = uint4{w[4], w[5], w[6], w[7]};
                    }
                }
            });
        if (has_nan) drop_nan_edges(in, sp, X, Y, Z);  // uniform
        const int nv = diso_bits::popc64(X) + diso_bits::popc64(Y) + diso_bits::popc64(Z), na = diso_bits::popc64(A);
        wv += nv;
        wf += nf;
        wa += na;
        if (valid) fl |= P.flags[s];
        if constexpr (WRITE) {
            if (valid) {
                // counts of at most 192, 320 and 64, for the segment bases
                const uint32_t cnt = (uint32_t)nv | (uint32_t)nf << 8 | (uint32_t)na << 24;
                if (s_cnt)
                    s_cnt[s - block_lo] = cnt;
                else
                    seg[s].v = (int64_t)cnt;
                P.xy[s] = Plane2{X, Y};
                P.za[s] = Plane2{Z, A};
                if (DMC) P.m[s] = Plane2{m0, m1};
            }
        }
    }
}

// count_tiles over the segments [lo, hi) of the launch.
template <typename S, int ALGO, bool BATCH, bool WRITE>
__device__ __forceinline__ void count_range(const CountSrc<S> &src, const BatchGrid<S> *__restrict__ grids,
                                            SegBase *seg, const Planes &P, bool has_nan, int64_t lo, int64_t hi,
                                            int wave, int lane, int64_t &wv, int64_t &wf, int64_t &wa,
                                            uint32_t &wfl, uint32_t *s_cnt, int64_t block_lo) {
    if constexpr (!BATCH) {
        count_tiles<S, ALGO == DISO_DMC, WRITE>(src.in, 0, lo, hi, wave, lane, has_nan, P, seg, wv, wf, wa, wfl,
                                             s_cnt, block_lo);
    } else {
        // the range may span several grids: one pass per grid, its parameters in scalar registers
        int gi = batch_grid_of(grids, src.ngrids, lo);
        for (int64_t s = lo; s < hi; ++gi) {  // block-uniform
            const In<S> in = load_uniform(&grids[gi].in);
            const int64_t first = grids[gi].seg_first;
            const int64_t end = first + in.geo.nseg < hi ? first + in.geo.nseg : hi;
            uint32_t gfl = 0;
            if (grids[gi].algo == DISO_MC)
                count_tiles<S, false, WRITE>(in, first, s, end, wave, lane, has_nan, P, seg, wv, wf, wa, gfl, s_cnt, block_lo);
            else
                count_tiles<S, true, WRITE>(in, first, s, end, wave, lane, has_nan, P, seg, wv, wf, wa, gfl, s_cnt, block_lo);
            wfl |= gfl;
            if constexpr (WRITE) {
                gfl = wave_or(gfl);
                if (lane == 0 && gfl) atomicOr(src.gflags + gi, gfl);
            }
            s = end;
        }
    }
}

template <typename S, int ALGO, bool BATCH>
__global__ __launch_bounds__(kCountBlock, kCountWaves / 2) void count_kernel(CountSrc<S> src,
                                                                           const BatchGrid<S> *__restrict__ grids,
                                                                           SegBase *seg, Planes planes, uint8_t *ctl,
                                                                           int64_t nblocks, HostTotals *host,
                                                                           uint64_t seq) {
    __shared__ int64_t s_v[kCountWaves], s_f[kCountWaves], s_a[kCountWaves];
    __shared__ uint32_t s_fl[kCountWaves];
    __shared__ uint32_t s_epoch, s_dirty_other, s_next;
    __shared__ uint64_t s_word, s_word2;
    __shared__ uint32_t s_cnt[kCountLds];
    __shared__ uint64_t s_sum[2][kCountWaves];

    CtlHeader *hdr = reinterpret_cast<CtlHeader *>(ctl);
    uint64_t *words = reinterpret_cast<uint64_t *>(ctl + kCtlHeader);
    const int tid = threadIdx.x, wave = wave_id(), lane = tid % kWave;
    const int64_t nseg = src.nseg;
    const int64_t b = blockIdx.x;
    const int64_t lo = b * nseg / nblocks, hi = (b + 1) * nseg / nblocks;

    if (tid == 0) {
        const uint32_t ep = __hip_atomic_load(&hdr->epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_epoch = ep;
        s_dirty_other = __hip_atomic_load(&hdr->dirty[diso_scan::buffer_of(ep) ^ 1u], __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT);
    }
    const bool has_nan = __builtin_amdgcn_readfirstlane(
                             (int)__hip_atomic_load(&hdr->nan, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0;

    // The block's sums of one set of per-lane counts, in every thread. Two barriers.
    auto block_sums = [&](int64_t &v, int64_t &f, int64_t &a, uint32_t &fl) {
        v = wave_sum64(v);
        f = wave_sum64(f);
        a = wave_sum64(a);
        fl = wave_or(fl);
        __syncthreads();  // s_v / s_f / s_a reuse
        if (lane == 0) {
            s_v[wave] = v;
            s_f[wave] = f;
            s_a[wave] = a;
            s_fl[wave] = fl;
        }
        __syncthreads();
        v = f = a = 0;
        fl = 0;
#pragma unroll
        for (int w = 0; w < kCountWaves; ++w) {
            v += s_v[w];
            f += s_f[w];
            a += s_a[w];
            fl |= s_fl[w];
        }
    };

    // 1. Count: the block's segments, one lane each; the counts of up to kCountLds segments stay in
    // LDS (more: in `seg`) for phase 4.
    const bool in_lds = hi - lo <= kCountLds;
    int64_t av = 0, af = 0, aa = 0;
    uint32_t afl = 0;
    count_range<S, ALGO, BATCH, true>(src, grids, seg, planes, has_nan, lo, hi, wave, lane, av, af, aa, afl,
                                          in_lds ? s_cnt : nullptr, lo);
    block_sums(av, af, aa, afl);  // (its barriers also make the header reads visible)
    const uint32_t epoch = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_epoch);
    const uint32_t parity = diso_scan::buffer_of(epoch), tag = diso_scan::tag_of(epoch);
    // block j's two words: words 2 j (vertices, faces, flags) and 2 j + 1 (active cells)
    uint64_t *cur = words + (int64_t)parity * 2 * kMaxCountBlocks;
    if (tid == 0) {
        st_relaxed(cur + 2 * b, diso_scan::pack(av, af, afl, tag));
        st_relaxed(cur + 2 * b + 1, diso_scan::pack_cells(aa, tag));
    }

    // 2. Exclusive prefix of this block = sum of all predecessors' aggregates. A predecessor that
    // has not published within `recount_spins` reads is not waited for any longer: this block
    // counts that range itself (read-only; the same sums), so no block waits on one that may not
    // be running (several launches sharing the device fill the XCDs' slots). The last block alone
    // waits for every predecessor's words: a block publishes after reading the epoch, so once all
    // have published the last block may advance it; every other block ends in bounded time, so the
    // blocks it waits for are all dispatched.
    const bool last = b == nblocks - 1;
    const uint32_t spin_limit = last ? kSpinLimit / (uint32_t)(kMaxCountBlocks / kCountBlock) : src.recount_spins;
    int64_t ev = 0, ef = 0, ea = 0;
    uint32_t efl = 0;
    uint32_t miss = 0;  // bit k: predecessor tid + k * kCountBlock did not publish in time
    for (int64_t j = tid, k = 0; j < b; j += kCountBlock, ++k) {
        uint64_t w, w2;
        uint32_t spins = 0;
        do {
            w = ld_relaxed(cur + 2 * j);
            w2 = ld_relaxed(cur + 2 * j + 1);
        } while (!(diso_scan::published(w, tag) && diso_scan::published(w2, tag)) && ++spins < spin_limit);
        if (!(diso_scan::published(w, tag) && diso_scan::published(w2, tag))) {
            miss |= 1u << k;
        } else {
            ev += diso_scan::count_v(w);
            ef += diso_scan::count_f(w);
            ea += diso_scan::count_cells(w2);
            efl |= diso_scan::flags_of(w);
        }
    }
    block_sums(ev, ef, ea, efl);
    // the missing predecessors, lowest first, one at a time by the whole block
    for (;;) {
        if (tid == 0) s_next = 0xffffffffu;
        __syncthreads();
        if (miss) atomicMin(&s_next, (uint32_t)(tid + __builtin_ctz(miss) * kCountBlock));  // LDS
        __syncthreads();
        const uint32_t j = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_next);
        if (j == 0xffffffffu) break;  // block-uniform
        if (last) efl |= DISO_TOTAL_SCAN_TIMEOUT;  // never expected: the epoch may advance early
        if (tid == (int)(j % kCountBlock)) {  // one read for the whole block: every wave takes the same branch
            miss &= ~(1u << (j / kCountBlock));
            s_word = ld_relaxed(cur + 2 * (int64_t)j);
            s_word2 = ld_relaxed(cur + 2 * (int64_t)j + 1);
        }
        __syncthreads();
        const uint64_t w = s_word, w2 = s_word2;
        int64_t rv = 0, rf = 0, ra = 0;
        uint32_t rfl = 0;
        if (__builtin_amdgcn_readfirstlane((int)(diso_scan::published(w, tag) && diso_scan::published(w2, tag)))) {
            if (tid == 0) {  // published meanwhile; counted once
                rv = diso_scan::count_v(w);
                rf = diso_scan::count_f(w);
                ra = diso_scan::count_cells(w2);
                rfl = diso_scan::flags_of(w);
            }
        } else {
            count_range<S, ALGO, BATCH, false>(src, grids, seg, planes, has_nan, (int64_t)j * nseg / nblocks,
                                               ((int64_t)j + 1) * nseg / nblocks, wave, lane, rv, rf, ra, rfl, nullptr, 0);
        }
        block_sums(rv, rf, ra, rfl);
        ev += rv;
        ef += rf;
        ea += ra;
        efl |= rfl;
    }
    if (last && tid == 0) {
        SegBase *tot = seg + nseg;
        tot[0].v = ev + av;
        tot[0].f = ef + af;
        tot[1].v = (int64_t)(efl | afl);
        tot[1].f = ALGO;
        if (host) {  // a host thread waits for `seq` (diso_extract)
            auto put_host = [](auto *p, auto v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); };
            put_host(&host->v, ev + av);
            put_host(&host->f, ef + af);
            put_host(&host->flags, (int64_t)(efl | afl));
            __hip_atomic_store(&host->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        if (nseg >= 4) *planes.nunits = (uint32_t)((ea + aa + kWave - 1) / kWave);
        __hip_atomic_store(&hdr->dirty[parity], (uint32_t)(2 * nblocks), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&hdr->dirty[parity ^ 1u], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&hdr->nan, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&hdr->epoch, epoch + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // 3. Clear this block's share of the other word buffer for the next call.
    {
        const int64_t n = (int64_t)__builtin_amdgcn_readfirstlane((int)s_dirty_other);
        const int64_t per = (n + nblocks - 1) / nblocks;
        const int64_t c0 = b * per, c1 = c0 + per < n ? c0 + per : n;
        uint64_t *other = words + (int64_t)(parity ^ 1u) * 2 * kMaxCountBlocks;
        for (int64_t i = c0 + tid; i < c1; i += kCountBlock) st_relaxed(other + i, 0ull);
    }

    // 4. Segment bases: exclusive scan of the block's segment counts, 512 segments at a time. A wave's
    // sums fit 16-bit fields (64 segments: at most 12,288 vertices, 20,480 faces, 4,096 cells).
    __syncthreads();  // s_v / s_f / s_a reuse; phase-1 counts complete
    for (int64_t base = lo; base < hi; base += kCountBlock) {
        const int64_t s = base + tid;
        uint32_t c = 0;
        if (s < hi)
            c = in_lds ? s_cnt[s - lo]
                       : (uint32_t)__hip_atomic_load(reinterpret_cast<uint64_t *>(&seg[s].v), __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t cvf = (c & 0xff) | ((c >> 8) & 0xffff) << 16, ca = c >> 24;
        const uint32_t ivf = wave_incl_dpp(cvf), ia = wave_incl_dpp(ca);
        const int par = (int)((base - lo) / kCountBlock) & 1;  // two sets of sums: one barrier a round
        if (lane == kWave - 1) s_sum[par][wave] = (uint64_t)ivf | (uint64_t)ia << 32;
        __syncthreads();
        int64_t ov = ev, of = ef, oa = ea;
#pragma unroll
        for (int w = 0; w < kCountWaves; ++w) {
            const uint64_t t = s_sum[par][w];
            const int64_t tv = (int64_t)(t & 0xffff), tf = (int64_t)((t >> 16) & 0xffff), ta = (int64_t)(t >> 32);
            if (w < wave) {
                ov += tv;
                of += tf;
                oa += ta;
            }
            ev += tv;
            ef += tf;
            ea += ta;
        }
        if (s < hi) {
            seg[s].v = ov + (int64_t)((ivf & 0xffff) - (cvf & 0xffff));
            seg[s].f = of + (int64_t)((ivf >> 16) - (cvf >> 16));
            const int64_t a0 = oa + (int64_t)(ia - ca);
            planes.abase[s] = (uint16_t)a0;
            const int64_t u = (a0 + kWave - 1) / kWave;  // the unit, if any, that starts in this segment
            if (u * kWave < a0 + (int64_t)ca) planes.unit[u] = (uint32_t)s;
        }
    }
}

// ------------------------------------------------------------------------------------------
// Pass 2: emission
//
// Work compaction, twice. A wave takes units of 64 active cells, wherever they lie: 256^3 noisy, MC /
// DMC 156 / 289 us with a wave per segment, 124 / 163 so; 384^3 smooth 217 and 63. And each lane
// publishes its cell's items (MC vertices and triangles; DMC edge vertices, patch vertices and
// quads) into a dense per-wave list in LDS at its in-wave prefix, which the wave then processes 64
// items at a time. Every item is computed exactly once, and item k is the unit's k-th output row, so
// consecutive lanes write consecutive rows (coalesced stores). MC is bound by the latency between a
// unit's dependent loads (vector instructions take two fifths of the issue slots).

// Largest run length: the segments that four gathering waves take (bwd_tile_of), a launch parameter
// (diso_set_param).
constexpr int kMaxRun = kWave;

struct OutCfg {
    int flags;
    int64_t vcap, fcap;  // capacities in rows
};

template <typename S>
__device__ __forceinline__ V3<S> epilogue(V3<S> p, int flags, const Norm<S> &nm) {
    if (flags & DISO_FLAG_SHIFT) {  // verts - 1 (diso/__init__.py:56)
        p.x = p.x - S(1);
        p.y = p.y - S(1);
        p.z = p.z - S(1);
    }
    if (flags & DISO_FLAG_NORMALIZE) {  // verts / (dims - 1) (diso/__init__.py:57-60)
        p.x = div_by(p.x, nm.c[0], nm.r[0]);
        p.y = div_by(p.y, nm.c[1], nm.r[1]);
        p.z = div_by(p.z, nm.c[2], nm.r[2]);
    }
    return p;
}

// Triangle row f = (a, b, c), as three int64 or int32 indices (the int32 row in one 12-byte store).
typedef int i32x3u __attribute__((ext_vector_type(3), aligned(4)));
__device__ __forceinline__ void store_tri(void *__restrict__ faces, int64_t f, int64_t a, int64_t b, int64_t c,
                                          int flags) {
    if (flags & DISO_FLAG_INDEX64) {
        int64_t *p = reinterpret_cast<int64_t *>(faces) + 3 * f;
        put(p + 0, a);
        put(p + 1, b);
        put(p + 2, c);
    } else {
        const i32x3u v = {(int)a, (int)b, (int)c};
        __builtin_nontemporal_store(v, reinterpret_cast<i32x3u *>(reinterpret_cast<int32_t *>(faces) + 3 * f));
    }
}

// Quad q = base + rel[0..3], as four int64 or int32 indices; `vec`: `faces` is 16-byte aligned,
// so the quad goes out in 16-byte stores.
typedef long long i64x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void store_quad(void *__restrict__ faces, int64_t q, int64_t base, const int32_t *rel,
                                           int flags, bool vec) {
    if (flags & DISO_FLAG_INDEX64) {
        int64_t *f = reinterpret_cast<int64_t *>(faces) + 4 * q;
        if (vec) {
            put(reinterpret_cast<i64x2 *>(f), i64x2{base + rel[0], base + rel[1]});
            put(reinterpret_cast<i64x2 *>(f) + 1, i64x2{base + rel[2], base + rel[3]});
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) put(f + j, (int64_t)(base + rel[j]));
        }
    } else {
        int32_t *f = reinterpret_cast<int32_t *>(faces) + 4 * q;
        if (vec) {
            put(reinterpret_cast<i32x4 *>(f), i32x4{(int32_t)(base + rel[0]), (int32_t)(base + rel[1]),
                                                  (int32_t)(base + rel[2]), (int32_t)(base + rel[3])});
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) put(f + j, (int32_t)(base + rel[j]));
        }
    }
}

template <typename S>
__device__ __forceinline__ void store_vertex(S *__restrict__ verts, int64_t i, int64_t cap, V3<S> p) {
    if (i < cap) {
        put(verts + 3 * i + 0, p.x);
        put(verts + 3 * i + 1, p.y);
        put(verts + 3 * i + 2, p.z);
    }
}

// Active cells in units of 64, one lane per cell, whatever segments they lie in (so that lanes are
// full on sparse surfaces too). A unit's cells are found from the segments between its first one and
// the next unit's first one: lane i loads segment U0 + i (unit_load, a unit ahead) and each segment
// with cells writes them to `list` at its place. Where more than 64 segments lie in between (a sparse
// stretch), each lane searches its cell's segment instead. unit_cells returns the number of cells
// (of the part of the unit that the load stands for); lane k < n gets cell k's segment (of the launch) and position in it, the other lanes a copy of one.
struct UnitGrid {
    const SegBase *__restrict__ seg;  // launch-level arrays
    Planes P;
    int64_t first, last;  // the grid's first and last segment
    int64_t v0, f0;       // bases of its first segment
};

// Position of the r-th set bit of m (r < popcount).
__device__ __forceinline__ int select64(uint64_t m, int r) {
    uint32_t w = (uint32_t)m;
    int p = 0, c = __popc(w);
    if (r >= c) r -= c, w = (uint32_t)(m >> 32), p = 32;
#pragma unroll
    for (int h = 16; h; h >>= 1) {
        c = __popc(w & ((1u << h) - 1));
        const bool up = r >= c;
        r -= up ? c : 0;
        p += up ? h : 0;
        w = up ? w >> h : w;
    }
    return p;
}

struct UnitLoad {
    uint32_t u;
    int from, to;    // which of its cells
    int64_t U0, U1;  // first and last segment that can hold its cells
    uint64_t A;      // lane i: segment U0 + i
    uint16_t abase;
};
__device__ __forceinline__ UnitLoad unit_load(const UnitGrid &G, uint32_t part, int split, uint32_t nunits, int lane) {
    UnitLoad r;
    const uint32_t u = part >> split;
    r.u = u;
    r.from = (int)(part & ((1u << split) - 1)) * (kWave >> split);
    r.to = r.from + (kWave >> split);
    const int64_t a = G.P.unit[u], b = u + 1 < nunits ? (int64_t)G.P.unit[u + 1] : G.last;
    r.U0 = a > G.first ? a : G.first;
    r.U1 = b < G.last ? b : G.last;
    const int64_t s = r.U0 + lane <= r.U1 ? r.U0 + lane : r.U1;
    r.A = G.P.za[s].b;
    r.abase = G.P.abase[s];
    return r;
}

__device__ __forceinline__ int unit_cells(const UnitGrid &G, const UnitLoad &U, uint16_t *list, int lane,
                                          uint32_t *s_out, int *l_out) {
    const int64_t U0 = U.U0, U1 = U.U1;
    const uint16_t c0 = (uint16_t)(U.u * (uint32_t)kWave);  // number of the unit's first cell
    if (U1 - U0 < kWave) {  // wave-uniform
        const bool in = lane <= (int)(U1 - U0);
        const uint64_t A = in ? U.A : 0ull;
        const int st = in ? (int)(int16_t)(uint16_t)(U.abase - c0) : 0;
        const int s0 = __builtin_amdgcn_readfirstlane(st);
        const int k0 = s0 > U.from ? s0 : U.from;  // (in a batch, the first s0 cells belong to the grid before)
        const int len = U.to - k0;
        int n = 0;
        for (uint64_t act = __ballot(A != 0); act; act &= act - 1) {
            const int j = (int)__builtin_ctzll(act);
            const uint64_t m = (uint64_t)readlane64((int64_t)A, j);
            const int at = __builtin_amdgcn_readlane(st, j) - k0;
            if (at >= len) break;
            const int k = at + lanes_below(m);
            if (__builtin_amdgcn_inverse_ballot_w64(m) && k >= 0 && k < len) list[k] = (uint16_t)(j << 6 | lane);
            n = at + (int)__popcll(m);
        }
        n = n < len ? n : len;
        if (n <= 0) return 0;
        wave_lds_sync();
        const int w = list[lane < n ? lane : n - 1];
        *s_out = (uint32_t)(U0 + (w >> 6));
        *l_out = w & 63;
        wave_lds_sync();
        return n;
    }
    const int s0 = (int)(int16_t)(uint16_t)(G.P.abase[U0] - c0), k0 = s0 > U.from ? s0 : U.from;
    const int c = k0 + lane;  // this lane's cell of the unit
    int64_t lo = U0, hi = U1;
    while (lo < hi) {  // the last segment whose cells start at or before c
        const int64_t mid = (lo + hi + 1) >> 1;
        if ((int)(int16_t)(uint16_t)(G.P.abase[mid] - c0) <= c)
            lo = mid;
        else
            hi = mid - 1;
    }
    const uint64_t A = G.P.za[lo].b;
    const int r = c - (int)(int16_t)(uint16_t)(G.P.abase[lo] - c0);
    const uint64_t ok = __ballot(c < U.to && r < (int)__popcll(A));
    const int n = (int)__popcll(ok);  // the valid lanes are the first ones
    const int l = (ok >> lane) & 1 ? select64(A, r) : 0;
    const int from = lane < n ? lane : 0;
    *s_out = (uint32_t)__shfl((int)(uint32_t)lo, from, kWave);
    *l_out = __shfl(l, from, kWave);
    return n;
}

// A wave's units first, first + step, ... below hi: work(load, next) for each, which returns next(), the
// load of the unit after (called where those loads should be issued: before the work's own stores,
// which the in-order memory counter would otherwise put between them and their use).
template <typename F>
__device__ __forceinline__ void unit_loop(const UnitGrid &G, uint32_t first, uint32_t hi, uint32_t step, int split,
                                          uint32_t nunits, int lane, F work) {
    if (first >= hi) return;  // wave-uniform
    UnitLoad cur = unit_load(G, first, split, nunits, lane);
    for (uint32_t u = first;;) {
        const bool more = step < hi - u;
        const uint32_t un = more ? u + step : u;
        cur = work(cur, [&]() { return unit_load(G, un, split, nunits, lane); });
        if (!more) break;
        u = un;
    }
}

// The units of a launch as a wave goes through them: XCD x takes the x-th eighth, its waves in turn,
// so that at any time an XCD's waves work on neighbouring cells (whose rows share its L2). The grid
// has a multiple of eight blocks. Where there are few units, the time is one wave's chain through one:
// a unit is then cut in two or four, up to kFewParts parts in all (two waves per SIMD). 32^3 noisy, MC /
// DMC 6.6 / 10.4 us whole and 5.7 / 7.8 so, 64^3 6.7 / 10.6 and 6.4 / 9.3; with up to 4096 parts 64^3 takes
// 8.4 / 11.4.
constexpr uint32_t kFewParts = 2048;
template <typename F>
__device__ __forceinline__ void for_units(const UnitGrid &G, uint32_t nunits, int64_t block, int64_t nblocks, int wave,
                                          int lane, F work) {
    const uint32_t xcd = (uint32_t)(block % 8), per = (uint32_t)(nblocks / 8) * kWavesPerBlock;
    const int split = nunits <= kFewParts / 4 ? 2 : (nunits <= kFewParts / 2 ? 1 : 0);
    const uint64_t parts = (uint64_t)nunits << split;
    const uint32_t u0 = (uint32_t)(parts * xcd / 8), u1 = (uint32_t)(parts * (xcd + 1) / 8);
    unit_loop(G, u0 + (uint32_t)(block / 8) * kWavesPerBlock + (uint32_t)wave, u1, per, split, nunits, lane, work);
}

__device__ __forceinline__ int bit_at(uint64_t w, int l) {
    return (int)((((l & 32) ? (uint32_t)(w >> 32) : (uint32_t)w) >> (l & 31)) & 1u);
}

// MC emission, one unit of 64 active cells at a time: its vertices are the crossing edges its cells
// own (all owners of crossing edges are active), its triangles those of its cells; both are
// contiguous rows, in the reference's order (src/cumc.cu:370-410,564-649). Vertex item = (cell,
// axis); triangle item = (cell, triangle), whose corners' table edges come from the case word.
struct McEmitLds {
    int32_t cand[kWave][12];  // vertex id of each table edge, relative to the unit's first vertex
    int32_t cx[kWave], cy[kWave], cz[kWave];
    uint64_t cw[kWave];           // the cells' case words
    uint16_t tri[kWave * 5 + 1];  // triangle items: cell << 3 | triangle
    uint8_t vert[kWave * 3 + 1];  // vertex items: cell * 4 + axis
    // (the last entry of each list takes the writes of the lanes with nothing to list there)
};

// Vertices of a row before position l (b = bits below l), and the row's counts at l.
struct RowEdges {
    uint64_t X, Y, Z;
    __device__ __forceinline__ int below(uint64_t b) const {
        return (int)__popcll(X & b) + (int)__popcll(Y & b) + (int)__popcll(Z & b);
    }
};

template <typename S, bool DEF, typename Next>
__device__ __forceinline__ UnitLoad emit_mc_unit(const In<S> &in, const UnitGrid &G, const UnitLoad &U, Next next,
                                             S *__restrict__ verts, void *__restrict__ faces, const OutCfg &out,
                                             const Norm<S> &nm, const uint64_t *s_case, McEmitLds &L, int lane) {
    wave_lds_sync();  // the previous unit's LDS reads are done
    uint32_t s;
    int l;
    const int n = unit_cells(G, U, L.tri, lane, &s, &l);
    if (n == 0) return next();  // wave-uniform
    const Geo &g = in.geo;
    const SegPos sp = seg_pos(g, (int64_t)s - G.first);
    const bool on = lane < n;
    const uint64_t b = (1ull << l) - 1;

    // the cell's row and rows +x, +y, +x+y (an active cell has them): edges owned there
    const int64_t s10 = (int64_t)s + xstride(g), s01 = (int64_t)s + g.nchunk, s11 = s10 + g.nchunk;
    const uint32_t code = G.P.codes[(int64_t)s * kWave + l];
    const Plane2 *__restrict__ XY = G.P.xy, *__restrict__ ZA = G.P.za;
    const RowEdges e00{XY[s].a, XY[s].b, ZA[s].a}, e10{XY[s10].a, XY[s10].b, ZA[s10].a}, e01{XY[s01].a, XY[s01].b, ZA[s01].a},
        e11{XY[s11].a, XY[s11].b, ZA[s11].a};
    const int64_t v10 = G.seg[s10].v, v01 = G.seg[s01].v, v11 = G.seg[s11].v;
    // x edges at z + 1 in rows 00 and 10
    int xn00 = l < kWave - 1 ? bit_at(e00.X, l + 1) : 0, xn10 = l < kWave - 1 ? bit_at(e10.X, l + 1) : 0;
    if (l == kWave - 1 && sp.chunk + 1 < g.nchunk) {
        xn00 = (int)(XY[s + 1].a & 1);
        xn10 = (int)(XY[s10 + 1].a & 1);
    }

    // first vertex and triangle of the unit: those of its first cell
    const uint64_t b0 = (uint64_t)readlane64((int64_t)b, 0);
    const uint32_t s0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)s);
    const Plane2 q0 = load_uniform(&XY[s0]), w0 = load_uniform(&ZA[s0]);
    const int64_t vabs = G.seg[s0].v + RowEdges{q0.a, q0.b, w0.a}.below(b0), vbase = vabs - G.v0;
    const bool before = __builtin_amdgcn_inverse_ballot_w64(w0.b & b0);  // its segment's cells before it
    const uint32_t bt = before ? (uint32_t)DISO_MC_NTRI(s_case[G.P.codes[(int64_t)s0 * kWave + lane]]) : 0u;
    const int64_t tbase = G.seg[s0].f - G.f0 + __builtin_amdgcn_readlane((int)wave_incl_dpp(bt), kWave - 1);

    const uint64_t cw = s_case[code];
    const int ntri = on ? DISO_MC_NTRI(cw) : 0;
    const int x00 = bit_at(e00.X, l), y00 = bit_at(e00.Y, l), z00 = bit_at(e00.Z, l);
    const int n00 = x00 + y00 + z00;
    const int x10 = bit_at(e10.X, l), n10 = x10 + bit_at(e10.Y, l) + bit_at(e10.Z, l);
    const int n01 = bit_at(e01.X, l) + bit_at(e01.Y, l) + bit_at(e01.Z, l);
    const int n11 = bit_at(e11.X, l) + bit_at(e11.Y, l) + bit_at(e11.Z, l);
    // exclusive prefixes of the vertices (<= 192) and triangles (<= 320) in one scan
    const uint32_t c = on ? (uint32_t)n00 | (uint32_t)ntri << 16 : 0u;
    const uint32_t ic = wave_incl_dpp(c), ec = ic - c, tc = (uint32_t)__builtin_amdgcn_readlane((int)ic, kWave - 1);
    const int pv = (int)(ec & 0xffff), pt = (int)(ec >> 16), tv = (int)(tc & 0xffff), tt = (int)(tc >> 16);
    const int32_t r10 = (int32_t)(v10 - vabs) + e10.below(b), r01 = (int32_t)(v01 - vabs) + e01.below(b),
                  r11 = (int32_t)(v11 - vabs) + e11.below(b);

    if (on) {
        // A corner on table edge e lies on an edge owned by the cell at (cell + edge offset); its id is
        // that owner's first vertex plus the rank of the edge's axis among the owner's crossing axes
        // (what create_cell_mc_tris_kernel finds by linear search, src/cumc.cu:586-608). Owners are the
        // cell, its +x, +y, +x+y neighbours and their +z neighbours, whose first vertex is the current
        // one's first vertex plus its count.
        int32_t *d = L.cand[lane];
        d[0] = pv;
        d[1] = r10 + n10 - 1;
        d[2] = pv + n00;
        d[3] = pv + n00 - 1;
        d[4] = r01;
        d[5] = r11 + n11 - 1;
        d[6] = r01 + n01;
        d[7] = r01 + n01 - 1;
        d[8] = pv + x00;
        d[9] = r10 + x10;
        d[10] = r10 + n10 + xn10;
        d[11] = pv + n00 + xn00;
        L.cx[lane] = sp.px;
        L.cy[lane] = sp.py;
        L.cz[lane] = sp.chunk * kWave + l;
        L.cw[lane] = cw;
    }
    // list writes without per-lane branches: what is not listed goes to the spare last entry
    L.vert[on && x00 ? pv : 3 * kWave] = (uint8_t)(lane * 4);
    L.vert[on && y00 ? pv + x00 : 3 * kWave] = (uint8_t)(lane * 4 + 1);
    L.vert[on && z00 ? pv + x00 + y00 : 3 * kWave] = (uint8_t)(lane * 4 + 2);
#pragma unroll
    for (int t = 0; t < 5; ++t) L.tri[t < ntri ? pt + t : 5 * kWave] = (uint16_t)((lane << 3) | t);
    wave_lds_sync();

    const UnitLoad after = next();
    for (int k = lane; k < tv; k += kWave) {
        const int it = L.vert[k], src = it >> 2, a = it & 3;
        const V3<S> p = edge_vertex<S, DEF>(in, L.cx[src], L.cy[src], L.cz[src], a);
        store_vertex(verts, vbase + k, out.vcap, epilogue(p, out.flags, nm));
    }
    // triangle k of the unit per lane: its cell's case word once, the three corners' table edges and
    // vertex ids (independent LDS reads), then the three indices as one row
    for (int k = lane; k < tt; k += kWave) {
        const int64_t f = tbase + k;
        if (f >= out.fcap) continue;
        const int it = L.tri[k], src = it >> 3, t = it & 7;
        const uint64_t w = L.cw[src];
        const int32_t *cand = L.cand[src];
        store_tri(faces, f, vbase + cand[DISO_MC_EDGE(w, 3 * t)], vbase + cand[DISO_MC_EDGE(w, 3 * t + 1)],
                  vbase + cand[DISO_MC_EDGE(w, 3 * t + 2)], out.flags);
    }
    return after;
}

__device__ __forceinline__ void load_mc_cases(uint64_t *s_case) {
    for (int i = threadIdx.x; i < 256; i += kBlock) s_case[i] = kMcCase[i];
}

template <typename S, bool DEF>
__global__ __launch_bounds__(kBlock, 6) void emit_mc_kernel(In<S> in, const SegBase *__restrict__ seg, Planes planes,
                                                         S *__restrict__ verts, void *__restrict__ faces, OutCfg out,
                                                         Norm<S> nm) {
    __shared__ uint64_t s_case[256];
    __shared__ McEmitLds s_lds[kWavesPerBlock];
    const int wave = wave_id(), lane = threadIdx.x % kWave;
    const SegBase *tot = seg + in.geo.nseg;
    if (tot[0].v > out.vcap || tot[0].f > out.fcap) return;
    load_mc_cases(s_case);
    __syncthreads();
    const uint32_t nunits = *planes.nunits;
    const UnitGrid G{seg, planes, 0, in.geo.nseg - 1, 0, 0};
    for_units(G, nunits, blockIdx.x, gridDim.x, wave, lane, [&](const UnitLoad &U, auto next) {
        return emit_mc_unit<S, DEF>(in, G, U, next, verts, faces, out, nm, s_case, s_lds[wave], lane);
    });
}

// DMC emission. Patch-vertex item = (lane, patch): the mean of the MC vertices on the patch's
// edges, summed from zero in ascending edge order and scaled by 1/num (src/cudualmc.cu:907-955);
// each MC vertex is evaluated with the same expression as the MC pass, so it has the same bits.
// Quad item = (lane, axis, leaving) of an owned crossing edge (src/cudualmc.cu:1027-1056): its
// corners are the vertices of the patches holding the edge in the four cells around it, which
// lie in rows R00, Rm0 (-x), R0m (-y), Rmm (-x-y) at this z and z-1. Cell codes come from the
// count pass, so no sample is read to classify.

// Quad stencil (src/cudualmc.cu:504-513) as cell index ci and edge id: entry k of type ty.
// Types 3..5 (edges leaving the inside) list the cells of types 0..2 in the order 0,3,2,1.
__device__ constexpr int stencil_ci(int ty, int k) {
    constexpr int q[3][4] = {{0, 2, 3, 1}, {0, 1, 5, 4}, {0, 4, 6, 2}};
    return ty < 3 ? q[ty][k] : q[ty - 3][(4 - k) & 3];
}
__device__ constexpr int stencil_eid(int ty, int k) {
    constexpr int q[3][4] = {{0, 4, 6, 2}, {8, 11, 10, 9}, {3, 1, 5, 7}};
    return ty < 3 ? q[ty][k] : q[ty - 3][(4 - k) & 3];
}

// The edge and quad tables as the kernels evaluate them (eox..eax, stencil_ci / stencil_eid) agree
// with the tables' entries (diso_tables.h: edge offsets and axes, quad cell offsets and edge ids).
__device__ constexpr bool tables_agree() {
    const int ofs[12][3] = {DISO_EDGE_OFS_VALUES};
    const int axis[12] = {DISO_EDGE_AXIS_VALUES};
    const int quad[6][4][4] = {DISO_QUAD_VALUES};
    for (int e = 0; e < 12; ++e)
        if (eox(e) != ofs[e][0] || eoy(e) != ofs[e][1] || eoz(e) != ofs[e][2] || eax(e) != axis[e]) return false;
    for (int ty = 0; ty < 6; ++ty)
        for (int k = 0; k < 4; ++k) {
            const int *c = quad[ty][k];
            if (stencil_ci(ty, k) != -4 * c[0] - 2 * c[1] - c[2] || stencil_eid(ty, k) != c[3]) return false;
        }
    return true;
}
static_assert(tables_agree(), "edge / quad tables");

// Edges of a dual cell that start at its own z (the other four, on its top face, are the next
// position's): kinds 0..7 in ascending edge number, with the edge's offsets and axis as bit masks
// over the kinds. Top edges 2, 6, 10, 11 are kinds 0, 3, 7, 6 of the next position.
__host__ __device__ constexpr int kind_edge(int k) { return k + (k >= 2) + (k >= 5); }  // 0 1 3 4 5 7 8 9
constexpr int kTopEdges[4] = {2, 6, 10, 11}, kTopKinds[4] = {0, 3, 7, 6};
constexpr int kKindX = 0x92, kKindY = 0x38, kKindAxisZ = 0x36, kKindAxisY = 0xC0;
__device__ constexpr bool kinds_ok() {
    for (int k = 0; k < 8; ++k) {
        const int e = kind_edge(k);
        if (eoz(e) || eox(e) != ((kKindX >> k) & 1) || eoy(e) != ((kKindY >> k) & 1) ||
            eax(e) != ((kKindAxisZ >> k) & 1 ? 2 : (kKindAxisY >> k) & 1))
            return false;
    }
    for (int t = 0; t < 4; ++t) {
        const int e = kTopEdges[t], d = kind_edge(kTopKinds[t]);
        if (!eoz(e) || eox(e) != eox(d) || eoy(e) != eoy(d) || eax(e) != eax(d)) return false;
    }
    return true;
}
static_assert(kinds_ok(), "edge kinds");
// An edge of the cell as a bit: its kind at the cell's own position, or 8 + its kind at the next.
__host__ __device__ constexpr int edge_bit(int e) {
    for (int k = 0; k < 8; ++k)
        if (kind_edge(k) == e) return k;
    for (int t = 0; t < 4; ++t)
        if (kTopEdges[t] == e) return 8 + kTopKinds[t];
    return 16;
}
__host__ __device__ constexpr uint64_t edge_bits() {  // all twelve, four bits each
    uint64_t w = 0;
    for (int e = 0; e < 12; ++e) w |= (uint64_t)edge_bit(e) << (4 * e);
    return w;
}
// The kinds that cross in a cell of code c (Morton corner order); a cell of the inverted code has
// the same. And the top edges that cross, as kinds of the next position.
__host__ __device__ constexpr uint32_t own_kinds(uint32_t c) {
    const uint32_t x = c ^ (c >> 1), y = c ^ (c >> 2), z = c ^ (c >> 4);
    return (x & 1) | (z & 2) | (z & 1) << 2 | (x & 4) << 1 | (z & 8) << 1 | (z & 4) << 3 | (y & 3) << 6;
}
__host__ __device__ constexpr uint32_t top_kinds(uint32_t c) {
    const uint32_t x = c ^ (c >> 1), y = c ^ (c >> 2);
    return ((x >> 4) & 1) | ((x >> 6) & 1) << 3 | ((y >> 4) & 3) << 6;
}

// MC vertices kept per unit; a unit with more recomputes them per patch. White noise averages 256
// per unit (8 kinds, half of them crossing, 64 cells) and stays below 320.
constexpr int kEdgeSlots = 320;

template <typename S>
struct DmcEmitLds {
    // entry k + 1: cell k's first edge slot (bits 0-9), whether its sample is inside (bit 10), the
    // kinds that cross (bits 16-23), its code (bits 24-31); entry 0: the code of the cell below cell
    // 0; entry n + 1: the slots and kinds of the position above the last cell
    uint32_t cw[kWave + 2];
    int64_t idx[kWave + 1];                         // the cells (and that position): index of the sample
    S cx[kWave + 1], cy[kWave + 1], cz[kWave + 1];  // there (as if it were stored), position, and which
    uint8_t stored[kWave + 1];                      // of the corners are stored (bit dx | dy << 1 | dz << 2)
    uint16_t pp[kWave];            // patches of the unit before the cell's
    uint8_t patch[kWave * 4 + 1];  // patch items: cell * 4 + patch
    uint8_t quad[kWave * 3 + 1];   // quad items: cell * 4 + axis
    // (the last entry of each list takes the writes of the lanes with nothing to list there)
    uint16_t eitem[kEdgeSlots + 1];  // edge items, from slot 1: cell * 8 + kind (entry 0: spare)
    union {
        struct {  // neighbour rows -x, -y, -x-y, until the quads are written
            int32_t nf[3][kWave];  // first patch of the row's cell at z, relative to the unit's first
            uint32_t nc[kWave];    // codes: row -x at z and z - 1, row -y at z and z - 1
            uint8_t nd[kWave];     // code: row -x-y at z
        };
        S ev[3][kEdgeSlots + 1];  // then the MC vertices by slot; entry 0 holds zeros
    };
};

// Edges of the patches of every DMC case as edge_bit()s, 16 bits per patch, derived at compile time
// from the case table.
struct PatchEdgeTable {
    uint64_t m[256];
};
constexpr PatchEdgeTable make_patch_edges() {
    const uint64_t cases[256] = {DISO_DMC_CASE_VALUES};
    PatchEdgeTable t{};
    for (int c = 0; c < 256; ++c) {
        uint64_t w = 0;
        for (int e = 0; e < 12; ++e) {
            const int k = DISO_DMC_PATCH_OF(cases[c], e);
            if (k < 4) w |= 1ull << (16 * k + edge_bit(e));
        }
        t.m[c] = w;
    }
    return t;
}
__constant__ PatchEdgeTable kDmcPatchEdges = make_patch_edges();

// An edge kind: its ends' sample indices relative to the position's and their bits in the stored
// corners, its start's offset and its direction.
template <typename S>
struct alignas(16) KindEnds {
    int64_t d0, d1;
    S ox, oy, ax, ay, az;
    uint16_t c0, c1;
};

// The tables of the DMC emission, in LDS: the case words with each code's own_kinds in the free top
// byte, the patches' edges, the edge kinds in the grid's strides, and 1/n for the possible patch sizes
// (n = 1..7; correctly rounded).
template <typename S>
struct DmcTables {
    uint64_t cases[256], edges[256];
    KindEnds<S> kind[8];
    S rcp[8];
    __device__ __forceinline__ void load(const Geo &g) {
        const int t = threadIdx.x;
        for (int i = t; i < 256; i += kBlock) {
            cases[i] = kDmcCase[i] | (uint64_t)own_kinds((uint32_t)i) << 56;
            edges[i] = kDmcPatchEdges.m[i];
        }
        if (t < 8) {
            const int dx = (kKindX >> t) & 1, dy = (kKindY >> t) & 1;
            const int a = (kKindAxisZ >> t) & 1 ? 2 : (kKindAxisY >> t) & 1;
            const int64_t sy = g.n2, sx = (int64_t)g.n1 * g.n2, d0 = (dx ? sx : 0) + (dy ? sy : 0);
            const int c0 = dx | dy << 1;
            kind[t] = KindEnds<S>{d0, d0 + (a == 0 ? sx : (a == 1 ? sy : 1)), S(dx), S(dy),
                                  S(a == 0), S(a == 1), S(a == 2), (uint16_t)c0, (uint16_t)(c0 + (1 << a))};
            rcp[t] = t ? S(1) / S(t) : S(0);
        }
    }
};

// Patches before position l of a segment (b = bits below l).
__device__ __forceinline__ int patches_below(uint64_t A, Plane2 m, uint64_t b) {
    return (int)__popcll(A & b) + (int)__popcll(m.a & b) + 2 * (int)__popcll(m.b & b);
}
// Which corners of the cell at a position are stored samples (bit dx | dy << 1 | dz << 2).
__device__ __forceinline__ uint32_t stored_corners(const Geo &g, int x, int y, int z) {
    const int a = x - g.off, b = y - g.off, c = z - g.off;
    const uint32_t mx = ((unsigned)a < (unsigned)g.n0 ? 0x55u : 0u) | ((unsigned)(a + 1) < (unsigned)g.n0 ? 0xaau : 0u);
    const uint32_t my = ((unsigned)b < (unsigned)g.n1 ? 0x33u : 0u) | ((unsigned)(b + 1) < (unsigned)g.n1 ? 0xccu : 0u);
    const uint32_t mz = ((unsigned)c < (unsigned)g.n2 ? 0x0fu : 0u) | ((unsigned)(c + 1) < (unsigned)g.n2 ? 0xf0u : 0u);
    return mx & my & mz;
}

// MC vertex of the edge of kind K at a position (c: its coordinates; stored, idx: as in DmcEmitLds) as
// a patch sums it, lerp_vertex()'s expression: zero where the edge does not cross (on NaN samples only,
// for an edge whose ends' inside bits differ). An end that is not stored reads as the pad value with a
// zero deform (it loads element 0, so no lane needs its own execution mask around the loads).
template <typename S, bool DEF>
__device__ __forceinline__ V3<S> patch_edge_vertex(const In<S> &in, const KindEnds<S> &K, int64_t idx, uint32_t stored,
                                                   V3<S> c) {
    const bool ok0 = (stored >> K.c0) & 1, ok1 = (stored >> K.c1) & 1;
    const int64_t j0 = ok0 ? idx + K.d0 : 0, j1 = ok1 ? idx + K.d1 : 0;
    S d0 = in.sdf[j0], d1 = in.sdf[j1];
    V3<S> f0{}, f1{};
    if (DEF) {
        f0 = V3<S>{in.deform[3 * j0], in.deform[3 * j0 + 1], in.deform[3 * j0 + 2]};
        f1 = V3<S>{in.deform[3 * j1], in.deform[3 * j1 + 1], in.deform[3 * j1 + 2]};
    }
    if (__any(!ok0 || !ok1)) {  // wave-uniform
        d0 = ok0 ? d0 : in.pad;
        d1 = ok1 ? d1 : in.pad;
        f0 = V3<S>{ok0 ? f0.x : S(0), ok0 ? f0.y : S(0), ok0 ? f0.z : S(0)};
        f1 = V3<S>{ok1 ? f1.x : S(0), ok1 ? f1.y : S(0), ok1 ? f1.z : S(0)};
    }
    const S t = interp_t(d0, d1, in.iso);
    // (positions are whole numbers below 2^21: their sums are exact)
    V3<S> p0 = {c.x + K.ox, c.y + K.oy, c.z}, p1 = {p0.x + K.ax, p0.y + K.ay, p0.z + K.az};
    if (DEF) {
        p0 = add3(p0, f0);
        p1 = add3(p1, f1);
    }
    const bool nan = __builtin_isunordered(d0, d1);
    return V3<S>{nan ? S(0) : p0.x + (p1.x - p0.x) * t, nan ? S(0) : p0.y + (p1.y - p0.y) * t,
                 nan ? S(0) : p0.z + (p1.z - p0.z) * t};
}

// One unit of 64 active cells: its patch vertices and the quads of the edges its cells own. Both are
// contiguous rows of the output, in the cells' order. Bound by vector instructions (four fifths of the
// issue slots on white noise), so what a cell's edges share is worked out once per cell, and the rest
// comes from small tables. Per edge position, index and bounds, and per patch the slots bit by bit:
// 128x120x136 white noise 104 us, 256^3 noisy 173, 512^3 430; so 96, 163, 396.
template <typename S, bool DEF, typename Next>
__device__ __forceinline__ UnitLoad emit_dmc_unit(const In<S> &in, const UnitGrid &G, const UnitLoad &U, Next next,
                                              S *__restrict__ verts, void *__restrict__ faces,
                                              uint8_t *__restrict__ vinfo, const OutCfg &out, const Norm<S> &nm,
                                              const DmcTables<S> &T, DmcEmitLds<S> &L, int lane) {
    wave_lds_sync();  // the previous unit's LDS reads are done
    uint32_t s;
    int l;
    const int n = unit_cells(G, U, L.eitem, lane, &s, &l);
    if (n == 0) return next();  // wave-uniform
    const Geo &g = in.geo;
    const SegPos sp = seg_pos(g, (int64_t)s - G.first);
    const int px = sp.px, py = sp.py, z = sp.chunk * kWave + l;
    const bool on = lane < n;

    // Loads: the cell's own planes and code; of rows -x, -y, -x-y the patch planes, the base and the
    // codes at z and z - 1 (a cell that shares a crossing edge with an active one is active, so the
    // codes that are used have been written).
    const Plane2 qxy = G.P.xy[s], qza = G.P.za[s];
    const bool rx = px > 0, ry = py > 0, rz = z > 0;
    const int64_t sx = rx ? xstride(g) : 0, sy = ry ? g.nchunk : 0;
    const int64_t s10 = (int64_t)s - sx, s01 = (int64_t)s - sy, s11 = rx && ry ? (int64_t)s - sx - sy : (int64_t)s;
    const int below1 = rz ? 1 : 0;
    const uint8_t *cd = G.P.codes + l;
    uint32_t code = cd[(int64_t)s * kWave];
    uint32_t cx0 = cd[s10 * kWave], cx1 = (cd - below1)[s10 * kWave];
    uint32_t cy0 = cd[s01 * kWave], cy1 = (cd - below1)[s01 * kWave];
    uint32_t cxy = cd[s11 * kWave];
    uint32_t cz1 = (cd - below1)[(int64_t)s * kWave];
    const uint64_t inside = G.P.inside[s];
    const uint64_t ax = G.P.za[s10].b, ay = G.P.za[s01].b, aw = G.P.za[s11].b;
    const Plane2 mx = G.P.m[s10], my = G.P.m[s01], mw = G.P.m[s11];
    const int64_t fx = G.seg[s10].f, fy = G.seg[s01].f, fw = G.seg[s11].f, fs = G.seg[s].f;
    const uint64_t b = (1ull << l) - 1;

    // first patch and first quad of the unit: those of its first cell
    const uint64_t b0 = (uint64_t)readlane64((int64_t)b, 0);
    const uint32_t s0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)s);
    const Plane2 q0 = load_uniform(&G.P.xy[s0]), w0 = load_uniform(&G.P.za[s0]), m0 = load_uniform(&G.P.m[s0]);
    const int64_t pbase = G.seg[s0].f - G.f0 + patches_below(w0.b, m0, b0);
    const int64_t qbase = G.seg[s0].v - G.v0 + RowEdges{q0.a, q0.b, w0.a}.below(b0);
    const int64_t pabs = pbase + G.f0;

    // crossing kinds of the edges at the cell's own z; where the owner's row anchors no cells, or
    // (top edges) the next position, an edge counts as not crossing
    const bool gx = px + 1 < g.g0 - 1, gy = py + 1 < g.g1 - 1, gz = z + 1 < g.g2 - 1;
    const uint32_t keep = (gx ? 0xffu : 0x7du) & (gy ? 0xffu : 0xd7u) & (gx && gy ? 0xffu : 0xefu);
    const uint64_t cwd = T.cases[code];
    const uint32_t kb = on ? (uint32_t)(cwd >> 56) & keep : 0u;
    const int np = on ? DISO_DMC_NPATCH(cwd) : 0;
    const int ex = on ? bit_at(qxy.a, l) : 0, ey = on ? bit_at(qxy.b, l) : 0, ez = on ? bit_at(qza.a, l) : 0;
    // exclusive prefixes of the edge slots (<= 512), patches (<= 256) and quads (<= 192): one scan
    const uint32_t c = (uint32_t)__popc(kb) | (uint32_t)np << 10 | (uint32_t)(ex + ey + ez) << 20;
    const uint32_t ic = wave_incl_dpp(c), ec = ic - c;
    const uint32_t tc = (uint32_t)__builtin_amdgcn_readlane((int)ic, kWave - 1);
    const int pe = (int)(ec & 0x3ff), pp = (int)((ec >> 10) & 0x3ff), pq = (int)(ec >> 20);
    const int te = (int)(tc & 0x3ff), tp = (int)((tc >> 10) & 0x3ff), tq = (int)(tc >> 20);
    // the position above the last cell: its crossing kinds are that cell's top edges
    const uint32_t lcode = (uint32_t)__builtin_amdgcn_readlane((int)code, n - 1);
    const uint32_t lkeep = (uint32_t)__builtin_amdgcn_readlane((int)(gz ? keep : 0u), n - 1);
    const uint32_t hk = top_kinds(lcode) & lkeep;
    const int nslot = te + __popc(hk);
    const bool slots = nslot <= kEdgeSlots;  // wave-uniform

    const uint32_t stored = stored_corners(g, px, py, z);
    const int64_t idx = data_index(in, px, py, z);
    if (on) {
        // bit 11: the top edges are the next cell's (they cross only where its position has a cell)
        L.cw[lane + 1] = (uint32_t)(pe + 1) | (uint32_t)bit_at(inside, l) << 10 | (gz ? 1u << 11 : 0u) | kb << 16 | code << 24;
        L.idx[lane] = idx;
        L.cx[lane] = S(px);
        L.cy[lane] = S(py);
        L.cz[lane] = S(z);
        L.stored[lane] = (uint8_t)stored;
        L.pp[lane] = (uint16_t)pp;
    }
    if (lane == n - 1) {
        L.idx[n] = idx + 1;
        L.cx[n] = S(px);
        L.cy[n] = S(py);
        L.cz[n] = S(z + 1);
        L.stored[n] = (uint8_t)(stored >> 4);  // (no edge of it that counts runs along z)
        L.cw[n + 1] = (uint32_t)(te + 1) | hk << 16;
    }
    if (lane == 0) L.cw[0] = (rz ? cz1 : 0u) << 24;
    // list writes without per-lane branches: what is not listed goes to the spare entry
#pragma unroll
    for (int k = 0; k < 4; ++k) L.patch[k < np ? pp + k : 4 * kWave] = (uint8_t)(lane * 4 + k);
    L.quad[ex ? pq : 3 * kWave] = (uint8_t)(lane * 4);
    L.quad[ey ? pq + ex : 3 * kWave] = (uint8_t)(lane * 4 + 1);
    L.quad[ez ? pq + ex + ey : 3 * kWave] = (uint8_t)(lane * 4 + 2);
    if (slots) {
        int r = pe + 1;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int x = (int)((kb >> k) & 1);
            L.eitem[x ? r : 0] = (uint16_t)(lane * 8 + k);
            r += x;
        }
        if (lane < 8 && ((hk >> lane) & 1)) L.eitem[te + 1 + __popc(hk & ((1u << lane) - 1))] = (uint16_t)(n * 8 + lane);
    }
    // neighbour rows (where there is none, the quad corner is one before the segment's first patch)
    const int32_t own0 = (int32_t)(fs - pabs);
    L.nf[0][lane] = rx ? (int32_t)(fx - pabs) + patches_below(ax, mx, b) : own0;
    L.nf[1][lane] = ry ? (int32_t)(fy - pabs) + patches_below(ay, my, b) : own0;
    L.nf[2][lane] = rx && ry ? (int32_t)(fw - pabs) + patches_below(aw, mw, b) : own0;
    L.nc[lane] = (rx ? cx0 | (rz ? cx1 << 8 : 0u) : 0u) | (ry ? cy0 << 16 | (rz ? cy1 << 24 : 0u) : 0u);
    L.nd[lane] = (uint8_t)(rx && ry ? cxy : 0u);
    wave_lds_sync();

    const UnitLoad after = next();
    // quads: corner 0 is the own cell's vertex; corners B, C, D those of the other three cells around
    // the edge (X: -y, -y below, below; Y: below, -x below, -x; Z: -x, -x-y, -y), in that order or,
    // where the edge leaves the inside, in reverse. A cell below a row's cell at z has its patches
    // right before that cell's.
    const bool vec = ((uintptr_t)faces & 15) == 0;  // a quad's four indices in 16-byte stores
    for (int k = lane; k < tq; k += kWave) {
        const int64_t qi = qbase + k;
        if (qi >= out.fcap) continue;
        const int it = L.quad[k], src = it >> 2, axis = it & 3;
        const uint32_t w = L.cw[src + 1], wb = L.cw[src] >> 24, nc = L.nc[src], nd = L.nd[src];
        const int32_t f0 = L.pp[src], fx0 = L.nf[0][src], fy0 = L.nf[1][src], fw0 = L.nf[2][src];
        const bool isx = axis == 0, isy = axis == 1;
        const uint32_t czb = L.cz[src] > S(0) ? wb : 0u;
        const uint64_t wa = T.cases[w >> 24];
        const uint64_t wB = T.cases[isx ? (nc >> 16) & 0xff : (isy ? czb : nc & 0xff)];
        const uint64_t wC = T.cases[isx ? nc >> 24 : (isy ? (nc >> 8) & 0xff : nd)];
        const uint64_t wD = T.cases[isx ? czb : (isy ? nc & 0xff : (nc >> 16) & 0xff)];
        const int pa = (int)(wa >> (isx ? 0 : (isy ? 24 : 9))) & 7;         // edges 0, 8, 3
        const int pB = (int)(wB >> (isx ? 12 : (isy ? 33 : 3))) & 7;        // edges 4, 11, 1
        const int pC = (int)(wC >> (isx ? 18 : (isy ? 30 : 15))) & 7;       // edges 6, 10, 5
        const int pD = (int)(wD >> (isx ? 6 : (isy ? 27 : 21))) & 7;        // edges 2, 9, 7
        const int32_t va = f0 + (pa == 7 ? -1 : pa);
        const int32_t vB = (isx ? fy0 : (isy ? f0 - DISO_DMC_NPATCH(wB) : fx0)) + (pB == 7 ? -1 : pB);
        const int32_t vC = (isx ? fy0 - DISO_DMC_NPATCH(wC) : (isy ? fx0 - DISO_DMC_NPATCH(wC) : fw0)) + (pC == 7 ? -1 : pC);
        const int32_t vD = (isx ? f0 - DISO_DMC_NPATCH(wD) : (isy ? fx0 : fy0)) + (pD == 7 ? -1 : pD);
        const bool leaving = (w >> 10) & 1;
        const int32_t rel[4] = {va, leaving ? vD : vB, vC, leaving ? vB : vD};
        store_quad(faces, qi, pbase, rel, out.flags, vec);
    }
    wave_lds_sync();  // the neighbour rows' entries give way to the vertices

    if (slots) {
        if (lane < 3) L.ev[lane][0] = S(0);
        // MC vertex of every crossing edge of the cells, once
        for (int i = lane; i < nslot; i += kWave) {
            const int it = L.eitem[i + 1], src = it >> 3, k = it & 7;
            const V3<S> p = patch_edge_vertex<S, DEF>(in, T.kind[k], L.idx[src], L.stored[src],
                                                      V3<S>{L.cx[src], L.cy[src], L.cz[src]});
            L.ev[0][i + 1] = p.x;
            L.ev[1][i + 1] = p.y;
            L.ev[2][i + 1] = p.z;
        }
        wave_lds_sync();
    }

    for (int k = lane; k < tp; k += kWave) {
        const int it = L.patch[k], src = it >> 2, pk = it & 3;
        const uint32_t w0 = L.cw[src + 1];
        const uint32_t em = (uint32_t)(T.edges[w0 >> 24] >> (16 * pk)) & 0xffffu;
        const int num = __popc(em);
        S sx2 = S(0), sy2 = S(0), sz2 = S(0);
        if (slots) {
            // the slots of all twelve edges first (as byte offsets), then all twelve vertices added in
            // ascending edge order, edges outside the patch (or not counted as crossing) reading the
            // zero entry: the running sum starts at +0 and so is never -0, and adding +0 leaves it
            // unchanged
            const uint32_t w1 = L.cw[src + 2];
            const uint32_t k0 = (w0 >> 16) & 0xff, k1 = (w0 >> 11) & 1 ? (w1 >> 16) & 0xff : 0u;
            const int e0 = (int)(em & k0), e1 = (int)((em >> 8) & k1);
            int r0 = (int)(w0 & 0x3ff) * (int)sizeof(S);
            const int r1 = (int)(w1 & 0x3ff);
            int sl[12];
#pragma unroll
            for (int k2 = 0; k2 < 8; ++k2) {
                sl[kind_edge(k2)] = r0 & __builtin_amdgcn_sbfe(e0, k2, 1);
                r0 += (int)__builtin_amdgcn_ubfe(k0, k2, 1) * (int)sizeof(S);
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int kd = kTopKinds[t];
                sl[kTopEdges[t]] =
                    (r1 + __popc(k1 & ((1u << kd) - 1))) * (int)sizeof(S) & __builtin_amdgcn_sbfe(e1, kd, 1);
            }
#pragma unroll
            for (int e = 0; e < 12; ++e) {
                const char *at = reinterpret_cast<const char *>(L.ev[0]) + sl[e];
                sx2 += reinterpret_cast<const S *>(at)[0];
                sy2 += reinterpret_cast<const S *>(at)[kEdgeSlots + 1];
                sz2 += reinterpret_cast<const S *>(at)[2 * (kEdgeSlots + 1)];
            }
        } else {
            const V3<S> c = {L.cx[src], L.cy[src], L.cz[src]};
            const bool okx = (int)c.x + 1 < g.g0 - 1, oky = (int)c.y + 1 < g.g1 - 1, okz = (int)c.z + 1 < g.g2 - 1;
            constexpr uint64_t kEdgeBits = edge_bits();
            for (int e = 0; e < 12; ++e) {  // ascending edge order
                const int bit = (int)(kEdgeBits >> (4 * e)) & 15, up = bit >> 3;
                if (!((em >> bit) & 1) || (eox(e) && !okx) || (eoy(e) && !oky) || (eoz(e) && !okz)) continue;
                const V3<S> p = patch_edge_vertex<S, DEF>(in, T.kind[bit & 7], L.idx[src] + up, L.stored[src] >> (4 * up),
                                                          V3<S>{c.x, c.y, c.z + S(up)});
                sx2 += p.x;
                sy2 += p.y;
                sz2 += p.z;
            }
        }
        const S r = T.rcp[num];
        store_vertex(verts, pbase + k, out.vcap, epilogue(V3<S>{sx2 * r, sy2 * r, sz2 * r}, out.flags, nm));
        if (pbase + k < out.vcap) put(vinfo + pbase + k, (uint8_t)(num | (pk << 3)));
    }
    return after;
}

template <typename S, bool DEF>
__global__ __launch_bounds__(kBlock, 5) void emit_dmc_kernel(In<S> in, const SegBase *__restrict__ seg, Planes planes,
                                                          S *__restrict__ verts, void *__restrict__ faces,
                                                          uint8_t *__restrict__ vinfo, OutCfg out, Norm<S> nm) {
    __shared__ DmcTables<S> s_tab;
    __shared__ DmcEmitLds<S> s_lds[kWavesPerBlock];
    const int wave = wave_id(), lane = threadIdx.x % kWave;
    const SegBase *tot = seg + in.geo.nseg;
    if (tot[0].v > out.fcap || tot[0].f > out.vcap) return;
    s_tab.load(in.geo);
    __syncthreads();
    const uint32_t nunits = *planes.nunits;
    const UnitGrid G{seg, planes, 0, in.geo.nseg - 1, 0, 0};
    for_units(G, nunits, blockIdx.x, gridDim.x, wave, lane, [&](const UnitLoad &U, auto next) {
        return emit_dmc_unit<S, DEF>(in, G, U, next, verts, faces, vinfo, out, nm, s_tab, s_lds[wave], lane);
    });
}

// ------------------------------------------------------------------------------------------
// Backward (gather, deterministic)
//
// MC: one lane per touched grid vertex (one with an incident crossing edge), compacted over a wave's
// run of segments; its incident crossing edges (at most six: the three it owns and the ones owned by
// its -x, -y, -z neighbours) become items of a dense per-wave list. Each item computes the adjoint of
// its edge vertex (adjComputeMcVert, src/cumc.cu:412-453) for the lane's endpoint; the owning lane
// adds its items up in a fixed order (slot 0..5), so results are deterministic and no atomics are
// used. Item slots: 0/1/2 = edge along x/y/z owned by the vertex (vertex is its start), 3/4/5 = edge
// along x/y/z owned by the -x/-y/-z neighbour (vertex is its end).
//
// DMC: dmc_edge_grad_kernel first turns the DMC vertex gradients into one upstream gradient per
// crossing edge (MC vertex order = quad order): the sum over the quad's four corners of (gradient
// of that patch vertex) / (edges in its patch), the adjoint of create_dmc_verts_kernel's mean
// (src/cudualmc.cu:907-955); with DISO_FLAG_REFERENCE_COMPAT each corner reads its cell's first
// patch instead (src/cudualmc.cu:990). The MC gather then runs on those edge gradients.

template <typename S>
struct AdjIn {
    const S *__restrict__ adj;  // [n, 3]
    int64_t n;
    int flags;
    Norm<S> nm;  // upstream scaling by 1/(dims-1) when the forward normalised
};

// Row i < n of the upstream gradient.
template <typename S>
__device__ __forceinline__ V3<S> load_adj_at(const AdjIn<S> &a, int64_t i) {
    V3<S> r = {a.adj[3 * i + 0], a.adj[3 * i + 1], a.adj[3 * i + 2]};
    if (a.flags & DISO_FLAG_NORMALIZE) {  // grad of verts / (dims - 1): g / (dims - 1)
        r.x = div_by(r.x, a.nm.c[0], a.nm.r[0]);
        r.y = div_by(r.y, a.nm.c[1], a.nm.r[1]);
        r.z = div_by(r.z, a.nm.c[2], a.nm.r[2]);
    }
    return r;
}
template <typename S>
__device__ __forceinline__ V3<S> load_adj(const AdjIn<S> &a, int64_t i) {
    return i >= 0 && i < a.n ? load_adj_at(a, i) : V3<S>{S(0), S(0), S(0)};
}

template <typename S>
struct Grad {
    S g, dx, dy, dz;
};

// 1 / dd of an edge, and the quotient a / dd. fp32: gradients are compared within a tolerance, so the
// hardware reciprocal (within an ulp) stands for the division.
template <typename S>
struct EdgeQuot {
    S dd;
    __device__ __forceinline__ explicit EdgeQuot(S d) : dd(d) {}
    __device__ __forceinline__ S of(S a) const { return a / dd; }
};
template <>
struct EdgeQuot<float> {
    float r;
    __device__ __forceinline__ explicit EdgeQuot(float d) : r(__builtin_amdgcn_rcpf(d)) {}
    __device__ __forceinline__ float of(float a) const { return a * r; }
};

// Adjoint of one edge vertex (upstream gradient gv) at one of the edge's ends: at integer position c
// with sample d and deform f; the other end (dO, fO) is one step along `axis` away, in direction dir
// (1 or -1). With t = (iso - d0) / (d1 - d0) and the vertex p0 + (p1 - p0) t
// (src/cumc.cu:343-368,412-453) the end's weight is w = (dO - iso) / (dO - d) at either end, and the
// sample's gradient -w / (dO - d) * (pO - p) . gv.
template <typename S, bool DEF>
__device__ __forceinline__ Grad<S> edge_adjoint(V3<S> c, int axis, S dir, S d, S dO, V3<S> f, V3<S> fO, S iso, V3<S> gv) {
    const EdgeQuot<S> q(dO - d);
    const S w = q.of(dO - iso);
    S dot;
    if (DEF) {
        const S sx = ((c.x + (axis == 0 ? dir : S(0))) + fO.x) - (c.x + f.x);
        const S sy = ((c.y + (axis == 1 ? dir : S(0))) + fO.y) - (c.y + f.y);
        const S sz = ((c.z + (axis == 2 ? dir : S(0))) + fO.z) - (c.z + f.z);
        dot = sx * gv.x + sy * gv.y + sz * gv.z;
    } else {
        dot = dir * (axis == 0 ? gv.x : (axis == 1 ? gv.y : gv.z));
    }
    const S g = -(q.of(w) * dot);
    if (!DEF) return Grad<S>{g, S(0), S(0), S(0)};
    const bool second = dir < S(0);
    const S t = clamp01<S>(second ? w : q.of(iso - d)), wt = second ? t : S(1) - t;
    return Grad<S>{g, wt * gv.x, wt * gv.y, wt * gv.z};
}

// Zeros p[a..b), by one wave: 16-byte stores between the aligned ends.
template <typename S>
__device__ __forceinline__ void fill_zero(S *__restrict__ p, int64_t a, int64_t b, int lane) {
    typedef S vec __attribute__((ext_vector_type(16 / sizeof(S))));
    constexpr int N = 16 / (int)sizeof(S);
    const int64_t mis = (int64_t)(((uintptr_t)p / sizeof(S)) % N);  // elements past a 16-byte boundary
    int64_t a1 = (a + mis + N - 1) / N * N - mis, b1 = (b + mis) / N * N - mis;
    if (a1 >= b1) a1 = b1 = b;
    if (a + lane < a1) put(p + a + lane, S(0));  // fewer than N elements, or (no aligned part) the whole
    for (int64_t i = a + kWave + lane; i < a1; i += kWave) put(p + i, S(0));
    for (int64_t i = a1 + (int64_t)lane * N; i < b1; i += kWave * N) put(reinterpret_cast<vec *>(p + i), vec(S(0)));
    if (b1 + lane < b) put(p + b1 + lane, S(0));
}

// The gather's blocks are single waves, so that none waits for another's share. Per kBwdGroup
// segments there is one that zeroes the gradients of the segments without a touched vertex (the
// vector-memory counter is in order and covers stores: a gathering wave that issued these stores
// would wait for them), and kBwdParts for each tile of at most kBwdTile segments, which gather 64
// touched vertices at a time in turn (a tile of a surface that runs along z holds up to 512). On
// 256^3 noisy / 203x256x181 smooth: tiles of 8 in one part 131 / 64 us, in two 127 / 60, in four 148 /
// 64; tiles of 4 in one part 129 / 60, of 16 149 / 83; groups of 64, 32, 16 segments 127 / 60,
// 128 / 55, 132 / 57. (A recomputing wave does not share a tile: each would recompute the planes. A tile
// of one segment has no second 64 vertices.) Small grids want smaller tiles (the tuned run lengths): one
// wave's chain of chunks is the kernel's time there. 32^3 noisy, tiles of 1, 2, 4, 8: 5.2, 6.3, 7.0, 10.1
// us; 64^3 19.9, 19.9, 11.4, 11.4.
constexpr int kBwdTile = 8;
constexpr int kBwdGroup = 32;
template <bool RECOMP>
constexpr int kBwdParts = RECOMP ? 1 : 2;

// LDS of a gathering wave.
template <typename S>
struct BwdLds {
    uint64_t pl[kBwdTile][10];   // crossing planes: X, Y, Z of the segment, of rows -x, -y; Z of the previous chunk
    int64_t at[kBwdTile];        // index of the sample at the segment's position 0 (as if it were stored)
    int32_t base[kBwdTile][3];   // first vertex of the segment, of rows -x, -y, relative to the tile's first
    int32_t px[kBwdTile], py[kBwdTile], z0[kBwdTile];  // its row, and its first z
    uint32_t rows[kBwdTile];     // which neighbour rows are stored: +x, +y, -x, -y in bits 0, 1, 3, 4
    int64_t idx[kWave];          // the chunk's vertices: sample index, integer position
    S pos[3][kWave];
    int32_t id[3][kWave];        // and first vertex ids: own edges, the x edge of -x, the y edge of -y
    uint16_t list[kWave];        // the vertices: segment << 6 | position
    uint16_t item[kWave * 6];    // vertex | slot << 6 | other end stored << 9 | id offset + 1 << 10
    Grad<S> res[2 * kWave];      // one round of item results
};

// Whether segment t (-1: none) owns a crossing edge.
__device__ __forceinline__ bool seg_owns_crossing(const SegBase *__restrict__ seg, int64_t t) {
    return t >= 0 && seg[t + 1].v != seg[t].v;
}

// The edges incident to a segment's vertices are owned by the segment itself, by the segments of
// rows -x and -y, and (the z edge into lane 0) by the previous chunk: whether any of them owns a
// crossing edge.
__device__ __forceinline__ bool seg_touched(const SegBase *__restrict__ seg, const Geo &g, int64_t s, SegPos sp) {
    return seg_owns_crossing(seg, s) || (sp.px > 0 && seg_owns_crossing(seg, s - xstride(g))) ||
           (sp.py > 0 && seg_owns_crossing(seg, s - g.nchunk)) ||
           (sp.chunk > 0 && seg_owns_crossing(seg, s - 1));
}

__device__ __forceinline__ float from_lane(float v, int lane4) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute(lane4, __float_as_int(v)));
}
__device__ __forceinline__ double from_lane(double v, int lane4) {
    return __hiloint2double(__builtin_amdgcn_ds_bpermute(lane4, __double2hiint(v)),
                            __builtin_amdgcn_ds_bpermute(lane4, __double2loint(v)));
}

// Index of the first stored sample at or after a segment's first position: the samples of segments
// [a, b) are the contiguous range [sample_start(a), sample_start(b)).
__device__ __forceinline__ int64_t sample_start(const Geo &g, const SegPos &sp) {
    const int64_t plane = (int64_t)g.n1 * g.n2;
    const int x = sp.px - g.off, y = sp.py - g.off, z = sp.chunk * kWave - g.off;
    if (x < 0) return 0;
    if (x >= g.n0) return g.n0 * plane;
    if (y < 0) return x * plane;
    if (y >= g.n1) return (x + 1) * plane;
    return x * plane + (int64_t)y * g.n2 + (z < 0 ? 0 : (z < g.n2 ? z : g.n2));
}

// Inside and below bits of a row's 64 samples from conceptual z0 on, for the wave-uniform row (px,
// py): the load (at a valid address, whatever the row) and the compares. Positions outside the stored
// grid take the pad's bits.
struct SideBits {
    uint64_t in, below;
};
template <typename S>
__device__ __forceinline__ S row_sample(const In<S> &in, int px, int py, int zv) {
    const Geo &g = in.geo;
    const int x = px - g.off, y = py - g.off;
    const bool row = (unsigned)x < (unsigned)g.n0 && (unsigned)y < (unsigned)g.n1;  // uniform
    return in.sdf[(row ? ((int64_t)x * g.n1 + y) * g.n2 : 0) + zv];
}
template <typename S>
__device__ __forceinline__ SideBits row_bits(const In<S> &in, int px, int py, uint64_t zs, S v) {
    const Geo &g = in.geo;
    const bool row = (unsigned)(px - g.off) < (unsigned)g.n0 && (unsigned)(py - g.off) < (unsigned)g.n1;
    const uint64_t st = row ? zs : 0ull, pi = in.pad >= in.iso ? ~0ull : 0ull, pb = in.pad < in.iso ? ~0ull : 0ull;
    return SideBits{(__ballot(v >= in.iso) & st) | (pi & ~st), (__ballot(v < in.iso) & st) | (pb & ~st)};
}
__device__ __forceinline__ uint64_t cross_bits(SideBits a, SideBits b) { return (a.below & b.in) | (b.below & a.in); }
__device__ __forceinline__ SideBits side_up(SideBits a, SideBits next, int bit) {
    return SideBits{diso_bits::up1(a.in, next.in >> bit), diso_bits::up1(a.below, next.below >> bit)};
}

// The crossing planes of BwdLds::pl from the samples (the recomputing backward), in two steps, so that
// the loads of one segment are in flight while another's are used: the samples of the segment's row
// and of the six around it that own or end its edges, and per lane one of the four positions past
// the segment's ends that count; then the planes, in scalar registers.
struct BwdPlanes {
    uint64_t w[10];
};
template <typename S>
struct BwdRows {
    S c, xp, yp, xm, ym, xmyp, xpym, e;
};
template <typename S>
__device__ __forceinline__ BwdRows<S> recompute_load(const In<S> &in, const SegPos &sp, int lane) {
    const Geo &g = in.geo;
    const int px = sp.px, py = sp.py, z0 = sp.chunk * kWave, z = z0 - g.off + lane;
    const int zv = z < 0 ? 0 : (z < g.n2 ? z : g.n2 - 1);
    BwdRows<S> r;
    r.c = row_sample(in, px, py, zv);
    r.xp = row_sample(in, px + 1, py, zv);
    r.yp = row_sample(in, px, py + 1, zv);
    r.xm = row_sample(in, px - 1, py, zv);
    r.ym = row_sample(in, px, py - 1, zv);
    r.xmyp = row_sample(in, px - 1, py + 1, zv);
    r.xpym = row_sample(in, px + 1, py - 1, zv);
    // lanes 0-2: position z0 + 64 of rows (0,0), (-1,0), (0,-1); the others: position z0 - 1 of row (0,0)
    r.e = sample(in, px - (lane == 1), py - (lane == 2), lane < 3 ? z0 + kWave : z0 - 1);
    return r;
}
template <typename S>
__device__ __forceinline__ BwdPlanes recompute_planes(const In<S> &in, const SegPos &sp, const BwdRows<S> &v) {
    const Geo &g = in.geo;
    const int px = sp.px, py = sp.py, z0 = sp.chunk * kWave;
    const uint64_t zs = diso_bits::low_bits(g.n2 + g.off - z0) & ~diso_bits::low_bits(g.off - z0);
    const SideBits c = row_bits(in, px, py, zs, v.c), xp = row_bits(in, px + 1, py, zs, v.xp),
                   yp = row_bits(in, px, py + 1, zs, v.yp), xm = row_bits(in, px - 1, py, zs, v.xm),
                   ym = row_bits(in, px, py - 1, zs, v.ym), xmyp = row_bits(in, px - 1, py + 1, zs, v.xmyp),
                   xpym = row_bits(in, px + 1, py - 1, zs, v.xpym);
    const SideBits eb{__ballot(v.e >= in.iso), __ballot(v.e < in.iso)};
    const uint64_t am = diso_bits::low_bits(g.g2 - 1 - z0);  // positions that anchor a cell
    const bool ax = px < g.g0 - 1, ay = py < g.g1 - 1;
    const uint64_t m00 = ax && ay ? am : 0ull, mx = px > 0 && ay ? am : 0ull, my = py > 0 && ax ? am : 0ull;
    BwdPlanes r;
    r.w[0] = cross_bits(c, xp) & m00;
    r.w[1] = cross_bits(c, yp) & m00;
    r.w[2] = cross_bits(c, side_up(c, eb, 0)) & m00;
    r.w[3] = cross_bits(xm, c) & mx;
    r.w[4] = cross_bits(xm, xmyp) & mx;
    r.w[5] = cross_bits(xm, side_up(xm, eb, 1)) & mx;
    r.w[6] = cross_bits(ym, xpym) & my;
    r.w[7] = cross_bits(ym, c) & my;
    r.w[8] = cross_bits(ym, side_up(ym, eb, 2)) & my;
    const SideBits prev{eb.in >> 3, eb.below >> 3};
    // the edge from z0 - 1 (in a previous chunk's top position)
    r.w[9] = sp.chunk > 0 && ax && ay && (cross_bits(prev, c) & 1) && z0 - 1 < g.g2 - 1 ? 1ull << 63 : 0ull;
    return r;
}

// Gather of up to 64 touched vertices (the first nv of L.list): lane k's gradients.
template <typename S, bool DEF>
__device__ __forceinline__ Grad<S> bwd_chunk(const In<S> &in, const AdjIn<S> &adj, int64_t vbase, int nv, BwdLds<S> &L,
                                             int lane) {
    const Geo &g = in.geo;
    const int w = L.list[lane < nv ? lane : 0], j = w >> 6, l = w & 63;
    const uint64_t *pl = L.pl[j];
    const RowEdges e00{pl[0], pl[1], pl[2]}, em0{pl[3], pl[4], pl[5]}, e0m{pl[6], pl[7], pl[8]};
    const uint64_t b = (1ull << l) - 1;
    const int x = bit_at(e00.X, l), y = bit_at(e00.Y, l), z = bit_at(e00.Z, l);
    const int xm = bit_at(em0.X, l), ym = bit_at(e0m.Y, l), zm = bit_at(diso_bits::down1(e00.Z, pl[9]), l);
    const int mask = lane < nv ? x | y << 1 | z << 2 | xm << 3 | ym << 4 | zm << 5 : 0;
    const int64_t idx = L.at[j] + l;
    const int zs = L.z0[j] + l - g.off;
    L.idx[lane] = idx;
    if (DEF) {
        L.pos[0][lane] = S(L.px[j]);
        L.pos[1][lane] = S(L.py[j]);
        L.pos[2][lane] = S(L.z0[j] + l);
    }
    L.id[0][lane] = L.base[j][0] + e00.below(b);
    L.id[1][lane] = L.base[j][1] + em0.below(b);
    L.id[2][lane] = L.base[j][2] + e0m.below(b) + bit_at(e0m.X, l);
    // the other end is a stored sample (else it is the pad)
    const uint32_t ok = L.rows[j] | (zs + 1 < g.n2 ? 4u : 0u) | (zs > 0 ? 32u : 0u);
    const uint32_t cB = (uint32_t)__popc(mask), iB = wave_incl_dpp(cB);
    const int first = (int)(iB - cB), last = (int)iB, total = __builtin_amdgcn_readlane((int)iB, kWave - 1);
    {
        const int off[6] = {1, 1 + x, 1 + x + y, 1, 1, 0};  // id offset + 1
        int r = first;
#pragma unroll
        for (int sl = 0; sl < 6; ++sl)
            if ((mask >> sl) & 1) L.item[r++] = (uint16_t)(lane | sl << 6 | (int)((ok >> sl) & 1) << 9 | off[sl] << 10);
    }
    wave_lds_sync();

    const int64_t sy = g.n2, sx = (int64_t)g.n1 * g.n2;
    // Adjoint of item k (an edge and its end that is the vertex).
    auto item = [&](int k) {
        const int it = L.item[k], src = it & 63, slot = (it >> 6) & 7, end = slot >= 3, axis = end ? slot - 3 : slot;
        const bool st = (it >> 9) & 1;
        const int64_t i0 = L.idx[src], step = axis == 0 ? sx : (axis == 1 ? sy : 1);
        const int64_t i1 = st ? (end ? i0 - step : i0 + step) : i0;
        const int id = L.id[slot == 3 ? 1 : (slot == 4 ? 2 : 0)][src] + (it >> 10) - 1;
        const S d = in.sdf[i0], dO = in.sdf[i1];
        V3<S> c = {S(0), S(0), S(0)}, f = c, fO = c;
        if (DEF) {
            c = V3<S>{L.pos[0][src], L.pos[1][src], L.pos[2][src]};
            const S *p0 = in.deform + 3 * i0, *p1 = in.deform + 3 * i1;
            f = V3<S>{p0[0], p0[1], p0[2]};
            const S u0 = p1[0], u1 = p1[1], u2 = p1[2];
            fO = V3<S>{st ? u0 : S(0), st ? u1 : S(0), st ? u2 : S(0)};
        }
        const V3<S> gv = load_adj(adj, vbase + id);
        return edge_adjoint<S, DEF>(c, axis, end ? S(-1) : S(1), d, st ? dO : in.pad, f, fO, in.iso, gv);
    };
    Grad<S> acc = {S(0), S(0), S(0), S(0)};
    // Rounds of up to 128 items: with more than 64 left, each lane takes two (the second clamped
    // to the last item, its result unused), so both gathers are in flight together.
    for (int r = 0; r < total; r += 2 * kWave) {
        if (r + kWave < total) {  // wave-uniform
            const int k1 = r + kWave + lane < total ? r + kWave + lane : total - 1;
            const Grad<S> r0 = item(r + lane), r1 = item(k1);
            L.res[lane] = r0;
            L.res[kWave + lane] = r1;
        } else if (r + lane < total) {
            L.res[lane] = item(r + lane);
        }
        wave_lds_sync();
        const int lo = first > r ? first : r, hi = last < r + 2 * kWave ? last : r + 2 * kWave;
        for (int k = lo; k < hi; ++k) {  // this lane's items of the round, in slot order
            const Grad<S> q = L.res[k - r];
            acc.g += q.g;
            acc.dx += q.dx;
            acc.dy += q.dy;
            acc.dz += q.dz;
        }
        wave_lds_sync();
    }
    return acc;
}

// What a lane knows of its segment in the backward: its place, its stored positions and the index of
// the sample at its position 0.
struct BwdSeg {
    SegPos sp;
    uint64_t have;
    int64_t at;
    uint32_t rows;
};
template <typename S>
__device__ __forceinline__ BwdSeg bwd_seg(const In<S> &in, int64_t s, bool valid) {
    const Geo &g = in.geo;
    BwdSeg r;
    r.sp = seg_pos(g, s);
    const int x = r.sp.px - g.off, y = r.sp.py - g.off, z = r.sp.chunk * kWave - g.off;
    const bool row = (unsigned)x < (unsigned)g.n0 && (unsigned)y < (unsigned)g.n1;
    r.have = row && valid ? diso_bits::low_bits(g.n2 - z) & ~diso_bits::low_bits(-z) : 0ull;
    r.at = ((int64_t)x * g.n1 + y) * g.n2 + z;
    r.rows = (x + 1 < g.n0 ? 1u : 0u) | (y + 1 < g.n1 ? 2u : 0u) | (x > 0 ? 8u : 0u) | (y > 0 ? 16u : 0u);
    return r;
}

// Crossing planes of lane i's segment s, as BwdLds::pl.
__device__ __forceinline__ BwdPlanes stored_planes(const SegCtx &sc, const Geo &g, int64_t s, const SegPos &sp) {
    BwdPlanes r;
    const bool rx = sp.px > 0, ry = sp.py > 0;
    const int64_t sm0 = rx ? s - xstride(g) : s, s0m = ry ? s - g.nchunk : s;
    const Plane2 a = sc.xy[s], b = sc.xy[sm0], c = sc.xy[s0m];
    const uint64_t az = sc.za[s].a, bz = sc.za[sm0].a, cz = sc.za[s0m].a;
    r.w[0] = a.a, r.w[1] = a.b, r.w[2] = az;
    r.w[3] = rx ? b.a : 0, r.w[4] = rx ? b.b : 0, r.w[5] = rx ? bz : 0;
    r.w[6] = ry ? c.a : 0, r.w[7] = ry ? c.b : 0, r.w[8] = ry ? cz : 0;
    r.w[9] = sp.chunk > 0 ? sc.za[s - 1].a : 0ull;
    return r;
}
// Positions with an incident crossing edge.
__device__ __forceinline__ uint64_t touched_bits(const uint64_t *w) {
    return w[0] | w[1] | w[2] | w[3] | w[7] | diso_bits::down1(w[2], w[9]);
}

// Zero gradients of those of kBwdGroup segments from lo on that the gathering waves leave out (the samples of
// consecutive segments are contiguous, so runs of them are zeroed together).
template <typename S, bool DEF, bool RECOMP>
__device__ __forceinline__ void bwd_zero(const In<S> &in, const SegCtx &sc, int64_t lo, S *__restrict__ adj_sdf,
                                         S *__restrict__ adj_deform, int lane) {
    const Geo &g = in.geo;
    const int64_t all = (int64_t)g.n0 * g.n1 * g.n2, s = lo + lane;
    const int n = g.nseg - lo < kBwdGroup ? (int)(g.nseg - lo) : kBwdGroup;
    const BwdSeg q = bwd_seg(in, lane < n ? s : lo, lane < n);
    bool touched = false;
    if (lane < n)
        touched = RECOMP ? q.have && seg_touched(sc.seg, g, s, q.sp)
                         : (touched_bits(stored_planes(sc, g, s, q.sp).w) & q.have) != 0;
    const int64_t start = lane < n ? sample_start(g, q.sp) : all;
    const int64_t end = lo + n < g.nseg ? sample_start(g, seg_pos(g, lo + n)) : all;
    for (uint64_t idle = ~__ballot(touched) & diso_bits::low_bits(n); idle;) {  // wave-uniform
        const int a = (int)__builtin_ctzll(idle);
        const uint64_t rest = ~(idle >> a);
        const int len = rest ? (int)__builtin_ctzll(rest) : kWave;
        const int64_t i0 = readlane64(start, a), i1 = a + len < n ? readlane64(start, a + len) : end;
        fill_zero(adj_sdf, i0, i1, lane);
        if (DEF) fill_zero(adj_deform, 3 * i0, 3 * i1, lane);
        idle &= ~(diso_bits::low_bits(len) << a);
    }
}

// Gather of the segments [lo, lo + n) of a grid (n <= kBwdTile) by one wave: 64 of their touched
// vertices at a time, each segment's gradients then written as a row, zeros included.
template <typename S, bool DEF, bool RECOMP>
__device__ __forceinline__ void bwd_tile(const In<S> &in, const SegCtx &sc, int64_t lo, int n, const AdjIn<S> &adj,
                                         S *__restrict__ adj_sdf, S *__restrict__ adj_deform, BwdLds<S> &L, int part, int lane) {
    const Geo &g = in.geo;
    const bool acc = (adj.flags & DISO_FLAG_ACCUMULATE) != 0;
    const int64_t s = lo + (lane < n ? lane : 0);  // lane i: segment lo + i
    const BwdSeg q = bwd_seg(in, s, lane < n);
    const int64_t sm0 = q.sp.px > 0 ? s - xstride(g) : s, s0m = q.sp.py > 0 ? s - g.nchunk : s;
    const int64_t v00 = sc.seg[s].v, vm0 = sc.seg[sm0].v, v0m = sc.seg[s0m].v;  // (issued with the planes)
    uint64_t cand, T = 0;
    if constexpr (RECOMP) {
        // the planes from the samples, for the segments that can have a touched vertex (by the bases)
        cand = __ballot(q.have && seg_touched(sc.seg, g, s, q.sp));
        if (cand) {
            int j = (int)__builtin_ctzll(cand);
            BwdRows<S> rows = recompute_load(in, pos_of_lane(q.sp, j), lane);
            for (uint64_t c = cand & (cand - 1);; c &= c - 1) {  // wave-uniform
                const BwdRows<S> cur = rows;
                const int at = j;
                if (c) {
                    j = (int)__builtin_ctzll(c);
                    rows = recompute_load(in, pos_of_lane(q.sp, j), lane);
                }
                const BwdPlanes p = recompute_planes(in, pos_of_lane(q.sp, at), cur);
                if (lane == 0)
                    for (int k = 0; k < 10; ++k) L.pl[at][k] = p.w[k];
                if (!c) break;
            }
        }
        wave_lds_sync();
        if ((cand >> lane) & 1) T = touched_bits(L.pl[lane]) & q.have;
    } else {
        const BwdPlanes p = stored_planes(sc, g, s, q.sp);
        T = touched_bits(p.w) & q.have;
        cand = __ballot(T != 0);
        if (lane < n)
            for (int k = 0; k < 10; ++k) L.pl[lane][k] = p.w[k];
    }
    if (!cand) return;
    const int64_t v0 = readlane64(v00, 0);
    if (lane < n) {
        L.at[lane] = q.at;
        L.px[lane] = q.sp.px;
        L.py[lane] = q.sp.py;
        L.z0[lane] = q.sp.chunk * kWave;
        L.rows[lane] = q.rows;
        L.base[lane][0] = (int32_t)(v00 - v0);
        L.base[lane][1] = (int32_t)(vm0 - v0);
        L.base[lane][2] = (int32_t)(v0m - v0);
    }
    const uint32_t cT = (uint32_t)__popcll(T), iT = wave_incl_dpp(cT);
    const int pre = (int)(iT - cT), total = __builtin_amdgcn_readlane((int)iT, kWave - 1);
    for (int c0 = part * kWave; c0 < total || (RECOMP && c0 == 0); c0 += kBwdParts<RECOMP> * kWave) {  // wave-uniform
        const int nv = total - c0 < kWave ? total - c0 : kWave;
        const uint64_t segs = __ballot(T != 0 && pre < c0 + nv && (int)iT > c0);
        for (uint64_t a = segs; a; a &= a - 1) {
            const int j = (int)__builtin_ctzll(a);
            const uint64_t t = (uint64_t)readlane64((int64_t)T, j);
            const int k = __builtin_amdgcn_readlane(pre, j) - c0 + lanes_below(t);
            if (__builtin_amdgcn_inverse_ballot_w64(t) && k >= 0 && k < kWave) L.list[k] = (uint16_t)(j << 6 | lane);
        }
        wave_lds_sync();
        Grad<S> r = {S(0), S(0), S(0), S(0)};
        if (nv > 0) r = bwd_chunk<S, DEF>(in, adj, v0 - sc.v0, nv, L, lane);
        // rows of the segments with a vertex in the chunk (and, with the first chunk, of those that
        // turned out to have none)
        for (uint64_t a = segs | (RECOMP && c0 == 0 && !acc ? cand & ~__ballot(T != 0) : 0ull); a; a &= a - 1) {
            const int j = (int)__builtin_ctzll(a);
            const uint64_t t = (uint64_t)readlane64((int64_t)T, j), h = (uint64_t)readlane64((int64_t)q.have, j);
            const int at = __builtin_amdgcn_readlane(pre, j) - c0, k = at + lanes_below(t);
            const int from = (k & (kWave - 1)) << 2;
            Grad<S> w;
            w.g = from_lane(r.g, from);
            if (DEF) {
                w.dx = from_lane(r.dx, from);
                w.dy = from_lane(r.dy, from);
                w.dz = from_lane(r.dz, from);
            }
            const bool mine = __builtin_amdgcn_inverse_ballot_w64(t) && k >= 0 && k < nv;
            const bool zero = at >= 0 && __builtin_amdgcn_inverse_ballot_w64(h & ~t);  // with the segment's first vertex
            const int64_t i = readlane64(q.at, j) + lane;
            if (acc) {
                if (mine) {
                    adj_sdf[i] += w.g;
                    if (DEF) {
                        adj_deform[3 * i + 0] += w.dx;
                        adj_deform[3 * i + 1] += w.dy;
                        adj_deform[3 * i + 2] += w.dz;
                    }
                }
            } else if (mine || zero) {
                put(adj_sdf + i, mine ? w.g : S(0));
                if (DEF) {
                    put(adj_deform + 3 * i + 0, mine ? w.dx : S(0));
                    put(adj_deform + 3 * i + 1, mine ? w.dy : S(0));
                    put(adj_deform + 3 * i + 2, mine ? w.dz : S(0));
                }
            }
        }
        wave_lds_sync();
    }
}

// Block k of the blocks of one grid (bwd_blocks of them).
template <typename S, bool DEF, bool RECOMP>
__device__ __forceinline__ void bwd_wave(const In<S> &in, const SegCtx &sc, int64_t k, int tile, const AdjIn<S> &adj,
                                         S *__restrict__ adj_sdf, S *__restrict__ adj_deform) {
    __shared__ BwdLds<S> s_lds;
    const int lane = threadIdx.x, parts = tile > 1 ? kBwdParts<RECOMP> : 1, per = kBwdGroup / tile * parts + 1;
    const int64_t group = k / per;
    const int i = (int)(k - group * per);
    if (i == 0) {
        if (!(adj.flags & DISO_FLAG_ACCUMULATE)) bwd_zero<S, DEF, RECOMP>(in, sc, group * kBwdGroup, adj_sdf, adj_deform, lane);
        return;
    }
    const int64_t lo = group * kBwdGroup + (i - 1) / parts * tile, left = in.geo.nseg - lo;
    if (left > 0) bwd_tile<S, DEF, RECOMP>(in, sc, lo, (int)(left < tile ? left : tile), adj, adj_sdf, adj_deform, s_lds, (i - 1) % parts, lane);
}

template <typename S, bool DEF, bool RECOMP>
__global__ __launch_bounds__(kWave) void bwd_mc_kernel(In<S> in, const SegBase *__restrict__ seg, AdjIn<S> adj,
                                                       S *__restrict__ adj_sdf, S *__restrict__ adj_deform,
                                                       int tile, int64_t nblocks) {
    const SegCtx sc = seg_ctx(seg, planes_of(seg, in.geo.nseg));
    const int64_t b = xcd_stripe(block_number(), nblocks);
    if (b < nblocks) bwd_wave<S, DEF, RECOMP>(in, sc, b, tile, adj, adj_sdf, adj_deform);
}

// A quad's four indices in 16-byte loads (any address an index may have).
typedef int64_t Index2 __attribute__((ext_vector_type(2), aligned(8)));
typedef int32_t Index4 __attribute__((ext_vector_type(4), aligned(4)));
struct QuadIds {
    Index2 a, b;
};
__device__ __forceinline__ QuadIds load_quad(const void *__restrict__ quads, int64_t q, int flags) {
    if (flags & DISO_FLAG_INDEX64) {
        const Index2 *p = reinterpret_cast<const Index2 *>(static_cast<const int64_t *>(quads) + 4 * q);
        return QuadIds{p[0], p[1]};
    }
    const Index4 v = *reinterpret_cast<const Index4 *>(static_cast<const int32_t *>(quads) + 4 * q);
    return QuadIds{Index2{v.x, v.y}, Index2{v.z, v.w}};
}

// Per-edge upstream gradient of a DMC forward: ge[q] = sum over the quad's corners v of
// (dL/dv) / (edges in v's patch), corners in the quad's order, for a wave's 64 quads from q0 on. Bound
// by the latency of the gather: a corner out of range adds nothing, but loads row 0, so that all four
// corners' loads are in flight together (a branch around each: 256^3 noisy 63 us, 512^3 123; so 59,
// 118). The quads are read once, by non-temporal loads, so that they do not displace what the gather
// after this re-reads (with ordinary loads it takes 136 us, so 120); 64-bit ones pass through LDS, each
// load covering whole lines (without that, 63 us, and a batch's 381 instead of 321).
template <typename S>
__device__ __forceinline__ void edge_grad_wave(const void *__restrict__ quads, int64_t q0, int64_t n,
                                               const uint8_t *__restrict__ vinfo, const AdjIn<S> &adj, const S *s_rcp,
                                               Index2 *s_quad, S *__restrict__ ge) {
    const bool compat = (adj.flags & DISO_FLAG_REFERENCE_COMPAT) != 0;
    const int lane = threadIdx.x % kWave;
    const int64_t q = q0 + lane, left = n - q0;
    if (left <= 0) return;  // wave-uniform
    QuadIds w;
    if (adj.flags & DISO_FLAG_INDEX64) {
        const Index2 *p = reinterpret_cast<const Index2 *>(static_cast<const int64_t *>(quads) + 4 * q0);
        const int last = left < kWave ? 2 * (int)left - 1 : 2 * kWave - 1;
        s_quad[lane] = __builtin_nontemporal_load(p + (lane < last ? lane : last));
        s_quad[lane + kWave] = __builtin_nontemporal_load(p + (lane + kWave < last ? lane + kWave : last));
        wave_lds_sync();
        w = QuadIds{s_quad[2 * lane], s_quad[2 * lane + 1]};
    } else {
        const Index4 *p = reinterpret_cast<const Index4 *>(static_cast<const int32_t *>(quads) + 4 * q0);
        const Index4 v = __builtin_nontemporal_load(p + (lane < left ? lane : 0));
        w = QuadIds{Index2{v.x, v.y}, Index2{v.z, v.w}};
    }
    const int64_t qv[4] = {w.a.x, w.a.y, w.b.x, w.b.y};
    V3<S> sum = {S(0), S(0), S(0)};
    if (adj.n > 0) {  // uniform
        int64_t at[4];
        bool ok[4];
        int info[4];
        V3<S> a[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            ok[k] = (qv[k] >= 0) & (qv[k] < adj.n);
            at[k] = ok[k] ? qv[k] : 0;
            info[k] = vinfo[at[k]];
        }
        if (compat) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int64_t first = at[k] - (info[k] >> 3);
                ok[k] &= first >= 0;
                at[k] = first >= 0 ? first : 0;
            }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) a[k] = load_adj_at(adj, at[k]);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const S r = s_rcp[info[k] & 7];
            sum.x += ok[k] ? a[k].x * r : S(0);
            sum.y += ok[k] ? a[k].y * r : S(0);
            sum.z += ok[k] ? a[k].z * r : S(0);
        }
    }
    if (lane >= left) return;
    ge[3 * q + 0] = sum.x;
    ge[3 * q + 1] = sum.y;
    ge[3 * q + 2] = sum.z;
}

template <typename S>
__global__ __launch_bounds__(kBlock) void dmc_edge_grad_kernel(const void *__restrict__ quads, int64_t nq,
                                                               const SegBase *__restrict__ tot,
                                                               const uint8_t *__restrict__ vinfo, AdjIn<S> adj,
                                                               S *__restrict__ ge) {
    __shared__ S s_rcp[8];
    __shared__ Index2 s_quad[kWavesPerBlock][2 * kWave];
    if (threadIdx.x < 8) s_rcp[threadIdx.x] = threadIdx.x ? S(1) / S(threadIdx.x) : S(0);
    __syncthreads();
    // nq may be a capacity: the quads are the first tot->v rows (the count pass's total)
    const int64_t n = tot->v < nq ? tot->v : nq;
    // each XCD takes a contiguous eighth of the quads, so the vertex rows a quad shares with the
    // quads of the previous plane are still in that XCD's L2
    const int64_t q0 = xcd_block(blockIdx.x, gridDim.x) * kBlock + wave_id() * kWave;
    edge_grad_wave(quads, q0, n, vinfo, adj, s_rcp, s_quad[wave_id()], ge);
}

// ------------------------------------------------------------------------------------------
// Batched extraction: many grids (uneven dims, MC and DMC, with or without deform) per launch.
//
// The count pass runs once over the concatenation of all grids' segments (a grid's segments are
// consecutive, grids in batch order), so one single-pass scan yields every grid's bases; a grid's
// own output rows are its bases minus those of its first segment. Emission and backward launch
// blocks of one grid: a launch covers the blocks of every grid of one kind (algorithm x deform x
// recompute), listed in `gl` with the prefix of their block counts in `rf`; a block finds its grid
// by binary search over `rf`.

template <typename S>
__device__ __forceinline__ SegCtx batch_ctx(const BatchGrid<S> &G, const SegBase *seg, const Planes &q) {
    const int64_t f = G.seg_first;
    return SegCtx{seg + f, q.xy + f, q.za + f, seg[f].v, seg[f].f};
}

template <typename S>
__global__ void batch_totals_kernel(const BatchGrid<S> *__restrict__ grids, int n, int64_t nseg,
                                    const SegBase *__restrict__ seg, Planes planes, uint32_t *__restrict__ gflags,
                                    uint32_t *__restrict__ range, diso_totals_t *__restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const SegBase a = seg[grids[i].seg_first], e = seg[i + 1 < n ? grids[i + 1].seg_first : nseg];
    const int64_t cross = e.v - a.v, faces = e.f - a.f;
    const bool dmc = grids[i].algo == DISO_DMC;
    out[i].n_verts = dmc ? faces : cross;
    out[i].n_faces = dmc ? cross : faces;
    out[i].flags = (int64_t)(gflags[i] | ((uint32_t)seg[nseg + 1].v & DISO_TOTAL_SCAN_TIMEOUT));
    out[i].n_crossing = cross;
    gflags[i] = 0u;  // ready for the next batch
    // the grid's units: from the one that holds its first cell (the last to start before the grid's
    // segments, which may end before them too) to the last that starts in them
    const uint32_t nu = nseg >= 4 ? *planes.nunits : 0u;
    auto lower = [&](int64_t s) {  // units that start before segment s
        uint32_t lo = 0, hi = nu;
        while (lo < hi) {
            const uint32_t mid = lo + (hi - lo) / 2;
            if ((int64_t)planes.unit[mid] < s)
                lo = mid + 1;
            else
                hi = mid;
        }
        return lo;
    };
    const uint32_t u0 = lower(grids[i].seg_first), u1 = lower(i + 1 < n ? grids[i + 1].seg_first : nseg);
    range[2 * i] = u0 > 0 ? u0 - 1 : 0u;
    range[2 * i + 1] = u1;
}

// Batched emission: a grid's blocks go through its units in turn. Units are of the whole batch, so a
// grid's first and last may hold cells of its neighbours too (unit_cells leaves them out). tables(geo)
// fills the block's tables.
template <typename S, typename T, typename F>
__device__ __forceinline__ void batch_units(const BatchGrid<S> *__restrict__ grids, const int32_t *__restrict__ gl,
                                            const int64_t *__restrict__ rf, int m, const SegBase *__restrict__ seg,
                                            const Planes &planes, const uint32_t *__restrict__ range, int64_t nblocks,
                                            int wave, int lane, T tables, F f) {
    if (block_number() >= nblocks) return;
    const int64_t b = xcd_block(block_number(), nblocks);
    const int j = find_group(rf, m, b);
    const int gi = gl[j];
    const BatchGrid<S> &B = grids[gi];
    if (B.nv > B.vcap || B.nf > B.fcap) return;
    const In<S> in = B.in;
    tables(in.geo);
    __syncthreads();
    const int64_t first = B.seg_first;
    const UnitGrid G{seg, planes, first, first + in.geo.nseg - 1, seg[first].v, seg[first].f};
    const OutCfg out{B.flags, B.vcap, B.fcap};
    const uint32_t nunits = *planes.nunits, hi = range[2 * gi + 1], step = (uint32_t)(rf[j + 1] - rf[j]) * kWavesPerBlock;
    unit_loop(G, range[2 * gi] + (uint32_t)(b - rf[j]) * kWavesPerBlock + (uint32_t)wave, hi, step, 0, nunits, lane,
              [&](const UnitLoad &U, auto next) { return f(in, G, B, out, U, next); });
}

template <typename S, bool DEF>
__global__ __launch_bounds__(kBlock, 6) void emit_mc_batch_kernel(const BatchGrid<S> *__restrict__ grids,
                                                               const int32_t *__restrict__ gl,
                                                               const int64_t *__restrict__ rf, int m,
                                                               const SegBase *__restrict__ seg, Planes planes,
                                                               const uint32_t *__restrict__ range, int64_t nblocks) {
    __shared__ uint64_t s_case[256];
    __shared__ McEmitLds s_lds[kWavesPerBlock];
    const int wave = wave_id(), lane = threadIdx.x % kWave;
    batch_units(grids, gl, rf, m, seg, planes, range, nblocks, wave, lane, [&](const Geo &) { load_mc_cases(s_case); },
                [&](const In<S> &in, const UnitGrid &G, const BatchGrid<S> &B, const OutCfg &out, const UnitLoad &U, auto next) {
                    return emit_mc_unit<S, DEF>(in, G, U, next, B.verts, B.faces, out, B.nm, s_case, s_lds[wave], lane);
                });
}

template <typename S, bool DEF>
__global__ __launch_bounds__(kBlock, 5) void emit_dmc_batch_kernel(const BatchGrid<S> *__restrict__ grids,
                                                                const int32_t *__restrict__ gl,
                                                                const int64_t *__restrict__ rf, int m,
                                                                const SegBase *__restrict__ seg, Planes planes,
                                                                const uint32_t *__restrict__ range, int64_t nblocks) {
    __shared__ DmcTables<S> s_tab;
    __shared__ DmcEmitLds<S> s_lds[kWavesPerBlock];
    const int wave = wave_id(), lane = threadIdx.x % kWave;
    batch_units(grids, gl, rf, m, seg, planes, range, nblocks, wave, lane, [&](const Geo &g) { s_tab.load(g); },
                [&](const In<S> &in, const UnitGrid &G, const BatchGrid<S> &B, const OutCfg &out, const UnitLoad &U, auto next) {
                    return emit_dmc_unit<S, DEF>(in, G, U, next, (S *)B.verts, B.faces, B.vinfo, out, B.nm, s_tab, s_lds[wave], lane);
                });
}

// Per-edge upstream gradients of every DMC grid of the batch: blocks of kBlock quads of one grid.
template <typename S>
__global__ __launch_bounds__(kBlock) void dmc_edge_grad_batch_kernel(const BatchGrid<S> *__restrict__ grids,
                                                                     const int32_t *__restrict__ gl,
                                                                     const int64_t *__restrict__ rf, int m,
                                                                     S *__restrict__ ge) {
    __shared__ S s_rcp[8];
    __shared__ Index2 s_quad[kWavesPerBlock][2 * kWave];
    if (threadIdx.x < 8) s_rcp[threadIdx.x] = threadIdx.x ? S(1) / S(threadIdx.x) : S(0);
    __syncthreads();
    const int64_t b = xcd_block(blockIdx.x, gridDim.x);  // as dmc_edge_grad_kernel
    const int j = find_group(rf, m, b);
    const BatchGrid<S> &G = grids[gl[j]];
    const int64_t q0 = (b - rf[j]) * kBlock + wave_id() * kWave;
    const AdjIn<S> a{G.adj, G.nv, G.flags, G.nm};
    edge_grad_wave(G.faces, q0, G.nf, G.vinfo, a, s_rcp, s_quad[wave_id()], ge + 3 * G.q_first);
}

template <typename S, bool DEF, bool RECOMP>
__global__ __launch_bounds__(kWave) void bwd_batch_kernel(const BatchGrid<S> *__restrict__ grids,
                                                           const int32_t *__restrict__ gl,
                                                           const int64_t *__restrict__ rf, int m,
                                                           const SegBase *__restrict__ seg,
                                                           Planes planes,
                                                           const S *__restrict__ ge, int64_t nblocks) {
    const int64_t b = xcd_stripe(block_number(), nblocks);
    if (b >= nblocks) return;
    const int j = find_group(rf, m, b);
    const BatchGrid<S> &G = grids[gl[j]];
    const In<S> in = G.in;
    const SegCtx sc = batch_ctx(G, seg, planes);
    // DMC grids gather the per-edge gradients (already divided by the normalisation)
    const AdjIn<S> adj = G.algo == DISO_DMC ? AdjIn<S>{ge + 3 * G.q_first, G.nf, G.flags & ~DISO_FLAG_NORMALIZE, G.nm}
                                            : AdjIn<S>{G.adj, G.nv, G.flags, G.nm};
    bwd_wave<S, DEF, RECOMP>(in, sc, b - rf[j], G.tile, adj, G.adj_sdf, G.adj_deform);
}

// ------------------------------------------------------------------------------------------
// DiffDMC quad -> triangle split (diso/__init__.py:117-147)
//
// Each quad is cut along the diagonal whose worse triangle has the smaller largest corner cosine:
// cut (0,1,3)+(1,2,3) ("first") when score1 < score2, else (0,1,2)+(0,2,3); the output holds all
// first quads' pairs in quad order, then all the others'. split_score_kernel scores the quads of a
// contiguous range per wave and counts the first ones; split_emit_kernel gives each wave the prefix
// and the total of those counts (a block reads all of them: the grid is ~4 blocks per CU, so 16 KB)
// and writes the pairs in place, 64 quads at a time. The cosine arithmetic is
// F.normalize's (x / max(|x|, 1e-12), |x| = sqrt((x*x + y*y) + z*z)) and a left-to-right dot.

constexpr int kSplitBlock = 256;
constexpr int kSplitWaves = kSplitBlock / kWave;
constexpr int64_t kMaxSplitWaves = 4096;

template <typename S>
__device__ __forceinline__ V3<S> unit(V3<S> v) {
    const S n = sqrt(v.x * v.x + v.y * v.y + v.z * v.z);
    const S d = n < S(1e-12) ? S(1e-12) : n;  // clamp_min(eps); keeps a NaN norm
    return {v.x / d, v.y / d, v.z / d};
}

template <typename S>
__device__ __forceinline__ S nan_max(S a, S b) {  // torch.max / np.maximum: NaN wins
    return (a != a || a > b) ? a : b;
}

// The unit vectors of a quad's six vertex pairs, e[i][j] = unit(p_j - p_i), the others by
// negation: unit(-v) = -unit(v) exactly (same norm, sign-symmetric division), and a dot product
// of negated vectors is the negated dot product exactly, so each corner cosine below has the bits
// of normalising its two edge vectors itself (24 normalisations per quad become 6).
template <typename S>
struct QuadUnits {
    V3<S> e[4][4];
    __device__ __forceinline__ QuadUnits(const V3<S> *p) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = i + 1; j < 4; ++j) {
                e[i][j] = unit(V3<S>{p[j].x - p[i].x, p[j].y - p[i].y, p[j].z - p[i].z});
                e[j][i] = V3<S>{-e[i][j].x, -e[i][j].y, -e[i][j].z};
            }
    }
    // cosine at corner o between the edges to a and to b (u first, then w, left-to-right dot)
    __device__ __forceinline__ S cosine(int o, int a, int b) const {
        const V3<S> &u = e[o][a], &w = e[o][b];
        return u.x * w.x + u.y * w.y + u.z * w.z;
    }
    // largest corner cosine of triangle (a, b, c), corners in the order a, b, c
    // (diso/__init__.py:127-136)
    __device__ __forceinline__ S worst(int a, int b, int c) const {
        return nan_max(nan_max(cosine(a, b, c), cosine(b, c, a)), cosine(c, a, b));
    }
};

template <typename S>
__device__ __forceinline__ V3<S> load_vert(const S *__restrict__ v, int64_t i) {
    return {v[3 * i + 0], v[3 * i + 1], v[3 * i + 2]};
}

typedef uint32_t Count4 __attribute__((ext_vector_type(kSplitWaves), aligned(4)));  // a block's counts

template <typename S>
__global__ __launch_bounds__(kSplitBlock) void split_score_kernel(const S *__restrict__ verts, int64_t nv,
                                                                  const void *__restrict__ quads, int64_t nq,
                                                                  int flags, uint8_t *__restrict__ first,
                                                                  uint32_t *__restrict__ counts, int64_t nranges) {
    const int lane = threadIdx.x % kWave;
    const int64_t r = (int64_t)blockIdx.x * kSplitWaves + wave_id(), lo = r * nq / nranges, hi = (r + 1) * nq / nranges;
    uint32_t cnt = 0;
    for (int64_t q = lo + lane; q < hi; q += kWave) {
        const QuadIds quad = load_quad(quads, q, flags);
        const int64_t id[4] = {quad.a.x, quad.a.y, quad.b.x, quad.b.y};
        bool ok = true;
#pragma unroll
        for (int k = 0; k < 4; ++k) ok &= id[k] >= 0 && id[k] < nv;
        uint8_t f = 0;
        if (ok) {
            const V3<S> p[4] = {load_vert(verts, id[0]), load_vert(verts, id[1]), load_vert(verts, id[2]),
                                load_vert(verts, id[3])};
            const QuadUnits<S> qu(p);
            const S s1 = nan_max(qu.worst(0, 1, 3), qu.worst(1, 2, 3));
            const S s2 = nan_max(qu.worst(0, 1, 2), qu.worst(0, 2, 3));
            f = s1 < s2;
        }
        first[q] = f;
        cnt += f;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) cnt += (uint32_t)__shfl_xor((int)cnt, o, kWave);
    if (lane == 0) counts[r] = cnt;
}

// Bound by its stores, 48 bytes a quad. Storing each lane's pair where it belongs left lines half
// written when the next lane's row went to the other list; the pairs of a wave's 64 quads are
// therefore put in order in LDS and leave as two runs of consecutive 16-byte stores, the next 64
// quads' loads ahead of them. 3.1 million quads of white noise: 89 -> 49 us (200 MB with the quads read
// again, 4.1 TB/s; with ordinary stores 52).
__global__ __launch_bounds__(kSplitBlock) void split_emit_kernel(const void *__restrict__ quads, int64_t nq,
                                                                 int flags, const uint8_t *__restrict__ first,
                                                                 const uint32_t *__restrict__ counts,
                                                                 int64_t nranges, int64_t *__restrict__ tris) {
    __shared__ int64_t s_pre[kSplitWaves], s_tot[kSplitWaves];
    __shared__ Index2 s_row[kSplitWaves][kWave * 3];
    const int tid = threadIdx.x, lane = tid % kWave, wave = wave_id();
    const int64_t r = (int64_t)blockIdx.x * kSplitWaves + wave;
    const int64_t lo = r * nq / nranges, hi = (r + 1) * nq / nranges;
    // First quads in the ranges before this block's, and in all of them.
    int64_t pre = 0, tot = 0;
    const Count4 *blocks = reinterpret_cast<const Count4 *>(counts);
    for (int64_t j = tid; j < nranges / kSplitWaves; j += kSplitBlock) {
        const Count4 k = blocks[j];
        const int64_t c = (int64_t)k.x + k.y + k.z + k.w;
        tot += c;
        pre += j < (int64_t)blockIdx.x ? c : 0;
    }
    const Count4 own = blocks[blockIdx.x];
    pre = wave_sum64(pre);
    tot = wave_sum64(tot);
    if (lane == 0) {
        s_pre[wave] = pre;
        s_tot[wave] = tot;
    }
    __syncthreads();
    int64_t run = 0, n1 = 0;
#pragma unroll
    for (int w = 0; w < kSplitWaves; ++w) {
        run += s_pre[w] + (w < wave ? (int64_t)own[w] : 0);
        n1 += s_tot[w];
    }
    if (lo >= hi) return;
    Index2 *row = s_row[wave];
    auto at = [&](int64_t base) { return base + lane < hi ? base + lane : hi - 1; };
    QuadIds v = load_quad(quads, at(lo), flags);
    uint8_t fb = first[at(lo)];
    for (int64_t base = lo; base < hi; base += kWave) {
        const int n = hi - base < kWave ? (int)(hi - base) : kWave;
        const QuadIds w = v;
        const bool f = fb && lane < n;
        v = load_quad(quads, at(base + kWave), flags);
        fb = first[at(base + kWave)];
        const uint64_t bal = __ballot(f);
        const int nf = (int)__popcll(bal), below = lanes_below(bal);
        // the pair's place among the 64: the first quads' rows, then the others', each in quad order
        Index2 *d = row + 3 * (f ? below : nf + lane - below);
        if (lane < n) {
            d[0] = w.a;
            d[1] = Index2{f ? w.b.y : w.b.x, f ? w.a.y : w.a.x};
            d[2] = w.b;
        }
        wave_lds_sync();
        // rows run.. of the first half, or of the second half at the rank among the others
        Index2 *t1 = reinterpret_cast<Index2 *>(tris + 6 * run);
        Index2 *t2 = reinterpret_cast<Index2 *>(tris + 6 * (n1 + (base - run) - nf));
        for (int i = lane; i < 3 * n; i += kWave) __builtin_nontemporal_store(row[i], (i < 3 * nf ? t1 : t2) + i);  // (8-byte aligned)
        wave_lds_sync();
        run += nf;
    }
}

// ------------------------------------------------------------------------------------------
// Host side

thread_local char g_err[512] = "";

int fail(int code, const char *fmt, ...) __attribute__((format(printf, 2, 3)));
int fail(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

int check_hip(hipError_t e, const char *what) {
    if (e == hipSuccess) return DISO_OK;
    return fail(DISO_E_HIP, "%s: %s", what, hipGetErrorString(e));
}

// Launch parameters (diso_set_param, diso_set_bucket_param): the segments that four waves of the
// backward take and count blocks per CU, each per size bucket, and the recount spins. A launch takes the bucket of
// its segment count (a batched launch: the segments of all its grids); the bucket limits lie
// between the segment counts of cubic grids of 32, 64, 128, 256 and 512 samples per side with
// the virtual pad (1,156 / 8,712 / 50,700 / 332,820 / 2,377,764 segments).
constexpr int kBuckets = DISO_PARAM_BUCKETS;
constexpr int64_t kBucketLimit[kBuckets - 1] = {3200, 21000, 130000, 900000};
struct Params {
    int run[kBuckets] = {32, 32, 32, 32, 32};
    int count_per_cu[kBuckets] = {kCountBlocksPerCU, kCountBlocksPerCU, kCountBlocksPerCU, kCountBlocksPerCU,
                                  kCountBlocksPerCU};
    int recount_spins = 8192;
};
Params g_params;

int bucket_of(int64_t nseg) {
    int b = 0;
    while (b < kBuckets - 1 && nseg > kBucketLimit[b]) ++b;
    return b;
}
int run_for(int64_t nseg) { return g_params.run[bucket_of(nseg)]; }

// Validates a per-bucket parameter value; returns its table (nullptr after fail()).
int *bucket_table(int which, int value) {
    switch (which) {
        case DISO_PARAM_RUN:
            if (value < 1 || value > kMaxRun) {
                fail(DISO_E_INVALID, "run length must be in [1, %d]", kMaxRun);
                return nullptr;
            }
            return g_params.run;
        case DISO_PARAM_COUNT_BLOCKS_PER_CU:
            if (value < 1 || value > kCountBlocksPerCU) {
                fail(DISO_E_INVALID, "count blocks per CU must be in [1, %d]", kCountBlocksPerCU);
                return nullptr;
            }
            return g_params.count_per_cu;
        default:
            fail(DISO_E_INVALID, "parameter %d has no size buckets", which);
            return nullptr;
    }
}

bool make_geo(int64_t X, int64_t Y, int64_t Z, int flags, Geo *g) {
    if (X < 1 || Y < 1 || Z < 1) return false;
    const int64_t lim = 1 << 20;
    if (X > lim || Y > lim || Z > lim) return false;
    const int pad = (flags & DISO_FLAG_VIRTUAL_PAD) ? 2 : 0;
    g->n0 = (int)X;
    g->n1 = (int)Y;
    g->n2 = (int)Z;
    g->g0 = (int)X + pad;
    g->g1 = (int)Y + pad;
    g->g2 = (int)Z + pad;
    g->off = pad / 2;
    g->nchunk = (g->g2 + kWave - 1) / kWave;
    g->nseg = (int64_t)g->g0 * g->g1 * g->nchunk;
    g->rchunk = 1.0 / g->nchunk;
    g->rg1 = 1.0 / g->g1;
    // Per-block aggregates must fit the 29/30-bit fields of the scan words; segment ids 32 bits.
    return (int64_t)g->g0 * g->g1 * g->g2 < (1ll << 36) && g->nseg < (1ll << 32);
}

// Segment bases (+ two totals entries), then the classification planes.
int64_t bases_bytes_for(const Geo &g) { return (g.nseg + 2) * (int64_t)sizeof(SegBase); }
int64_t seg_bytes_for(const Geo &g) { return bases_bytes_for(g) + g.nseg * kSegStateBytes; }
int64_t ctl_bytes_for(const Geo &) { return kCtlHeader + 4 * kMaxCountBlocks * (int64_t)sizeof(uint64_t); }

// Number of count blocks: about kCountBlocksPerCU per CU of the current device, so that every
// block is resident at once, and never more than the segments or the word buffer allow.
int cu_count() {
    static int cus[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
    if (cus[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cus[dev] = n;
    }
    return cus[dev];
}

// Count blocks of one CU that can be resident at once for count-kernel instance `kernel` (the
// single-pass scan wants every block resident; queried once per instance).
template <auto Kernel>
int count_resident_per_cu() {
    static int n = 0;
    if (n == 0) {
        int r = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&r, Kernel, kCountBlock, 0) != hipSuccess || r < 1) r = 1;
        n = r;
    }
    return n;
}

int64_t count_blocks(int64_t nseg, int resident_per_cu) {
    const int want = g_params.count_per_cu[bucket_of(nseg)];
    const int per_cu = want < resident_per_cu ? want : resident_per_cu;
    int64_t nb = (int64_t)cu_count() * per_cu;
    const int64_t min_nb = (nseg + (1ll << 20) - 1) >> 20;  // <= 2^20 segments per block keeps the
    const int64_t full = (nseg + kCountBlock - 1) / kCountBlock;
    if (nb > full) nb = full;   // a lane per segment: no more blocks than full waves
    if (nb < min_nb) nb = min_nb;                          // aggregate fields from overflowing
    if (nb > kMaxCountBlocks) nb = kMaxCountBlocks;
    if (nb > nseg) nb = nseg;
    return nb < 1 ? 1 : nb;
}

// The launch shape of at least `blocks` blocks whose kernel takes them by block_number().
dim3 shape_of(int64_t blocks, int threads) {
    const diso_launch::Shape s = diso_launch::shape_of(blocks, threads);
    return dim3(s.x, s.y);
}

int mask_tile_of(int64_t nseg) {
    return nseg <= (int64_t)cu_count() * kWavesPerBlock * kMaskTile ? kMaskSmallTile : kMaskTile;
}
dim3 mask_shape(int64_t nseg) {
    const int64_t per = (int64_t)mask_tile_of(nseg) * kWavesPerBlock;
    return shape_of((nseg + per - 1) / per, kBlock);
}

template <typename S>
In<S> make_in(const void *sdf, const void *deform, double iso, const Geo &g) {
    In<S> in;
    in.sdf = static_cast<const S *>(sdf);
    in.deform = static_cast<const S *>(deform);
    in.iso = (S)iso;
    in.pad = (S)(iso + 1.0);
    in.geo = g;
    return in;
}

template <typename S>
int launch_count(int algo, const void *sdf, double iso, const Geo &g, void *seg, void *ctl, hipStream_t st,
                 HostTotals *host = nullptr, uint64_t seq = 0) {
    CountSrc<S> src{};
    src.in = make_in<S>(sdf, nullptr, iso, g);
    src.nseg = g.nseg;
    src.recount_spins = (uint32_t)g_params.recount_spins;
    SegBase *sb = (SegBase *)seg;
    const Planes P = planes_of(sb, g.nseg);
    hipLaunchKernelGGL((mask_kernel<S, false>), mask_shape(g.nseg), dim3(kBlock), 0, st, src,
                       (const BatchGrid<S> *)nullptr, P, (uint8_t *)ctl, mask_tile_of(g.nseg));
    int rc = check_hip(hipGetLastError(), "mask kernel launch");
    if (rc) return rc;
    if (algo == DISO_MC) {
        const int64_t nb = count_blocks(g.nseg, count_resident_per_cu<count_kernel<S, DISO_MC, false>>());
        hipLaunchKernelGGL((count_kernel<S, DISO_MC, false>), dim3((unsigned)nb), dim3(kCountBlock), 0, st, src,
                           (const BatchGrid<S> *)nullptr, sb, P, (uint8_t *)ctl, nb, host, seq);
    } else {
        const int64_t nb = count_blocks(g.nseg, count_resident_per_cu<count_kernel<S, DISO_DMC, false>>());
        hipLaunchKernelGGL((count_kernel<S, DISO_DMC, false>), dim3((unsigned)nb), dim3(kCountBlock), 0, st, src,
                           (const BatchGrid<S> *)nullptr, sb, P, (uint8_t *)ctl, nb, host, seq);
    }
    return check_hip(hipGetLastError(), "count kernel launch");
}

// The run length is what four gathering waves take: a wave's tile is a quarter of it, down to a power
// of two (tiles divide the kBwdGroup segments that share a zeroing wave).
int bwd_tile_of(int64_t nseg) {
    int t = 1;
    while (2 * t <= run_for(nseg) / kWavesPerBlock && 2 * t <= kBwdTile) t *= 2;
    return t;
}
int64_t bwd_blocks(int64_t nseg, bool recompute) {
    const int tile = bwd_tile_of(nseg);
    const int parts = tile == 1 ? 1 : (recompute ? kBwdParts<true> : kBwdParts<false>);
    return (nseg + kBwdGroup - 1) / kBwdGroup * (kBwdGroup / tile * parts + 1);
}

template <typename S>
Norm<S> norm_of(const Geo &g) {
    Norm<S> nm;
    const int n[3] = {g.n0, g.n1, g.n2};
    for (int a = 0; a < 3; ++a) {
        nm.c[a] = (S)n[a] - S(1);
        nm.r[a] = S(1) / nm.c[a];
    }
    return nm;
}

// Blocks of a unit emission whose cells number at most `cells` (a cell has at least one triangle /
// patch, so a face / vertex capacity bounds them): a wave per unit or part of one, at most
// kUnitBlocksPerCU blocks per CU (then each wave goes through several units), a multiple of the eight
// XCDs.
constexpr int kUnitBlocksPerCU = 10;
int64_t unit_blocks(int64_t cells) {
    int64_t nb = cells / (kWave * kWavesPerBlock) + 1;
    constexpr int64_t few = kFewParts / kWavesPerBlock;  // (for_units may cut units in four)
    if (nb < few) nb = 4 * nb < few ? 4 * nb : few;
    const int64_t most = (int64_t)cu_count() * kUnitBlocksPerCU;
    if (nb > most) nb = most;
    return (nb + 7) / 8 * 8;
}

template <typename S>
int launch_emit(int algo, const void *sdf, const void *deform, double iso, int flags, const Geo &g,
                const void *seg, void *verts, int64_t vcap, void *faces, int64_t fcap, void *vinfo, hipStream_t st) {
    In<S> in = make_in<S>(sdf, deform, iso, g);
    const Norm<S> nm = norm_of<S>(g);
    const SegBase *sb = (const SegBase *)seg;
    const OutCfg out{flags, vcap, fcap};
    if (g.nseg < 4) return DISO_OK;  // no cell
    const Planes P = planes_of(sb, g.nseg);
    const dim3 block(kBlock), grid((unsigned)unit_blocks(algo == DISO_MC ? fcap : vcap));
    if (algo == DISO_MC) {
        if (deform)
            hipLaunchKernelGGL((emit_mc_kernel<S, true>), grid, block, 0, st, in, sb, P, (S *)verts, faces, out, nm);
        else
            hipLaunchKernelGGL((emit_mc_kernel<S, false>), grid, block, 0, st, in, sb, P, (S *)verts, faces, out, nm);
    } else {
        if (deform)
            hipLaunchKernelGGL((emit_dmc_kernel<S, true>), grid, block, 0, st, in, sb, P, (S *)verts, faces,
                               (uint8_t *)vinfo, out, nm);
        else
            hipLaunchKernelGGL((emit_dmc_kernel<S, false>), grid, block, 0, st, in, sb, P, (S *)verts, faces,
                               (uint8_t *)vinfo, out, nm);
    }
    return check_hip(hipGetLastError(), "emit kernel launch");
}

template <typename S>
int launch_backward(int algo, const void *sdf, const void *deform, double iso, int flags, const Geo &g,
                    const void *seg, const void *faces, int64_t nfaces, const void *vinfo, const void *adj_verts,
                    int64_t nverts, void *adj_sdf, void *adj_deform, void *scratch, hipStream_t st) {
    In<S> in = make_in<S>(sdf, deform, iso, g);
    AdjIn<S> a;
    a.adj = (const S *)adj_verts;
    a.n = nverts;
    a.flags = flags;
    a.nm = norm_of<S>(g);
    const int tile = bwd_tile_of(g.nseg);
    const int64_t nb = bwd_blocks(g.nseg, (flags & DISO_FLAG_RECOMPUTE) != 0);
    const SegBase *sb = (const SegBase *)seg;
    S *gs = (S *)adj_sdf, *gd = (S *)(deform ? adj_deform : nullptr);
    if (algo == DISO_DMC) {
        // per-edge upstream gradients from the quads, then the MC gather on them
        if (nfaces > 0) {
            const int64_t eb = (nfaces + kBlock - 1) / kBlock;
            hipLaunchKernelGGL((dmc_edge_grad_kernel<S>), dim3((unsigned)eb), dim3(kBlock), 0, st, faces, nfaces,
                               sb + g.nseg, (const uint8_t *)vinfo, a, (S *)scratch);
            int rc = check_hip(hipGetLastError(), "edge gradient kernel launch");
            if (rc) return rc;
        }
        a.adj = (const S *)scratch;
        a.n = nfaces;
        a.flags = flags & ~DISO_FLAG_NORMALIZE;  // applied by the edge gradient kernel
    }
    const dim3 grid = shape_of(stripe_blocks(nb), kWave), block(kWave);
    const bool rec = (flags & DISO_FLAG_RECOMPUTE) != 0;
    if (deform && rec)
        hipLaunchKernelGGL((bwd_mc_kernel<S, true, true>), grid, block, 0, st, in, sb, a, gs, gd, tile, nb);
    else if (deform)
        hipLaunchKernelGGL((bwd_mc_kernel<S, true, false>), grid, block, 0, st, in, sb, a, gs, gd, tile, nb);
    else if (rec)
        hipLaunchKernelGGL((bwd_mc_kernel<S, false, true>), grid, block, 0, st, in, sb, a, gs, gd, tile, nb);
    else
        hipLaunchKernelGGL((bwd_mc_kernel<S, false, false>), grid, block, 0, st, in, sb, a, gs, gd, tile, nb);
    return check_hip(hipGetLastError(), "backward kernel launch");
}

// Split: about 4 blocks per CU, each wave over a contiguous range of quads.
int64_t split_blocks(int64_t nq) {
    int64_t nb = (int64_t)cu_count() * 4;
    const int64_t need = (nq + kSplitBlock - 1) / kSplitBlock;
    if (nb > need) nb = need;
    if (nb > kMaxSplitWaves / kSplitWaves) nb = kMaxSplitWaves / kSplitWaves;
    return nb < 1 ? 1 : nb;
}

int64_t split_scratch_bytes(int64_t nq) { return kMaxSplitWaves * (int64_t)sizeof(uint32_t) + nq; }

template <typename S>
int launch_split(const void *verts, int64_t nv, const void *quads, int64_t nq, int flags, int64_t *tris,
                 void *scratch, hipStream_t st) {
    const int64_t nb = split_blocks(nq), nr = nb * kSplitWaves;
    uint32_t *counts = static_cast<uint32_t *>(scratch);
    uint8_t *first = static_cast<uint8_t *>(scratch) + kMaxSplitWaves * sizeof(uint32_t);
    hipLaunchKernelGGL((split_score_kernel<S>), dim3((unsigned)nb), dim3(kSplitBlock), 0, st, (const S *)verts, nv,
                       quads, nq, flags, first, counts, nr);
    int rc = check_hip(hipGetLastError(), "split score kernel launch");
    if (rc) return rc;
    hipLaunchKernelGGL(split_emit_kernel, dim3((unsigned)nb), dim3(kSplitBlock), 0, st, quads, nq, flags,
                       (const uint8_t *)first, (const uint32_t *)counts, nr, tris);
    return check_hip(hipGetLastError(), "split emit kernel launch");
}

int check_common(int algo, int dtype, int64_t X, int64_t Y, int64_t Z, int flags, Geo *g) {
    if (algo != DISO_MC && algo != DISO_DMC) return fail(DISO_E_INVALID, "algo must be DISO_MC or DISO_DMC");
    if (dtype != DISO_F32 && dtype != DISO_F64) return fail(DISO_E_INVALID, "dtype must be DISO_F32 or DISO_F64");
    if (!make_geo(X, Y, Z, flags, g))
        return fail(DISO_E_INVALID, "unsupported grid dims (%lld, %lld, %lld)", (long long)X, (long long)Y,
                    (long long)Z);
    return DISO_OK;
}

// Pinned staging for the totals copy, one per host thread, kept for the life of the process (a
// copy into pinned memory completes without a bounce through a pageable buffer).
SegBase *pinned_totals() {
    thread_local SegBase *p = nullptr;
    if (!p) {
        void *q = nullptr;
        if (hipHostMalloc(&q, 2 * sizeof(SegBase), hipHostMallocDefault) == hipSuccess) p = (SegBase *)q;
    }
    return p;
}

// `pinned`: stage the copy in this thread's pinned buffer (allocated on first use); otherwise in
// a stack buffer (diso_count_noalloc allocates nothing).
int read_totals(const Geo &g, const void *seg, diso_totals_t *t, hipStream_t st, bool pinned = true) {
    SegBase local[2];
    SegBase *tot = pinned ? pinned_totals() : nullptr;
    if (!tot) tot = local;
    int rc = check_hip(hipMemcpyAsync(tot, (const SegBase *)seg + g.nseg, 2 * sizeof(SegBase), hipMemcpyDeviceToHost,
                                      st),
                       "totals copy");
    if (rc) return rc;
    rc = check_hip(hipStreamSynchronize(st), "stream synchronize");
    if (rc) return rc;
    // Segment bases count (crossing edges, MC triangles | DMC patches); the count kernel records
    // which algorithm produced them.
    const bool dmc = tot[1].f == DISO_DMC;
    t->n_verts = dmc ? tot[0].f : tot[0].v;
    t->n_faces = dmc ? tot[0].v : tot[0].f;
    t->flags = tot[1].v;
    t->n_crossing = tot[0].v;
    return DISO_OK;
}

// This thread's landing place for totals written by the count kernel (handed to a later thread when
// this one ends), and the number of its next call (a kernel of an abandoned call writes an old number).
struct Landing {
    HostTotals *host = nullptr;
    uint64_t seq = 0;
};
Landing *make_landing() { return new Landing; }
Landing &landing() {
    Landing &l = *diso_host::thread_object<Landing, make_landing>();
    if (!l.host) {
        void *q = nullptr;
        if (hipHostMalloc(&q, sizeof(HostTotals), hipHostMallocCoherent | hipHostMallocMapped | hipHostMallocPortable) ==
            hipSuccess) {
            l.host = (HostTotals *)q;
            l.host->seq = 0;
        }
    }
    return l;
}

// Waits until the count has written number `seq`; the stream's state tells of a failed launch.
int wait_totals(const HostTotals *h, uint64_t seq, hipStream_t st) {
    auto written = [&]() { return __atomic_load_n(&h->seq, __ATOMIC_ACQUIRE) == seq; };
    return diso_host::wait_until(written, [&]() {
        const hipError_t e = hipStreamQuery(st);
        if (e == hipErrorNotReady) return (int)DISO_OK;
        if (e != hipSuccess) return check_hip(e, "count pass");
        return written() ? (int)DISO_OK : fail(DISO_E_HIP, "count pass ended without totals");
    });
}

// ---- batches

int64_t align256(int64_t x) { return (x + 255) & ~(int64_t)255; }

constexpr int kBatchGroups = 9;  // emit: MC/DMC x deform; backward: deform x recompute; DMC edges

// Where everything of a batch lives in its workspace: the device descriptors, the launch-group
// tables, the per-grid totals, then the segment bases and classification planes of all grids.
struct BatchLayout {
    int n = 0;
    int64_t nseg = 0;
    std::vector<Geo> geo;
    std::vector<int64_t> seg_first;
    int64_t off_desc = 0, off_groups = 0, off_totals = 0, off_seg = 0, off_planes = 0, off_range = 0, total = 0;
};

int64_t group_bytes(int n) { return align256((int64_t)n * 4) + align256((int64_t)(n + 1) * 8); }

bool batch_layout(const diso_grid_t *grids, int n, BatchLayout *L) {
    if (!grids || n < 1) return false;
    L->n = n;
    L->geo.resize(n);
    L->seg_first.resize(n);
    int64_t nseg = 0;
    for (int i = 0; i < n; ++i) {
        if (!make_geo(grids[i].X, grids[i].Y, grids[i].Z, grids[i].flags, &L->geo[i])) return false;
        L->seg_first[i] = nseg;
        nseg += L->geo[i].nseg;
    }
    if (nseg >= (1ll << 32)) return false;
    L->nseg = nseg;
    L->off_desc = 0;
    L->off_groups = align256((int64_t)n * (int64_t)sizeof(BatchGrid<double>));
    L->off_totals = L->off_groups + kBatchGroups * group_bytes(n);
    L->off_range = L->off_totals + align256((int64_t)n * (int64_t)sizeof(diso_totals_t));
    L->off_seg = L->off_range + align256((int64_t)n * 8);
    L->off_planes = L->off_seg + (nseg + 2) * (int64_t)sizeof(SegBase);
    L->total = L->off_planes + nseg * kSegStateBytes;
    return true;
}

int64_t batch_ctl_bytes(int n) { return align256(ctl_bytes_for(Geo{})) + align256((int64_t)n * 4); }

int check_batch(int dtype, const diso_grid_t *grids, int n, BatchLayout *L) {
    if (dtype != DISO_F32 && dtype != DISO_F64) return fail(DISO_E_INVALID, "dtype must be DISO_F32 or DISO_F64");
    if (!grids || n < 1) return fail(DISO_E_INVALID, "empty batch");
    for (int i = 0; i < n; ++i) {
        if (grids[i].algo != DISO_MC && grids[i].algo != DISO_DMC)
            return fail(DISO_E_INVALID, "grid %d: algo must be DISO_MC or DISO_DMC", i);
        if (!grids[i].sdf) return fail(DISO_E_INVALID, "grid %d: null sdf", i);
    }
    if (!batch_layout(grids, n, L)) return fail(DISO_E_INVALID, "unsupported grid dims in the batch");
    return DISO_OK;
}

// Device descriptors of a batch, as far as the host knows them at this point of the pipeline.
template <typename S>
std::vector<BatchGrid<S>> batch_desc(const diso_grid_t *grids, const BatchLayout &L) {
    std::vector<BatchGrid<S>> d(L.n);
    int64_t q = 0;
    for (int i = 0; i < L.n; ++i) {
        const diso_grid_t &G = grids[i];
        BatchGrid<S> &D = d[i];
        memset(&D, 0, sizeof(D));
        D.in = make_in<S>(G.sdf, G.deform, G.iso, L.geo[i]);
        D.nm = norm_of<S>(L.geo[i]);
        D.algo = G.algo;
        D.flags = G.flags;
        D.seg_first = L.seg_first[i];
        D.nv = G.totals.n_verts;
        D.nf = G.totals.n_faces;
        D.verts = (S *)G.verts;
        D.faces = G.faces;
        D.vinfo = (uint8_t *)G.vinfo;
        D.vcap = G.vert_capacity;
        D.fcap = G.face_capacity;
        D.adj = (const S *)G.adj_verts;
        D.adj_sdf = (S *)G.adj_sdf;
        D.adj_deform = (S *)G.adj_deform;
        D.q_first = q;
        D.tile = bwd_tile_of(L.geo[i].nseg);
        if (G.algo == DISO_DMC) q += G.totals.n_faces;
    }
    return d;
}

// One launch group: the grids it covers and the prefix of their block counts.
struct Group {
    std::vector<int32_t> gl;
    std::vector<int64_t> rf{0};
    void add(int i, int64_t blocks) {
        if (blocks <= 0) return;
        gl.push_back(i);
        rf.push_back(rf.back() + blocks);
    }
    int m() const { return (int)gl.size(); }
    int64_t blocks() const { return rf.back(); }
};

// Pinned host buffers of one host thread, kept for the life of the process: `up` stages
// host-to-device copies (reused once the copy recorded in `ev` has run, so the caller never waits
// for the device), `down` receives device-to-host copies.
struct Staging {
    void *up = nullptr, *down = nullptr;
    size_t up_cap = 0, down_cap = 0;
    hipEvent_t ev = nullptr;
    bool pending = false;
};
Staging &staging() {
    thread_local Staging s;
    return s;
}

int grow_pinned(void **p, size_t *cap, size_t n) {
    if (*cap >= n) return DISO_OK;
    if (*p) check_hip(hipHostFree(*p), "pinned free");
    *p = nullptr;
    *cap = 0;
    const size_t want = n < 65536 ? 65536 : n + n / 2;
    int rc = check_hip(hipHostMalloc(p, want, hipHostMallocDefault), "pinned allocation");
    if (rc) return rc;
    *cap = want;
    return DISO_OK;
}

// Copies n host bytes to `dst` on `st` through the pinned staging buffer, without waiting.
int stage_copy(void *dst, const void *src, size_t n, hipStream_t st) {
    Staging &S = staging();
    int rc;
    if (S.pending) {  // the previous copy from the buffer must have run before it is reused
        rc = check_hip(hipEventSynchronize(S.ev), "staging wait");
        if (rc) return rc;
        S.pending = false;
    }
    if (!S.ev && (rc = check_hip(hipEventCreateWithFlags(&S.ev, hipEventDisableTiming), "staging event"))) return rc;
    if ((rc = grow_pinned(&S.up, &S.up_cap, n))) return rc;
    memcpy(S.up, src, n);
    if ((rc = check_hip(hipMemcpyAsync(dst, S.up, n, hipMemcpyHostToDevice, st), "descriptor copy"))) return rc;
    if ((rc = check_hip(hipEventRecord(S.ev, st), "staging event"))) return rc;
    S.pending = true;
    return DISO_OK;
}

// Host staging of descriptors + group tables, copied into the workspace in one transfer.
template <typename S>
int upload_batch(void *ws, const BatchLayout &L, const std::vector<BatchGrid<S>> &d, const Group *groups, int ng,
                 hipStream_t st) {
    std::vector<uint8_t> h(L.off_totals, 0);
    memcpy(h.data() + L.off_desc, d.data(), d.size() * sizeof(BatchGrid<S>));
    for (int k = 0; k < ng; ++k) {
        uint8_t *base = h.data() + L.off_groups + k * group_bytes(L.n);
        memcpy(base, groups[k].gl.data(), groups[k].gl.size() * 4);
        memcpy(base + align256((int64_t)L.n * 4), groups[k].rf.data(), groups[k].rf.size() * 8);
    }
    return stage_copy(ws, h.data(), h.size(), st);
}

template <typename S>
struct BatchPtrs {
    BatchGrid<S> *desc;
    SegBase *seg;
    Planes planes;
    uint32_t *range;  // first and end unit of each grid
    diso_totals_t *totals;
    const int32_t *gl(const BatchLayout &L, int k, uint8_t *ws) const {
        return (const int32_t *)(ws + L.off_groups + k * group_bytes(L.n));
    }
    const int64_t *rf(const BatchLayout &L, int k, uint8_t *ws) const {
        return (const int64_t *)(ws + L.off_groups + k * group_bytes(L.n) + align256((int64_t)L.n * 4));
    }
};

template <typename S>
BatchPtrs<S> batch_ptrs(void *ws, const BatchLayout &L) {
    uint8_t *b = (uint8_t *)ws;
    return BatchPtrs<S>{(BatchGrid<S> *)(b + L.off_desc), (SegBase *)(b + L.off_seg),
                        planes_at(b + L.off_planes, L.nseg), (uint32_t *)(b + L.off_range),
                        (diso_totals_t *)(b + L.off_totals)};
}

template <typename S>
int batch_count(diso_grid_t *grids, const BatchLayout &L, void *ws, void *ctl, hipStream_t st) {
    const std::vector<BatchGrid<S>> d = batch_desc<S>(grids, L);
    int rc = upload_batch<S>(ws, L, d, nullptr, 0, st);
    if (rc) return rc;
    const BatchPtrs<S> P = batch_ptrs<S>(ws, L);
    CountSrc<S> src{};
    src.gflags = (uint32_t *)((uint8_t *)ctl + align256(ctl_bytes_for(Geo{})));
    src.ngrids = L.n;
    src.nseg = L.nseg;
    src.recount_spins = (uint32_t)g_params.recount_spins;
    hipLaunchKernelGGL((mask_kernel<S, true>), mask_shape(L.nseg), dim3(kBlock), 0, st, src,
                       (const BatchGrid<S> *)P.desc, P.planes, (uint8_t *)ctl, mask_tile_of(L.nseg));
    if ((rc = check_hip(hipGetLastError(), "batch mask kernel launch"))) return rc;
    const int64_t nb = count_blocks(L.nseg, count_resident_per_cu<count_kernel<S, DISO_MC, true>>());
    hipLaunchKernelGGL((count_kernel<S, DISO_MC, true>), dim3((unsigned)nb), dim3(kCountBlock), 0, st, src,
                       (const BatchGrid<S> *)P.desc, P.seg, P.planes, (uint8_t *)ctl, nb, (HostTotals *)nullptr,
                       (uint64_t)0);
    rc = check_hip(hipGetLastError(), "batch count kernel launch");
    if (rc) return rc;
    hipLaunchKernelGGL((batch_totals_kernel<S>), dim3((unsigned)((L.n + 255) / 256)), dim3(256), 0, st, P.desc, L.n,
                       L.nseg, P.seg, P.planes, src.gflags, P.range, P.totals);
    rc = check_hip(hipGetLastError(), "batch totals kernel launch");
    if (rc) return rc;
    Staging &stg = staging();
    const size_t tb = (size_t)L.n * sizeof(diso_totals_t);
    if ((rc = grow_pinned(&stg.down, &stg.down_cap, tb))) return rc;
    rc = check_hip(hipMemcpyAsync(stg.down, P.totals, tb, hipMemcpyDeviceToHost, st), "batch totals copy");
    if (rc) return rc;
    rc = check_hip(hipStreamSynchronize(st), "stream synchronize");
    if (rc) return rc;
    const diso_totals_t *t = (const diso_totals_t *)stg.down;
    for (int i = 0; i < L.n; ++i) {
        grids[i].totals = t[i];
        if (t[i].flags & DISO_TOTAL_SCAN_TIMEOUT) return fail(DISO_E_TIMEOUT, "single-pass scan did not complete");
    }
    return DISO_OK;
}

template <typename S>
int batch_emit(const diso_grid_t *grids, const BatchLayout &L, void *ws, hipStream_t st) {
    Group gr[4];  // MC, MC + deform, DMC, DMC + deform
    for (int i = 0; i < L.n; ++i) {
        const diso_grid_t &G = grids[i];
        if (G.totals.n_verts <= 0) continue;
        if (G.totals.n_verts > G.vert_capacity || G.totals.n_faces > G.face_capacity)
            return fail(DISO_E_CAPACITY, "grid %d: output buffers too small", i);
        if (!G.verts || !G.faces || (G.algo == DISO_DMC && !G.vinfo))
            return fail(DISO_E_INVALID, "grid %d: null output buffer", i);
        gr[2 * (G.algo == DISO_DMC) + (G.deform != nullptr)].add(
            i, (G.algo == DISO_DMC ? G.totals.n_verts : G.totals.n_faces / 2) / (kWave * kWavesPerBlock) + 1);
    }
    int rc = upload_batch<S>(ws, L, batch_desc<S>(grids, L), gr, 4, st);
    if (rc) return rc;
    const BatchPtrs<S> P = batch_ptrs<S>(ws, L);
    uint8_t *w = (uint8_t *)ws;
    for (int k = 0; k < 4; ++k) {
        const int64_t nb = gr[k].blocks();
        if (!nb) continue;
        const dim3 grid = shape_of(nb, kBlock), block(kBlock);
        const int32_t *gl = P.gl(L, k, w);
        const int64_t *rf = P.rf(L, k, w);
        const int m = gr[k].m();
        switch (k) {
            case 0: hipLaunchKernelGGL((emit_mc_batch_kernel<S, false>), grid, block, 0, st, P.desc, gl, rf, m, P.seg, P.planes, P.range, nb); break;
            case 1: hipLaunchKernelGGL((emit_mc_batch_kernel<S, true>), grid, block, 0, st, P.desc, gl, rf, m, P.seg, P.planes, P.range, nb); break;
            case 2: hipLaunchKernelGGL((emit_dmc_batch_kernel<S, false>), grid, block, 0, st, P.desc, gl, rf, m, P.seg, P.planes, P.range, nb); break;
            default: hipLaunchKernelGGL((emit_dmc_batch_kernel<S, true>), grid, block, 0, st, P.desc, gl, rf, m, P.seg, P.planes, P.range, nb); break;
        }
        rc = check_hip(hipGetLastError(), "batch emit kernel launch");
        if (rc) return rc;
    }
    return DISO_OK;
}

int64_t batch_scratch_bytes(int dtype, const diso_grid_t *grids, int n) {
    int64_t q = 0;
    for (int i = 0; i < n; ++i)
        if (grids[i].algo == DISO_DMC && grids[i].totals.n_faces > 0) q += grids[i].totals.n_faces;
    return q * 3 * (dtype == DISO_F32 ? 4 : 8);
}

template <typename S>
int batch_backward(const diso_grid_t *grids, const BatchLayout &L, void *ws, void *scratch, hipStream_t st) {
    Group gr[5];  // 0-3: gather, deform x recompute; 4: DMC per-edge gradients
    for (int i = 0; i < L.n; ++i) {
        const diso_grid_t &G = grids[i];
        if (!G.adj_sdf || G.totals.n_verts <= 0) continue;
        if (G.deform && !G.adj_deform) return fail(DISO_E_INVALID, "grid %d: adj_deform required", i);
        if (!G.adj_verts) return fail(DISO_E_INVALID, "grid %d: null adj_verts", i);
        if (G.algo == DISO_DMC) {
            if (!G.faces || !G.vinfo) return fail(DISO_E_INVALID, "grid %d: DMC backward needs quads and vinfo", i);
            gr[4].add(i, (G.totals.n_faces + kBlock - 1) / kBlock);
        }
        gr[2 * (G.deform != nullptr) + ((G.flags & DISO_FLAG_RECOMPUTE) != 0)].add(
            i, bwd_blocks(L.geo[i].nseg, (G.flags & DISO_FLAG_RECOMPUTE) != 0));
    }
    int rc = upload_batch<S>(ws, L, batch_desc<S>(grids, L), gr, 5, st);
    if (rc) return rc;
    const BatchPtrs<S> P = batch_ptrs<S>(ws, L);
    uint8_t *w = (uint8_t *)ws;
    S *ge = (S *)scratch;
    if (gr[4].blocks()) {
        hipLaunchKernelGGL((dmc_edge_grad_batch_kernel<S>), dim3((unsigned)gr[4].blocks()), dim3(kBlock), 0, st,
                           P.desc, P.gl(L, 4, w), P.rf(L, 4, w), gr[4].m(), ge);
        rc = check_hip(hipGetLastError(), "batch edge gradient kernel launch");
        if (rc) return rc;
    }
    for (int k = 0; k < 4; ++k) {
        const int64_t nb = gr[k].blocks();
        if (!nb) continue;
        const dim3 grid = shape_of(stripe_blocks(nb), kWave);
        const int32_t *gl = P.gl(L, k, w);
        const int64_t *rf = P.rf(L, k, w);
        const int m = gr[k].m();
        switch (k) {
            case 0: hipLaunchKernelGGL((bwd_batch_kernel<S, false, false>), grid, dim3(kWave), 0, st, P.desc, gl, rf, m, P.seg, P.planes, ge, nb); break;
            case 1: hipLaunchKernelGGL((bwd_batch_kernel<S, false, true>), grid, dim3(kWave), 0, st, P.desc, gl, rf, m, P.seg, P.planes, ge, nb); break;
            case 2: hipLaunchKernelGGL((bwd_batch_kernel<S, true, false>), grid, dim3(kWave), 0, st, P.desc, gl, rf, m, P.seg, P.planes, ge, nb); break;
            default: hipLaunchKernelGGL((bwd_batch_kernel<S, true, true>), grid, dim3(kWave), 0, st, P.desc, gl, rf, m, P.seg, P.planes, ge, nb); break;
        }
        rc = check_hip(hipGetLastError(), "batch backward kernel launch");
        if (rc) return rc;
    }
    return DISO_OK;
}

}  // namespace

// ------------------------------------------------------------------------------------------
// Counting without allocation (diso_count_noalloc): the single-pass scan's control block lives
// in this file-scope device array instead of a caller workspace. Each device holds its own copy
// (at its own address, from hipGetSymbolAddress) until the process ends. It is cleared once per
// device by a fill kernel on the first call's stream; after that the scan keeps it consistent
// from call to call (epoch-tagged words, each call clears the buffer the next one uses), so no
// per-call clearing is needed. Every call on a device shares the one array: calls that overlap
// in time on one device race.
constexpr int64_t kNoallocCtlBytes = kCtlHeader + 4 * kMaxCountBlocks * (int64_t)sizeof(uint64_t);
static_assert(kNoallocCtlBytes % 8 == 0, "control block is cleared in 8-byte words");
static __device__ __align__(256) uint8_t scratch[kNoallocCtlBytes];

static __global__ void clear_words_kernel(uint64_t *p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = 0ull;
}

namespace {

std::mutex g_scratch_mu;
void *g_scratch_ptr[64];  // device address of `scratch`, per device ordinal

// The current device's copy of `scratch` (looked up, and cleared on `st`, on the device's first
// call). Host code uses only this address, never the array's name.
int noalloc_ctl(hipStream_t st, void **out) {
    int dev = -1;
    int rc = check_hip(hipGetDevice(&dev), "hipGetDevice");
    if (rc) return rc;
    if (dev < 0 || dev >= 64) return fail(DISO_E_INVALID, "device ordinal %d out of range", dev);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        rc = check_hip(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
        if (rc) return rc;
        if (!p) return fail(DISO_E_HIP, "hipGetSymbolAddress(scratch) returned a null address");
        hipLaunchKernelGGL(clear_words_kernel, dim3(16), dim3(256), 0, st, (uint64_t *)p, kNoallocCtlBytes / 8);
        rc = check_hip(hipGetLastError(), "control block clear launch");
        if (rc) return rc;
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return DISO_OK;
}

}  // namespace

// ------------------------------------------------------------------------------------------
// C ABI

extern "C" {

const char *diso_last_error(void) { return g_err; }

const char *diso_version(void) { return "diso_hip 0.1.0 gfx950"; }

int64_t diso_seg_bytes(int64_t X, int64_t Y, int64_t Z, int flags) {
    Geo g;
    if (!make_geo(X, Y, Z, flags, &g)) return fail(DISO_E_INVALID, "unsupported grid dims");
    return (flags & DISO_FLAG_RECOMPUTE) ? bases_bytes_for(g) : seg_bytes_for(g);
}

int64_t diso_totals_offset(int64_t X, int64_t Y, int64_t Z, int flags) {
    Geo g;
    if (!make_geo(X, Y, Z, flags, &g)) return fail(DISO_E_INVALID, "unsupported grid dims");
    return g.nseg * (int64_t)sizeof(SegBase);
}

int64_t diso_ctl_bytes(int64_t X, int64_t Y, int64_t Z, int flags) {
    Geo g;
    if (!make_geo(X, Y, Z, flags, &g)) return fail(DISO_E_INVALID, "unsupported grid dims");
    return ctl_bytes_for(g);
}

int diso_count(int algo, int dtype, const void *sdf, int64_t X, int64_t Y, int64_t Z, double iso,
               int flags, void *seg, int64_t seg_bytes, void *ctl, int64_t ctl_bytes,
               diso_totals_t *totals_host, void *stream) {
    g_err[0] = 0;
    Geo g;
    int rc = check_common(algo, dtype, X, Y, Z, flags, &g);
    if (rc) return rc;
    if (!sdf || !seg || !ctl) return fail(DISO_E_INVALID, "null pointer argument");
    if (seg_bytes < seg_bytes_for(g))
        return fail(DISO_E_CAPACITY, "seg workspace too small: %lld < %lld bytes", (long long)seg_bytes,
                    (long long)seg_bytes_for(g));
    if (ctl_bytes < ctl_bytes_for(g))
        return fail(DISO_E_CAPACITY, "ctl workspace too small: %lld < %lld bytes", (long long)ctl_bytes,
                    (long long)ctl_bytes_for(g));
    hipStream_t st = (hipStream_t)stream;
    rc = dtype == DISO_F32 ? launch_count<float>(algo, sdf, iso, g, seg, ctl, st)
                           : launch_count<double>(algo, sdf, iso, g, seg, ctl, st);
    if (rc) return rc;
    if (totals_host) {
        rc = read_totals(g, seg, totals_host, st);
        if (rc) return rc;
        if (totals_host->flags & DISO_TOTAL_SCAN_TIMEOUT)
            return fail(DISO_E_TIMEOUT, "single-pass scan did not complete");
    }
    return DISO_OK;
}

int diso_count_noalloc(int algo, int dtype, const void *sdf, int64_t X, int64_t Y, int64_t Z, double iso,
                       int flags, void *seg, int64_t seg_bytes, diso_totals_t *totals_host, void *stream) {
    g_err[0] = 0;
    Geo g;
    int rc = check_common(algo, dtype, X, Y, Z, flags, &g);
    if (rc) return rc;
    if (!sdf || !seg) return fail(DISO_E_INVALID, "null pointer argument");
    if (seg_bytes < seg_bytes_for(g))
        return fail(DISO_E_CAPACITY, "seg workspace too small: %lld < %lld bytes", (long long)seg_bytes,
                    (long long)seg_bytes_for(g));
    if (ctl_bytes_for(g) > kNoallocCtlBytes)
        return fail(DISO_E_CAPACITY, "grid needs a %lld-byte control block, more than the %lld bytes of the "
                    "library's own", (long long)ctl_bytes_for(g), (long long)kNoallocCtlBytes);
    hipStream_t st = (hipStream_t)stream;
    void *ctl = nullptr;
    rc = noalloc_ctl(st, &ctl);
    if (rc) return rc;
    rc = dtype == DISO_F32 ? launch_count<float>(algo, sdf, iso, g, seg, ctl, st)
                           : launch_count<double>(algo, sdf, iso, g, seg, ctl, st);
    if (rc) return rc;
    if (totals_host) {
        rc = read_totals(g, seg, totals_host, st, false);
        if (rc) return rc;
        if (totals_host->flags & DISO_TOTAL_SCAN_TIMEOUT)
            return fail(DISO_E_TIMEOUT, "single-pass scan did not complete");
    }
    return DISO_OK;
}

int diso_read_totals(const void *seg, int64_t seg_bytes, int64_t X, int64_t Y, int64_t Z, int flags,
                     diso_totals_t *totals_host, void *stream) {
    g_err[0] = 0;
    Geo g;
    if (!make_geo(X, Y, Z, flags, &g)) return fail(DISO_E_INVALID, "unsupported grid dims");
    if (!seg || !totals_host) return fail(DISO_E_INVALID, "null pointer argument");
    if (seg_bytes < bases_bytes_for(g)) return fail(DISO_E_CAPACITY, "seg workspace too small");
    return read_totals(g, seg, totals_host, (hipStream_t)stream);
}

int64_t diso_scratch_bytes(int algo, int dtype, int64_t n_crossing) {
    if ((algo != DISO_MC && algo != DISO_DMC) || (dtype != DISO_F32 && dtype != DISO_F64) || n_crossing < 0)
        return fail(DISO_E_INVALID, "bad scratch query");
    if (algo == DISO_MC) return 0;
    return n_crossing * 3 * (dtype == DISO_F32 ? 4 : 8);
}

int diso_emit(int algo, int dtype, const void *sdf, const void *deform, int64_t X, int64_t Y, int64_t Z,
              double iso, int flags, const void *seg, int64_t seg_bytes, void *verts, int64_t vert_capacity,
              void *faces, int64_t face_capacity, void *vinfo, void *stream) {
    g_err[0] = 0;
    Geo g;
    int rc = check_common(algo, dtype, X, Y, Z, flags, &g);
    if (rc) return rc;
    if (!sdf || !seg) return fail(DISO_E_INVALID, "null pointer argument");
    if (seg_bytes < seg_bytes_for(g)) return fail(DISO_E_CAPACITY, "seg workspace too small");
    if (vert_capacity < 0 || face_capacity < 0) return fail(DISO_E_INVALID, "negative capacity");
    if ((vert_capacity && !verts) || (face_capacity && !faces)) return fail(DISO_E_INVALID, "null output buffer");
    if (algo == DISO_DMC && vert_capacity && !vinfo) return fail(DISO_E_INVALID, "DMC needs a vinfo buffer");
    hipStream_t st = (hipStream_t)stream;
    return dtype == DISO_F32 ? launch_emit<float>(algo, sdf, deform, iso, flags, g, seg, verts, vert_capacity, faces,
                                                  face_capacity, vinfo, st)
                             : launch_emit<double>(algo, sdf, deform, iso, flags, g, seg, verts, vert_capacity, faces,
                                                   face_capacity, vinfo, st);
}

int diso_extract(int algo, int dtype, const void *sdf, const void *deform, int64_t X, int64_t Y, int64_t Z, double iso,
                 int flags, void *seg, int64_t seg_bytes, void *ctl, int64_t ctl_bytes, void *verts,
                 int64_t vert_capacity, void *faces, int64_t face_capacity, void *vinfo, diso_totals_t *totals_host,
                 void *stream) {
    g_err[0] = 0;
    Geo g;
    int rc = check_common(algo, dtype, X, Y, Z, flags, &g);
    if (rc) return rc;
    if (!sdf || !seg || !ctl || !totals_host) return fail(DISO_E_INVALID, "null pointer argument");
    if (seg_bytes < seg_bytes_for(g)) return fail(DISO_E_CAPACITY, "seg workspace too small");
    if (ctl_bytes < ctl_bytes_for(g)) return fail(DISO_E_CAPACITY, "ctl workspace too small");
    if (vert_capacity < 0 || face_capacity < 0) return fail(DISO_E_INVALID, "negative capacity");
    if ((vert_capacity && !verts) || (face_capacity && !faces)) return fail(DISO_E_INVALID, "null output buffer");
    if (algo == DISO_DMC && vert_capacity && !vinfo) return fail(DISO_E_INVALID, "DMC needs a vinfo buffer");
    hipStream_t st = (hipStream_t)stream;
    if (st) {  // (the null stream cannot be captured) a captured count would never write what is waited for
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        rc = check_hip(hipStreamIsCapturing(st, &cap), "capture status");
        if (rc) return rc;
        if (cap != hipStreamCaptureStatusNone)
            return fail(DISO_E_INVALID, "the stream is being captured: the totals cannot be waited for");
    }
    Landing &land = landing();
    if (!land.host) return fail(DISO_E_HIP, "pinned allocation failed");
    const uint64_t seq = ++land.seq;
    const bool f32 = dtype == DISO_F32;
    rc = f32 ? launch_count<float>(algo, sdf, iso, g, seg, ctl, st, land.host, seq)
             : launch_count<double>(algo, sdf, iso, g, seg, ctl, st, land.host, seq);
    if (rc) return rc;
    if (vert_capacity || face_capacity)  // (else nothing could be written)
        rc = f32 ? launch_emit<float>(algo, sdf, deform, iso, flags, g, seg, verts, vert_capacity, faces, face_capacity, vinfo, st)
                 : launch_emit<double>(algo, sdf, deform, iso, flags, g, seg, verts, vert_capacity, faces, face_capacity, vinfo, st);
    const int rw = wait_totals(land.host, seq, st);
    if (rc || rw) return rc ? rc : rw;
    const HostTotals h = *land.host;
    totals_host->n_verts = algo == DISO_DMC ? h.f : h.v;
    totals_host->n_faces = algo == DISO_DMC ? h.v : h.f;
    totals_host->flags = h.flags;
    totals_host->n_crossing = h.v;
    if (h.flags & DISO_TOTAL_SCAN_TIMEOUT) return fail(DISO_E_TIMEOUT, "single-pass scan did not complete");
    return DISO_OK;
}

int diso_backward(int algo, int dtype, const void *sdf, const void *deform, int64_t X, int64_t Y, int64_t Z,
                  double iso, int flags, const void *seg, int64_t seg_bytes, const void *faces, int64_t n_faces,
                  const void *vinfo, const void *adj_verts, int64_t n_verts, void *adj_sdf, void *adj_deform,
                  void *scratch, int64_t scratch_bytes, void *stream) {
    g_err[0] = 0;
    Geo g;
    int rc = check_common(algo, dtype, X, Y, Z, flags, &g);
    if (rc) return rc;
    if (!sdf || !seg || !adj_sdf) return fail(DISO_E_INVALID, "null pointer argument");
    if (deform && !adj_deform) return fail(DISO_E_INVALID, "adj_deform required when deform is given");
    if (n_verts < 0 || (n_verts && !adj_verts)) return fail(DISO_E_INVALID, "bad adj_verts");
    if (seg_bytes < ((flags & DISO_FLAG_RECOMPUTE) ? bases_bytes_for(g) : seg_bytes_for(g)))
        return fail(DISO_E_CAPACITY, "seg workspace too small");
    if (algo == DISO_DMC) {
        if (n_faces < 0 || (n_faces && (!faces || !vinfo))) return fail(DISO_E_INVALID, "DMC backward needs the quads and vinfo");
        if (scratch_bytes < diso_scratch_bytes(algo, dtype, n_faces) || (n_faces && !scratch))
            return fail(DISO_E_CAPACITY, "scratch buffer too small for %lld quads", (long long)n_faces);
    }
    hipStream_t st = (hipStream_t)stream;
    return dtype == DISO_F32 ? launch_backward<float>(algo, sdf, deform, iso, flags, g, seg, faces, n_faces, vinfo,
                                                      adj_verts, n_verts, adj_sdf, adj_deform, scratch, st)
                             : launch_backward<double>(algo, sdf, deform, iso, flags, g, seg, faces, n_faces, vinfo,
                                                       adj_verts, n_verts, adj_sdf, adj_deform, scratch, st);
}

int64_t diso_split_scratch_bytes(int64_t n_quads) {
    if (n_quads < 0) return fail(DISO_E_INVALID, "negative quad count");
    return split_scratch_bytes(n_quads);
}

int diso_split(int dtype, const void *verts, int64_t n_verts, const void *quads, int64_t n_quads, int flags,
               int64_t *tris, int64_t tri_capacity, void *scratch, int64_t scratch_bytes, void *stream) {
    g_err[0] = 0;
    if (dtype != DISO_F32 && dtype != DISO_F64) return fail(DISO_E_INVALID, "dtype must be DISO_F32 or DISO_F64");
    if (n_quads < 0 || n_verts < 0) return fail(DISO_E_INVALID, "negative size");
    if (n_quads == 0) return DISO_OK;
    if (!verts || !quads || !tris || !scratch) return fail(DISO_E_INVALID, "null pointer argument");
    if (tri_capacity < 2 * n_quads)
        return fail(DISO_E_CAPACITY, "triangle buffer too small: %lld < %lld rows", (long long)tri_capacity,
                    (long long)(2 * n_quads));
    if (scratch_bytes < split_scratch_bytes(n_quads)) return fail(DISO_E_CAPACITY, "scratch buffer too small");
    hipStream_t st = (hipStream_t)stream;
    return dtype == DISO_F32 ? launch_split<float>(verts, n_verts, quads, n_quads, flags, tris, scratch, st)
                             : launch_split<double>(verts, n_verts, quads, n_quads, flags, tris, scratch, st);
}

int diso_set_param(int which, int value) {
    g_err[0] = 0;
    switch (which) {
        case DISO_PARAM_RUN:
        case DISO_PARAM_COUNT_BLOCKS_PER_CU: {
            int *t = bucket_table(which, value);
            if (!t) return DISO_E_INVALID;
            for (int b = 0; b < kBuckets; ++b) t[b] = value;
            return DISO_OK;
        }
        case DISO_PARAM_RECOUNT_SPINS:
            if (value < 0 || value > (int)kSpinLimit)
                return fail(DISO_E_INVALID, "recount spins must be in [0, %u]", kSpinLimit);
            g_params.recount_spins = value;
            return DISO_OK;
        default:
            return fail(DISO_E_INVALID, "unknown parameter %d", which);
    }
}

int diso_get_param(int which) {
    switch (which) {
        case DISO_PARAM_RUN: return g_params.run[kBuckets - 2];
        case DISO_PARAM_COUNT_BLOCKS_PER_CU: return g_params.count_per_cu[kBuckets - 2];
        case DISO_PARAM_RECOUNT_SPINS: return g_params.recount_spins;
        default: return fail(DISO_E_INVALID, "unknown parameter %d", which);
    }
}

int diso_set_bucket_param(int which, int bucket, int value) {
    g_err[0] = 0;
    if (bucket < 0 || bucket >= kBuckets) return fail(DISO_E_INVALID, "bucket must be in [0, %d]", kBuckets - 1);
    int *t = bucket_table(which, value);
    if (!t) return DISO_E_INVALID;
    t[bucket] = value;
    return DISO_OK;
}

int diso_get_bucket_param(int which, int bucket) {
    if (bucket < 0 || bucket >= kBuckets) return fail(DISO_E_INVALID, "bucket must be in [0, %d]", kBuckets - 1);
    switch (which) {
        case DISO_PARAM_RUN: return g_params.run[bucket];
        case DISO_PARAM_COUNT_BLOCKS_PER_CU: return g_params.count_per_cu[bucket];
        default: return fail(DISO_E_INVALID, "parameter %d has no size buckets", which);
    }
}

int diso_param_bucket(int64_t X, int64_t Y, int64_t Z, int flags) {
    Geo g;
    if (!make_geo(X, Y, Z, flags, &g)) return fail(DISO_E_INVALID, "bad grid dims");
    return bucket_of(g.nseg);
}

int64_t diso_batch_seg_bytes(const diso_grid_t *grids, int n) {
    BatchLayout L;
    if (!batch_layout(grids, n, &L)) return fail(DISO_E_INVALID, "bad batch");
    return L.total;
}

int64_t diso_batch_ctl_bytes(int n) {
    if (n < 1) return fail(DISO_E_INVALID, "empty batch");
    return batch_ctl_bytes(n);
}

int diso_batch_count(int dtype, diso_grid_t *grids, int n, void *seg, int64_t seg_bytes, void *ctl, int64_t ctl_bytes,
                     void *stream) {
    g_err[0] = 0;
    BatchLayout L;
    int rc = check_batch(dtype, grids, n, &L);
    if (rc) return rc;
    if (!seg || !ctl) return fail(DISO_E_INVALID, "null pointer argument");
    if (seg_bytes < L.total) return fail(DISO_E_CAPACITY, "batch workspace too small");
    if (ctl_bytes < batch_ctl_bytes(n)) return fail(DISO_E_CAPACITY, "batch ctl workspace too small");
    hipStream_t st = (hipStream_t)stream;
    return dtype == DISO_F32 ? batch_count<float>(grids, L, seg, ctl, st) : batch_count<double>(grids, L, seg, ctl, st);
}

int diso_batch_emit(int dtype, const diso_grid_t *grids, int n, void *seg, int64_t seg_bytes, void *stream) {
    g_err[0] = 0;
    BatchLayout L;
    int rc = check_batch(dtype, grids, n, &L);
    if (rc) return rc;
    if (!seg) return fail(DISO_E_INVALID, "null pointer argument");
    if (seg_bytes < L.total) return fail(DISO_E_CAPACITY, "batch workspace too small");
    hipStream_t st = (hipStream_t)stream;
    return dtype == DISO_F32 ? batch_emit<float>(grids, L, seg, st) : batch_emit<double>(grids, L, seg, st);
}

int64_t diso_batch_scratch_bytes(int dtype, const diso_grid_t *grids, int n) {
    if ((dtype != DISO_F32 && dtype != DISO_F64) || !grids || n < 1) return fail(DISO_E_INVALID, "bad batch");
    return batch_scratch_bytes(dtype, grids, n);
}

int diso_batch_backward(int dtype, const diso_grid_t *grids, int n, void *seg, int64_t seg_bytes, void *scratch,
                        int64_t scratch_bytes, void *stream) {
    g_err[0] = 0;
    BatchLayout L;
    int rc = check_batch(dtype, grids, n, &L);
    if (rc) return rc;
    if (!seg) return fail(DISO_E_INVALID, "null pointer argument");
    if (seg_bytes < L.total) return fail(DISO_E_CAPACITY, "batch workspace too small");
    const int64_t need = batch_scratch_bytes(dtype, grids, n);
    if (scratch_bytes < need || (need && !scratch)) return fail(DISO_E_CAPACITY, "batch scratch too small");
    hipStream_t st = (hipStream_t)stream;
    return dtype == DISO_F32 ? batch_backward<float>(grids, L, seg, scratch, st)
                             : batch_backward<double>(grids, L, seg, scratch, st);
}

}  // extern "C"
