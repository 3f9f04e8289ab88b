// diso_launch.h - which block of a launch does what: grid shapes and block orders.
//
// Plain C++ (host and device), so the arithmetic is testable on the CPU at sizes no test can launch.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define DISO_LAUNCH_HD __host__ __device__ inline __attribute__((always_inline))
#else
#define DISO_LAUNCH_HD inline
#endif

namespace diso_launch {

// Shape of a launch of at least `blocks` blocks of `threads` threads. A dimension may not reach 2^32
// threads, which single-wave blocks do at 2^26 blocks, so beyond that the blocks are laid out in
// rows: block number y * rows_x + x (linear), rows_x a multiple of eight so that block i still goes to
// XCD i % 8. Blocks past `blocks` have nothing to do.
struct Shape {
    uint32_t x, y;
};
constexpr int64_t kMaxThreadsX = 0xffffffffll;
DISO_LAUNCH_HD Shape shape_of(int64_t blocks, int threads) {
    const int64_t most = kMaxThreadsX / threads / 8 * 8;
    if (blocks <= most) return Shape{(uint32_t)blocks, 1u};
    const int64_t rows = (blocks + most - 1) / most;
    return Shape{(uint32_t)(((blocks + rows - 1) / rows + 7) / 8 * 8), (uint32_t)rows};
}

// Block index remap: the dispatcher deals consecutive workgroups round-robin to the 8 XCDs;
// this gives each XCD a contiguous run of logical blocks so that neighbouring rows (which a
// block re-reads as halo) share one XCD's L2.
DISO_LAUNCH_HD int64_t xcd_block(int64_t bid, int64_t nb) {
    int64_t q = nb / 8, r = nb % 8;
    int64_t xcd = bid % 8, k = bid / 8;
    return xcd * q + (xcd < r ? xcd : r) + k;
}

// The same in kStripes turns: an XCD takes one of every eight stripes of consecutive blocks, so that
// work that is uneven over the grid (a surface's faces) is spread over the XCDs while neighbouring
// rows still mostly share one. The grid is padded to `stripe_blocks` blocks; returns a block >= nb for
// the padding. The 256^3 noisy gather, in one turn (an eighth of the grid per XCD: the planes of a
// box's face fall to one) 176 us, in 2, 4, 8, 16, 32 turns 170, 141, 135, 131, 132 us.
constexpr int64_t kStripes = 16;
DISO_LAUNCH_HD int64_t stripe_len(int64_t nb) { return (nb + 8 * kStripes - 1) / (8 * kStripes); }
DISO_LAUNCH_HD int64_t stripe_blocks(int64_t nb) { return stripe_len(nb) * 8 * kStripes; }
DISO_LAUNCH_HD int64_t xcd_stripe(int64_t bid, int64_t nb) {
    const int64_t c = stripe_len(nb), k = bid / 8, turn = k / c;
    return (turn * 8 + bid % 8) * c + (k - turn * c);
}

}  // namespace diso_launch
