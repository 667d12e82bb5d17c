// w6a16_grid.h -- how the W6A16 tile kernel's workgroups map to tiles of the output.  Plain integer arithmetic, the same
// on the host and in the kernel, so that it can be carried through on the CPU at sizes no test could run.
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define W6_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define W6_HOST_DEVICE inline
#endif

namespace w6 {

// x / d as a multiplication and a shift (a 32-bit division takes the scalar unit some forty instructions).  Exact for
// every x < 2^31 and 1 <= d < 2^31: with d <= 2^l and mul = ceil(2^(31 + l) / d), mul d exceeds 2^(31 + l) by less than
// d <= 2^l, and x times that stays below 2^(31 + l).  mul < 2^32, since d > 2^(l - 1).
struct Divisor {
    uint32_t mul, shift;
};

inline Divisor divisor(uint32_t d) {
    uint32_t l = 0;
    while ((uint64_t(1) << l) < d) ++l;
    return {(uint32_t)(((uint64_t(1) << (31 + l)) + d - 1) / d), 31 + l};
}

W6_HOST_DEVICE uint32_t quotient(uint32_t x, Divisor d) { return (uint32_t)(((uint64_t)x * d.mul) >> d.shift); }

// A unit of 4 or 8 adjacent column tiles and all its M groups go to one XCD (workgroups are dealt to the XCDs in turn):
// neighbouring tiles share cache lines of the weights, the M groups all of them.  So workgroup x is number x / 8 of XCD
// x % 8, and an XCD takes its columns one after the other, each with all its M groups.
struct TileGrid {
    Divisor by_m_groups;
    uint32_t m_groups, unit_shift;  // log2 of a unit's workgroups (per M group)
    uint32_t first;                 // this launch's first workgroup, over 8
};

struct TilePos {
    uint32_t mg, column;  // M group; first column tile over the workgroup's column tiles (may lie past the last column)
};

W6_HOST_DEVICE TilePos tile_pos(const TileGrid& g, uint32_t x) {
    const uint32_t u = g.first + (x >> 3), v = quotient(u, g.by_m_groups), mask = (1u << g.unit_shift) - 1;
    return {u - v * g.m_groups, ((((v >> g.unit_shift) * 8 + (x & 7)) << g.unit_shift) + (v & mask))};
}

// The grid for `tiles` 16-column tiles, wg of them to a workgroup; returns its workgroups (below 2^34: u < 2^31).  Units of eight tiles (a whole
// line of the planes, a whole block of the packed layout) where they divide evenly among the XCDs or a workgroup takes
// eight, else of four.
inline uint64_t tile_grid(uint32_t tiles, uint32_t m_groups, uint32_t wg, TileGrid& g) {
    const uint32_t unit = wg == 8 || ((tiles + 7) / 8) % 8 == 0 ? 8 : 4, units = (tiles + unit - 1) / unit;
    g.by_m_groups = divisor(m_groups);
    g.m_groups = m_groups;
    g.unit_shift = g.first = 0;
    while ((wg << g.unit_shift) < unit) ++g.unit_shift;
    return ((uint64_t)((units + 7) / 8) << g.unit_shift) * m_groups * 8;
}

// Workgroups of `block` threads that one launch may have: the work-items of a grid's x dimension are counted in 32 bits.
inline uint32_t launch_limit(uint32_t block) { return 0x7FFFFFFFu / block & ~7u; }

}  // namespace w6
