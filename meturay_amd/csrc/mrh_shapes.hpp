// mrh_shapes.hpp — launch shapes: blocks of the traversal kernels for a number
// of rays and which block takes which of them, and how far down the octree
// filter's waves go.  Integer rules only, for the host and the kernels alike.
#pragma once

#include <cstdint>

namespace mrh {

// Few rays: a wave of the streaming walk starts with 32 or 16 instead of 64, so
// that it waits for the longest of fewer rays, as long as that makes no more
// than TRACE_SPLIT_WAVES waves, two a SIMD.  Past that the chip is busy, and
// waves of fewer rays only issue more.  Closest hits, 20,000 triangles: 50,000 /
// 100,000 / 140,000 / 200,000 rays in 100 / 105 / 118 / 142 us; split up to four
// waves a SIMD 111 / 116 / 118 / 142, up to eight 113 / 156 / 152 / 192.  500,000
// triangles and 50,000 rays: 232 us; up to one wave a SIMD 248.
constexpr uint32_t TRACE_MIN_SHIFT = 4, TRACE_MIN_GROUP = 1u << TRACE_MIN_SHIFT;
constexpr uint32_t TRACE_SPLIT_WAVES = 2048;

// Whether a traversal kernel runs the streaming walk, whose waves can take
// fewer than 64 rays; the others walk one ray a lane (the binary tree, the
// counting walk, a stack without an LDS part).
constexpr bool trace_streams(uint32_t width, uint32_t lds, bool counting) { return width == 4 && lds > 0 && !counting; }

// Waves for `rays` rays, `group` to a wave
constexpr uint64_t trace_waves(uint64_t rays, uint32_t group) { return (rays + group - 1) / group; }

// Blocks of `block` threads for up to `rays` rays: a multiple of 8 (one slice
// per XCD), at most `most` rounded up to one.  A streaming walk of few rays
// gets the waves that walk_split spreads them over.
constexpr uint32_t trace_blocks(uint64_t rays, bool stream, uint32_t block, uint64_t most)
{
    uint64_t waves = trace_waves(rays, 64);
    if (stream) {
        const uint64_t small = trace_waves(rays, TRACE_MIN_GROUP);
        const uint64_t split = small < TRACE_SPLIT_WAVES ? small : TRACE_SPLIT_WAVES;
        waves = waves > split ? waves : split;
    }
    const uint64_t want = (waves * 64 + block - 1) / block;
    const uint64_t some = want < most ? want : most;
    return (uint32_t)(some ? (some + 7) & ~7ull : 8);
}

// How a streaming walk of n rays uses a grid of `blocks` blocks (a multiple of
// 8) of `waves` waves: `group` rays to a wave to start with, in the first
// `used` blocks, a multiple of 8, so that every XCD has its share: 300,000 rays
// on 4,688 of 8,192 waves counted from the first logical block lie on five XCDs
// of eight (255 us in 20,000 triangles, 178 us so).
struct WalkSplit {
    uint32_t group, used;
};
constexpr WalkSplit walk_split(uint32_t n, uint32_t blocks, uint32_t waves)
{
    const uint32_t all = blocks * waves, split = all < TRACE_SPLIT_WAVES ? all : TRACE_SPLIT_WAVES;
    uint32_t shift = 6;   // of the group; shifts, since every wave of a launch starts here
    while (shift > TRACE_MIN_SHIFT && (n - 1) >> (shift - 1) < split) shift--;
    const uint32_t used = (n ? ((n - 1) >> shift) / waves + 8 : 8) & ~7u;
    return {1u << shift, used < blocks ? used : blocks};
}

// Logical index of block `b` of `blocks` (a multiple of 8) that gives each of
// the 8 XCDs (workgroups are handed to XCDs round-robin) a contiguous slice
// of the ray range, so neighbouring rays share an L2.
constexpr uint32_t xcd_slice(uint32_t b, uint32_t blocks) { return (b & 7u) * (blocks >> 3) + (b >> 3); }

// Stack entries past their LDS part, `entries` a thread: entry e of a thread is
// at spill_base + e * SPILL_STRIDE.  The entries of one depth of a wave's 64
// lanes are consecutive, so lanes that spill together share lines.  With each
// thread's entries together every lane touched a line of its own: a 1080p frame
// of 2 M triangles moved 27.1 GB in 14.9 ms, so it moves 25.5 GB in 14.6 ms.
constexpr uint32_t SPILL_STRIDE = 64;
constexpr uint64_t spill_base(uint64_t thread, uint32_t entries)
{
    return (thread >> 6) * entries * SPILL_STRIDE + (thread & (SPILL_STRIDE - 1));
}

// The octree level whose nodes the filter's waves go down from (k_svo_filter):
// two above the leaves, where each node is read and written once, as long as
// that level has SVO_FILTER_WAVES nodes, else one above, else the leaves
// themselves, every node climbing to its own means.  A wave that goes down
// takes its up to 73 nodes one after another, which few waves do not hide:
// full trees of depth 2 / 3 / 4 / 5 in 28 / 32 / 58 / 62 us, 77 / 92 / 99 / 120
// us always two levels down; 1 M points at depth 8 1691 us, 2006 us one level
// down and 2562 us climbing.
constexpr uint32_t SVO_FILTER_WAVES = 4096;
constexpr uint32_t svo_filter_base(uint32_t depth, const uint32_t* level_count)
{
    uint32_t base = depth >= 2 ? depth - 2 : 0;
    while (base < depth && level_count[base] < SVO_FILTER_WAVES) base++;
    return base;
}

}  // namespace mrh
