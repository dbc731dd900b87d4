// mrh_walk.hpp — launch shapes of the traversal kernels: blocks for a number
// of rays, and which block takes which of them.  Integer rules only, for the
// host and the kernels alike.
#pragma once

#include <cstdint>

namespace mrh {

// Rays a wave starts with when there are few: a launch whose rays leave
// waves free gives each wave 32 or 16 of them instead of 64, so a wave waits
// for the longest of fewer rays (walk4_stream).  16 measured best: guided
// 1024x768 renders 19.29 / 18.99 / 18.81 / 18.88 ms at 64 / 32 / 16 / 8.
constexpr uint32_t TRACE_MIN_GROUP = 16;

// Whether a traversal kernel runs the streaming walk, whose waves can take
// fewer than 64 rays; the others walk one ray a lane (the binary tree, the
// counting walk, a stack without an LDS part).
constexpr bool trace_streams(uint32_t width, uint32_t lds, bool counting) { return width == 4 && lds > 0 && !counting; }

// Blocks of `block` threads for `rays` rays, `group` of them to a wave: a
// multiple of 8 (one slice per XCD), at most `most` rounded up to one.
constexpr uint32_t trace_blocks(uint64_t rays, uint32_t group, uint32_t block, uint64_t most)
{
    const uint64_t lanes = rays * (64 / group);
    const uint64_t want = (lanes + block - 1) / block;
    const uint64_t some = want < most ? want : most;
    return (uint32_t)(some ? (some + 7) & ~7ull : 8);
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

}  // namespace mrh
