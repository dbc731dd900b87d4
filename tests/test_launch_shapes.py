"""Launch shapes (mrh_shapes.hpp) on the CPU: integer rules, compiled here with
the host compiler.  Every ray is taken once, and no XCD idles beside a full
one; the octree filter's waves go down only where there are many of them."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SIZES = [1, 15, 16, 17, 63, 64, 65, 255, 256, 257, 1000, 5001, 20_000, 65_536, 100_000, 131_072, 131_073, 140_000,
         262_144, 262_145, 300_000, 524_288, 524_289, 700_000, 2_073_600]
MOST = 256 * 8   # blocks of the whole chip at eight a CU

SRC = r"""
#include "mrh_shapes.hpp"
extern "C" uint32_t blocks(uint64_t n, int stream, uint32_t block, uint64_t most) { return mrh::trace_blocks(n, stream != 0, block, most); }
extern "C" void split(uint32_t n, uint32_t blocks, uint32_t waves, uint32_t* out)
{
    const mrh::WalkSplit s = mrh::walk_split(n, blocks, waves);
    out[0] = s.group;
    out[1] = s.used;
}
extern "C" int streams(uint32_t w, uint32_t lds, int counting) { return mrh::trace_streams(w, lds, counting != 0); }
extern "C" uint64_t spill(uint64_t t, uint32_t entries, uint32_t e) { return mrh::spill_base(t, entries) + e * mrh::SPILL_STRIDE; }
extern "C" uint32_t base(uint32_t depth, const uint32_t* count) { return mrh::svo_filter_base(depth, count); }
extern "C" uint32_t slice(uint32_t b, uint32_t n) { return mrh::xcd_slice(b, n); }
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("walk")
    (d / "w.cpp").write_text(SRC)
    so = str(d / "w.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-Wall", "-Werror", "-I",
                    os.path.join(ROOT, "meturay_amd", "csrc"), str(d / "w.cpp"), "-o", so], check=True)
    lib = C.CDLL(so)
    lib.blocks.argtypes = [C.c_uint64, C.c_int, C.c_uint32, C.c_uint64]
    lib.spill.argtypes, lib.spill.restype = [C.c_uint64, C.c_uint32, C.c_uint32], C.c_uint64
    return lib


@pytest.mark.parametrize("block", [128, 256, 512])
@pytest.mark.parametrize("most", [8, 256, MOST])
def test_one_ray_kernels_fill_every_xcd(rules, block, most):
    """A one-ray-per-lane kernel's rays i, i + grid * block, ...: with fewer
    rays than threads the XCDs' shares differ by eight blocks at most."""
    for n in SIZES:
        grid = rules.blocks(n, 0, block, most)
        assert grid % 8 == 0 and 8 <= grid <= (most + 7) // 8 * 8
        assert sorted(rules.slice(b, grid) for b in range(grid)) == list(range(grid))
        if n > grid * block:
            continue
        share = [0] * 8
        for b in range(grid):
            lo = rules.slice(b, grid) * block
            share[b % 8] += max(0, min(n, lo + block) - lo)
        assert sum(share) == n
        # up to 7 blocks that round the grid up are empty, one is half full
        assert max(share) - min(share) <= 8 * block, (n, share)


def split(rules, n, grid, waves):
    out = (C.c_uint32 * 2)()
    rules.split(n, grid, waves, out)
    return out[0], out[1]


@pytest.mark.parametrize("block", [128, 256, 512])
@pytest.mark.parametrize("most", [8, 256, MOST])
@pytest.mark.parametrize("exact", [1, 0])
def test_streaming_walk_takes_every_ray_once_on_all_xcds(rules, block, most, exact):
    """Groups of a streaming walk, in a grid made for its rays (a cast) and in
    one made for more of them (a later bounce of a frame)."""
    waves = block // 64
    for n in SIZES:
        grid = rules.blocks(n if exact else 2_100_000, 1, block, most)
        group, used = split(rules, n, grid, waves)
        assert group in (16, 32, 64) and used % 8 == 0 and 8 <= used <= grid
        assert sorted(rules.slice(b, used) for b in range(used)) == list(range(used))
        stride = used * waves * group
        if group < 64:
            assert stride >= n   # the walk's first lots do not reach a second stride
        share = [0] * 8          # a wave's rays: [g, g + group) for g = wave * group, + stride, ...
        for b in range(used):
            lo = rules.slice(b, used) * waves * group
            share[b % 8] += max(0, min(n, lo + waves * group) - lo)
        assert sum(share) == min(n, stride)
        if n <= stride:
            assert max(share) - min(share) <= 8 * waves * group, (n, share)


def test_few_rays_spread_only_as_far_as_it_pays(rules):
    """Waves of fewer than 64 rays are made for the chip's idle SIMDs, not
    instead of full ones: 140,000 rays are 2,188 full waves, two a SIMD."""
    for n, group in ((1, 16), (32_768, 16), (32_769, 32), (65_536, 32), (65_537, 64), (140_000, 64), (300_000, 64),
                     (2_000_000, 64)):
        grid = rules.blocks(n, 1, 256, MOST)
        assert split(rules, n, grid, 4)[0] == group, n
        assert split(rules, n, MOST, 4)[0] == group, n


@pytest.mark.parametrize("width,lds,counting,streams", [(4, 8, 0, 1), (4, 24, 0, 1), (4, 0, 0, 0), (4, 8, 1, 0),
                                                        (2, 8, 0, 0), (2, 0, 1, 0)])
def test_only_the_streaming_walk_takes_small_groups(rules, width, lds, counting, streams):
    assert rules.streams(width, lds, counting) == streams


@pytest.mark.parametrize("entries", [1, 8, 56, 120])
def test_spilled_entries_of_a_wave_share_lines(rules, entries):
    """8-byte entries: a depth of 64 lanes is 512 consecutive bytes, and no two
    (thread, depth) share a place in threads * entries of them."""
    threads = 3 * 64
    at = [[rules.spill(t, entries, e) for t in range(threads)] for e in range(entries)]
    assert sorted(sum(at, [])) == list(range(threads * entries))
    for row in at:
        for w in range(0, threads, 64):
            assert row[w:w + 64] == list(range(row[w], row[w] + 64))


@pytest.mark.parametrize("counts,base", [
    ([1, 8], 1), ([1, 8, 64], 2), ([1, 8, 64, 512, 4096, 32768], 4), ([1, 8, 64, 512, 4095, 32760], 5),
    ([1, 8, 64, 512, 4096, 32768, 262144], 4), ([1] * 11, 10),
    ([1, 8, 60, 300, 1200, 5000, 20_000, 80_000, 200_000, 400_000, 800_000], 8)])
def test_octree_filter_goes_down_from_a_level_of_many_nodes(rules, counts, base):
    """One wave per node of the base level: at least 4096 of them, or none
    that takes more than its own node."""
    depth = len(counts) - 1
    got = rules.base(depth, (C.c_uint32 * len(counts))(*counts))
    assert got == base
    assert got == depth or (depth - got <= 2 and counts[got] >= 4096)
