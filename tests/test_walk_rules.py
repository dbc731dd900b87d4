"""Launch shapes of the traversal kernels (mrh_walk.hpp) on the CPU: which
block takes which rays is an integer rule, compiled here with the host
compiler.  Every ray is taken once, and no XCD idles beside a full one."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SIZES = [1, 15, 16, 17, 63, 64, 65, 255, 256, 257, 1000, 5001, 20_000, 65_536, 100_000, 131_072, 131_073, 140_000,
         262_144, 262_145, 300_000, 524_288, 524_289, 700_000, 2_073_600]
MOST = 256 * 8   # blocks of the whole chip at eight a CU

SRC = r"""
#include "mrh_walk.hpp"
extern "C" uint32_t blocks(uint64_t n, uint32_t group, uint32_t block, uint64_t most) { return mrh::trace_blocks(n, group, block, most); }
extern "C" int streams(uint32_t w, uint32_t lds, int counting) { return mrh::trace_streams(w, lds, counting != 0); }
extern "C" uint64_t spill(uint64_t t, uint32_t entries, uint32_t e) { return mrh::spill_base(t, entries) + e * mrh::SPILL_STRIDE; }
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
    lib.blocks.argtypes = [C.c_uint64, C.c_uint32, C.c_uint32, C.c_uint64]
    lib.spill.argtypes, lib.spill.restype = [C.c_uint64, C.c_uint32, C.c_uint32], C.c_uint64
    return lib


@pytest.mark.parametrize("block", [128, 256, 512])
@pytest.mark.parametrize("most", [8, 256, MOST])
def test_one_ray_kernels_fill_every_xcd(rules, block, most):
    """A one-ray-per-lane kernel's rays i, i + grid * block, ...: with fewer
    rays than threads the XCDs' shares differ by eight blocks at most."""
    for n in SIZES:
        grid = rules.blocks(n, 64, block, most)
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
