"""The guide octree's filter (one wave per subtree of the last three levels, or
of two or one where those are few) against the oracle at its edges: trees of
one to three levels, a single path of nodes, few samples (bins filled from far
ancestors, or from none), and trees around the 4096 nodes a level needs."""
import numpy as np
import pytest

from meturay_amd import native as N
from test_gpu_guide import CUBE, assert_same_svo, clustered_points, dev, gpu_view

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("depth", [1, 2, 3, 4, 9])
@pytest.mark.parametrize("n,samples", [(1, 1), (1, 0), (7, 3), (5000, 40), (5000, 20000)])
def test_filter_equals_oracle(ctx, oracle, depth, n, samples):
    codes = oracle.svo_codes(clustered_points(n, 3 + n), CUBE, depth)
    check(ctx, oracle, codes, depth, samples)


# every cell of level `full`, its first leaf: 4096 nodes in it and below
@pytest.mark.parametrize("depth,full,missing", [(4, 4, 0), (5, 4, 0), (5, 4, 1), (6, 4, 0), (6, 4, 1)])
@pytest.mark.parametrize("samples", [30, 20000])
def test_filter_equals_oracle_where_the_base_level_changes(ctx, oracle, depth, full, missing, samples):
    codes = np.arange(8 ** full - missing, dtype=np.uint32) << np.uint32(3 * (depth - full))
    check(ctx, oracle, codes, depth, samples)


def check(ctx, oracle, codes, depth, samples):
    n = len(codes)
    rng = np.random.default_rng(depth * 100 + n + samples)
    pick = codes[rng.integers(0, n, samples)].astype(np.uint32)
    bins = rng.integers(0, 64, samples).astype(np.uint32)
    vals = rng.exponential(2.0, samples).astype(np.float32)
    svo = N.Svo(ctx)
    d = [dev(x) for x in (codes, pick, bins, vals)]
    torch.cuda.synchronize()
    svo.build(d[0], n, CUBE, depth)
    o = oracle.Svo.build(codes, CUBE, depth)
    if samples:
        svo.splat(d[1], d[2], d[3], samples)
        o.splat(pick, bins, vals)
    svo.filter()
    ctx.sync()
    o.filter()
    assert_same_svo(gpu_view(ctx, svo), o)
    svo.close()
    o.close()
