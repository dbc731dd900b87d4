"""Sorts and partitions at the edges of a tile (4096 keys; below it one block
does every pass) and of the histogram's chunk (8192), against numpy's stable
sort: 4- and 8-byte keys, partial digits, few distinct keys, both orders."""
import numpy as np
import pytest

from meturay_amd import native as N

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
SIZES = [1, 63, 65, 4095, 4096, 4097, 8193, 70_001]


def _dev(a):
    return torch.from_numpy(a.view(np.int64 if a.itemsize == 8 else np.int32)).cuda()


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("dtype,begin,end", [(np.uint32, 0, 32), (np.uint32, 3, 14), (np.uint64, 0, 63), (np.uint64, 30, 41)])
@pytest.mark.parametrize("descending,few", [(0, 0), (1, 1)])
def test_sort_pairs(ctx, n, dtype, begin, end, descending, few):
    rng = np.random.default_rng(n + end)
    bits = 8 * np.dtype(dtype).itemsize
    keys = rng.integers(0, 3 if few else 1 << 62, n, dtype=np.uint64)
    keys = (keys << np.uint64(begin + 2) if few else (keys * np.uint64(5))).astype(dtype)
    vals = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    d_k, d_v = _dev(keys), _dev(vals)
    o_k, o_v = torch.zeros_like(d_k), torch.zeros_like(d_v)
    torch.cuda.synchronize()
    ctx.check(N.lib().mrh_sort_pairs(ctx.h, N.ptr(d_k), N.ptr(d_v), N.ptr(o_k), N.ptr(o_v), n, bits // 8, begin, end,
                                     descending))
    ctx.sync()
    field = (keys >> dtype(begin)) & dtype((1 << (end - begin)) - 1)
    order = np.argsort(~field if descending else field, kind="stable")
    assert np.array_equal(o_k.cpu().numpy().view(dtype), keys[order])
    assert np.array_equal(o_v.cpu().numpy().view(np.uint32), vals[order])


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("begin,part,end", [(24, 24, 32), (0, 24, 32), (5, 9, 12)])
@pytest.mark.parametrize("noalloc", [0, 1])
def test_partition(ctx, n, begin, part, end, noalloc):
    rng = np.random.default_rng(n + part)
    keys = ((rng.integers(0, 6, n) << 24) | (rng.integers(0, 9, n) << 9) | rng.integers(0, 40, n)).astype(np.uint32)
    w = end - part
    d_k = _dev(keys)
    order = torch.zeros(n, dtype=torch.int32, device="cuda")
    offs = torch.full(((1 << w) + 1,), -1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    f = N.lib().mrh_partition_by_key_noalloc if noalloc else N.lib().mrh_partition_by_key
    ctx.check(f(ctx.h, N.ptr(d_k), n, begin, part, end, N.ptr(order), N.ptr(offs)))
    ctx.sync()
    field = (keys >> begin) & ((1 << (end - begin)) - 1)
    ref = np.argsort(~field, kind="stable")
    assert np.array_equal(order.cpu().numpy(), ref)
    digit = (1 << w) - 1 - ((keys >> part) & ((1 << w) - 1)).astype(np.int64)
    counts = np.bincount(digit, minlength=1 << w)
    assert np.array_equal(offs.cpu().numpy(), np.concatenate([[0], np.cumsum(counts)]))
