"""The voxeliser's and the payload's blocks at their edges, bit for bit against
the oracle: triangle counts around a wave's 64 and a block's 256, and leaves
with so many records that a block's normals do not fit its LDS; and walls that
lie side by side in a mesh rasterise side by side."""
import time

import numpy as np
import pytest

from test_gpu_cone import build_both, surface_vertices
from test_gpu_guide import dev
from test_gpu_vox import cube_of, soup, voxelize_gpu

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 255, 256, 257])
def test_triangle_counts_around_a_wave(ctx, oracle, n):
    tris = soup(np.random.default_rng(n), n)
    cube = cube_of(oracle, tris, 6)
    got, gprim = voxelize_gpu(ctx, tris, cube, 6, prims=True)
    want, wprim = oracle.voxelize(tris, cube, 6, prims=True)
    assert np.array_equal(got, want) and np.array_equal(gprim, wprim)


@pytest.mark.parametrize("n", [64, 40_000])
def test_neighbouring_walls_do_not_wait_for_each_other(ctx, n):
    """64 whole-cube triangles in a row, alone and among small ones, against
    one: each goes to a wave of its own, so the call takes about as long.  One
    wave for the 64 of them takes 64 times as long; the bound lies between
    the two in ratio (8), far from either."""
    rng = np.random.default_rng(n)
    small = (rng.uniform(0.1, 0.9, (n, 1, 3)) + rng.uniform(0, 1e-3, (n, 3, 3))).astype(np.float32).reshape(n, 9)
    wall = np.array([0, 0, 0.5, 1, 0, 0.5, 0, 1, 0.5], np.float32)
    cube = [-0.01, -0.01, -0.01, 1.02]

    def micros(walls):
        tris = small.copy()
        tris[n // 2 - 32:n // 2 - 32 + walls] = wall
        d_t = dev(tris.reshape(-1))
        torch.cuda.synchronize()
        best = np.inf
        for _ in range(4):
            t0 = time.perf_counter()
            ctx.svo_voxelize(d_t, n, cube, 9)   # the count pass, waited for
            best = min(best, time.perf_counter() - t0)
        return 1e6 * best

    one, many = micros(1), micros(64)
    assert many < 8 * one, (one, many)


@pytest.mark.parametrize("depth,n", [(2, 40), (2, 16000), (3, 2000), (4, 300), (5, 4000), (6, 500)])
def test_payload_normals_of_full_and_sparse_leaves(ctx, oracle, depth, n):
    rng = np.random.default_rng(10 * depth + n)
    tris = soup(rng, n)
    e = tris.reshape(-1, 3, 3)
    area = np.linalg.norm(np.cross(e[:, 1] - e[:, 0], e[:, 2] - e[:, 0]), axis=1)
    tris = np.ascontiguousarray(tris[area > 1e-9])   # a degenerate triangle has no normal
    cube = cube_of(oracle, tris, depth)
    codes, prims = oracle.voxelize(tris, cube, depth, prims=True)
    assert n < 16000 or len(codes) > 8 * 1536   # more than a block stages anything of
    svo, o = build_both(ctx, oracle, codes, cube, depth)
    verts = surface_vertices(rng, tris, 400)
    d_t, d_c, d_p, d_v = dev(tris.reshape(-1)), dev(codes), dev(prims), dev(verts.reshape(-1))
    d_irr = torch.empty(2 * o.nodes, device="cuda")
    d_nrm = torch.empty(3 * o.nodes, device="cuda")
    d_len = torch.empty(o.nodes, device="cuda")
    torch.cuda.synchronize()
    svo.payload(d_t, d_c, d_p, len(codes), d_v, len(verts), d_irr, d_nrm, d_len)
    ctx.sync()
    oi, on = o.payload(tris, codes, prims, verts)
    assert np.array_equal(d_irr.cpu().numpy().view(np.uint32), oi.ravel().view(np.uint32))
    assert np.array_equal(d_nrm.cpu().numpy().view(np.uint32), on[:, :3].ravel().view(np.uint32))
    assert np.array_equal(d_len.cpu().numpy().view(np.uint32), on[:, 3].view(np.uint32))
