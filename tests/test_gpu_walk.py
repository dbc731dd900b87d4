"""The streaming traversal (walk4_stream) against the oracle's one-ray walk
over the same 4-wide tree: equal bits at the edges of its ray groups (16, 32,
64 rays a wave, waves that take new rays), with stacks deeper than their LDS
part, coincident triangles (ties), axis-parallel rays and rays that end
before the scene."""
import numpy as np
import pytest

from meturay_amd import native as N

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _scene(n):
    tris = N.gen_random_tris(n, 40 + n)
    if n >= 64:
        tris[n // 2: n // 2 + n // 8] = tris[: n // 8]      # coincident pairs
        tris[n - 20:] = tris[5]                             # 20 copies of one
    return tris


def _rays(m, seed):
    rays = N.gen_random_rays(m, seed)
    k = np.arange(m)
    ax = k % 7 == 3
    rays[3:6, ax] = 0.0
    rays[3 + (k[ax] % 3), k[ax]] = np.where(k[ax] % 2 == 0, 1.0, -1.0)
    rays[6, k % 11 == 5] = 0.05                             # tmax inside the scene
    return rays


@pytest.mark.parametrize("lds", [8, 24])
@pytest.mark.parametrize("n,m", [(1, 70), (2, 1), (700, 15), (700, 17), (5000, 65), (5000, 4097),
                                 (5000, 32_769), (5000, 65_537),
                                 (60_000, 131_071), (60_000, 300_001), (60_000, 600_001)])
def test_stream_walk_equals_oracle(ctx, oracle, n, m, lds):
    tris, rays = _scene(n), _rays(m, n + m)
    old = ctx.tune_get("trace_lds_entries"), ctx.tune_get("trace_blocks_per_cu")
    ctx.tune("trace_lds_entries", lds)
    if m > 500_000:
        ctx.tune("trace_blocks_per_cu", 1)                  # every wave takes several groups
    try:
        d_t, d_r = torch.from_numpy(tris).cuda(), torch.from_numpy(rays).cuda()
        prim = torch.full((m,), 7, dtype=torch.int32, device="cuda")
        anyh, t, bary = torch.full_like(prim, 7), torch.full((m,), -1.0, device="cuda"), torch.zeros(2, m, device="cuda")
        torch.cuda.synchronize()
        b = N.Lbvh(ctx, d_t, n, 30)
        L, p = N.lib(), N.ptr
        ctx.check(L.mrh_trace_closest(ctx.h, b.h, p(d_r), m, m, 0.001, p(prim), p(t), p(bary), None))
        ctx.check(L.mrh_trace_any(ctx.h, b.h, p(d_r), m, m, 0.001, p(anyh)))
        ctx.sync()
        b.close()
    finally:
        ctx.tune("trace_lds_entries", old[0])
        ctx.tune("trace_blocks_per_cu", old[1])
    o = oracle.LBVH(tris, 30)
    rp, rt, rb = o.trace(rays, tmin=0.001, width=4)
    assert np.array_equal(prim.cpu().numpy().view(np.uint32), rp)
    assert t.cpu().numpy().tobytes() == rt.tobytes()
    assert bary.cpu().numpy().tobytes() == rb.tobytes()
    assert np.array_equal(anyh.cpu().numpy() != 0, rp != 0xFFFFFFFF)


@pytest.mark.parametrize("two_level", [0, 1])
@pytest.mark.parametrize("w,h", [(5, 3), (17, 31), (200, 111)])
def test_frame_equals_counting_walk(ctx, w, h, two_level):
    """A frame traced by the streaming walk (flat and two-level) and by the
    counting one-ray walk: the same paths, so the same segments and image up
    to the order of a pixel's adds (S^2 = 4 of them and a path's few
    emitters: 8 float adds at most)."""
    sc = N.gen_instanced_sphere_grid(15, 8, 8, 3, 4) if two_level else N.gen_sphere_grid(15, 8, 8, 3)
    scene = N.Scene(ctx, sc)
    img = [torch.zeros(h, w, 3, device="cuda") for _ in range(2)]
    torch.cuda.synchronize()
    st = [scene.render(img[k], w, h, 2, 9, 3, 5, nee=1, mis=1, count_traversal=bool(k)) for k in range(2)]
    scene.close()
    assert st[0].segments == st[1].segments
    assert list(st[0].bounce_rays) == list(st[1].bounce_rays)
    a, b = img[0].cpu().numpy(), img[1].cpu().numpy()
    assert np.all(np.abs(a - b) <= 8 * 2.0 ** -24 * np.maximum(np.abs(a), np.abs(b)).max())
