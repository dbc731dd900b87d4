"""A context's workspaces of the field-traced guide across calls: a small
render, a larger one of another scene and an incremental tracer with its own
buffers between two equal renders leave the second equal to the first.  What is
kept between calls is bounded, and given back when the device is full."""
import ctypes as C
from contextlib import closing

import numpy as np
import pytest

from meturay_amd import native as N

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("product", [0, 1])
def test_renders_share_workspaces(ctx, product):
    small, big = N.Scene(ctx, N.gen_sphere_grid(14, 6, 6, 4)), N.Scene(ctx, N.gen_sphere_grid(20, 10, 10, 5))
    kw = dict(iterations=2, svo_depth=6, min_bin_level=3, bin_ray_count=64, boundary_radiance=0.2)

    def shot(scene, w, h, **more):
        img = torch.zeros(h, w, 3, device="cuda")
        torch.cuda.synchronize()
        st, ws = scene.render_wfpg(img, w, h, 2, 5, 3, 9, **{**kw, **more})
        return img.cpu().numpy(), st.segments, ws

    a, seg_a, ws_a = shot(small, 40, 30)
    shot(big, 150, 110, svo_depth=8, product=product)
    t, more = C.c_void_p(), C.c_int32(1)
    p = N.RenderParams(33, 21, 2, 5, 3, 0, 1, 0, 0)
    wp = N.WfpgParams(2, 6, 0.5, 3, 64, 1.0, 0.2, product)
    L = N.lib()
    ctx.check(L.mrh_tracer_create(ctx.h, small.h, C.byref(p), C.byref(t)))
    ctx.check(L.mrh_tracer_set_wfpg(t, C.byref(wp)))
    cam = N.camera_desc(small.camera)
    ctx.check(L.mrh_tracer_generate_work(t, C.byref(cam)))
    ctx.check(L.mrh_tracer_render(t, C.byref(more)))
    b, seg_b, ws_b = shot(small, 40, 30)
    while more.value:
        ctx.check(L.mrh_tracer_render(t, C.byref(more)))
    L.mrh_tracer_destroy(t)
    small.close()
    big.close()
    assert seg_a == seg_b and ws_a.bins == ws_b.bins and ws_a.octree_nodes == ws_b.octree_nodes
    assert a.max() > 0 and np.allclose(a, b, rtol=1e-5, atol=1e-6 * a.max())


def free_bytes():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_large_renders_keep_a_bounded_part_of_their_memory():
    """4.2 M paths of up to 40 bounces in product mode need 4.7 GB for the path
    vertices, 1.1 GB for the BxDF fields and 0.4 GB for the rays; at most 4 GiB
    of it (and what sorts of these rays keep, below 0.5 GiB) stays."""
    w = h = 1024
    kw = dict(iterations=2, svo_depth=6, min_bin_level=3, bin_ray_count=512)
    with closing(N.Context(0)) as c, closing(N.Scene(c, N.gen_cornell(2))) as scene:
        img = torch.zeros(h, w, 3, device="cuda")
        torch.cuda.synchronize()
        scene.render_wfpg(img, 32, 32, 1, 4, 3, 9, product=1, **kw)
        scene.render_guided(img, w, h, 2, 40, 3, 9, iterations=2, svo_depth=6)   # the frame's own workspaces
        before, kept, mean = free_bytes(), [], []
        for product in (1, 0):
            scene.render_wfpg(img, w, h, 2, 40, 3, 9, product=product, **kw)
            kept.append(before - free_bytes())
            mean.append(float(img.mean()))
    assert max(kept) <= 4.5 * (1 << 30), kept
    assert mean[1] > 0 and abs(mean[0] / mean[1] - 1) < 0.05, mean


def test_kept_memory_goes_back_when_the_device_is_full():
    w, h = 512, 512
    kw = dict(iterations=2, svo_depth=6, min_bin_level=3, bin_ray_count=512)
    with closing(N.Context(0)) as c, closing(N.Scene(c, N.gen_cornell(2))) as scene:
        img = torch.zeros(h, w, 3, device="cuda")
        torch.cuda.synchronize()
        scene.render_wfpg(img, w, h, 2, 12, 3, 9, **kw)
        a, before, more = img.cpu().numpy(), free_bytes(), C.c_void_p()
        rc = N.lib().mrh_device_alloc(c.h, C.byref(more), 4 * torch.cuda.mem_get_info()[1])
        freed = free_bytes() - before
        scene.render_wfpg(img, w, h, 2, 12, 3, 9, **kw)
        b = img.cpu().numpy()
    assert rc == N.ERR_OOM
    # 1 M paths of 12 bounces: 28 B a vertex, 96 B a ray
    assert freed >= (w * h * 4) * (12 * 28 + 96), freed
    assert a.max() > 0 and np.allclose(a, b, rtol=1e-5, atol=1e-6 * a.max())
