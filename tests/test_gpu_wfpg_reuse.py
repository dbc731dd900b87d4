"""A context's workspaces of the field-traced guide across calls: a small
render, a larger one of another scene and an incremental tracer with its own
buffers between two equal renders leave the second equal to the first."""
import ctypes as C

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
