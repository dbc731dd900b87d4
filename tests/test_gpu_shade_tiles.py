"""The shade step's tile follows the frame's size: frames just under, at and
over the line between two tile sizes (four tiles a CU) render what the global
partition renders."""
import numpy as np
import pytest

from meturay_amd import native as N

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def render(ctx, scene, w, h, spp, nee):
    img = torch.zeros(w * h * 3, dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    st = scene.render(img.data_ptr(), w, h, spp, 3, 2, 7, nee=nee, mis=nee)
    return st.segments, img.cpu().numpy()


@pytest.mark.parametrize("nee", [0, 1])
@pytest.mark.parametrize("tile", [512, 1024, 2048])
@pytest.mark.parametrize("side", ["under", "at", "over"])
def test_tile_sizes_render_the_global_partitions_frame(ctx, tile, side, nee):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    w = 4 * cus
    h = tile // (2 if nee else 1)   # w * h rays (twice that with next event estimation) = tile * 4 * cus
    if side == "under":
        h -= 1
    elif side == "over":
        w, h = w + 1, h + 1
    scene = N.Scene(ctx, N.gen_cornell(2))
    old = {k: ctx.tune_get(k) for k in ("shade_partition", "shade_tile")}
    try:
        ctx.tune("shade_tile", tile)
        ctx.tune("shade_partition", 1)
        seg, got = render(ctx, scene, w, h, 1, nee)
        ctx.tune("shade_partition", 0)
        seg0, want = render(ctx, scene, w, h, 1, nee)
    finally:
        for k, v in old.items():
            ctx.tune(k, v)
        scene.close()
    assert seg == seg0
    # a pixel adds at most 3 bounces' two contributions in either order: each
    # addition rounds by at most 2^-24 of the (non-negative) sum
    assert np.allclose(got, want, rtol=6 * 2.0 ** -23, atol=1e-30)
