"""Filtered frames around the edges of the filter's pixel tiles (32 x 8) and
of the samples a tile stages at once (all rows, a few, one, and frames with too
many samples per pixel for tiles), against the oracle."""
import pytest

from meturay_amd import native as N
from test_gpu_filter import _filtered_pair, descs, same

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("kind,r", [("Box", 0.0), ("Box", 1.0), ("Tent", 0.5), ("Gaussian", 1.5), ("Mitchell", 2.5)])
@pytest.mark.parametrize("w,h,spp_axis", [(1, 1, 1), (31, 7, 1), (32, 8, 2), (33, 9, 3), (65, 17, 5), (34, 9, 7), (33, 9, 8)])
def test_tile_edges_match_oracle(ctx, oracle, kind, r, w, h, spp_axis):
    g, st, ref, seg = _filtered_pair(ctx, oracle, N.gen_cornell(2), w, h, spp_axis, 3, 3, 5, descs(kind, r))
    assert st.segments == seg
    assert same(kind, g, ref)
