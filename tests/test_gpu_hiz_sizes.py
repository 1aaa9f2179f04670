"""The depth pyramid (texutil::DownsampleDepth, ImageHelpers.cpp:149-247) at
frame sizes around its blocks' 128-pixel regions, with few and with many
levels: every level is bit-exact with the oracle, also when the same map is
built again from another frame."""
import numpy as np
import pytest

import oracle
from glimpsw_amd import scene as S
from tests import scenes as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(16, 16), (20, 200), (124, 128), (128, 128), (132, 260), (388, 252), (1024, 516),
                                  (1028, 1032), (2896, 1620)])
def test_depth_pyramid_sizes(gpu_ctx, size):
    import glimpsw_amd as g

    W, H = size
    sc = T.occluder_scene()
    ds = g.Scene(gpu_ctx, sc)
    dm = g.DepthMap(gpu_ctx, W, H)
    for yaw in (0.0, 0.3):
        view = S.make_view(W, H, view=S.view_matrix((0.0, 0.0, 0.0), yaw, 0.1), count=sc.count)
        fb = g.render_frame(gpu_ctx, ds, view)
        dm.build(fb)
        got, levels = dm.read()
        ofb, _, _ = oracle.render_frame(sc, view)
        want = oracle.hiz_build(ofb)
        print(f"[hiz] {W}x{H} yaw {yaw}: {levels} levels, {got.size} texels", flush=True)
        assert levels == oracle.hiz_levels(W, H) and got.size == want.size
        assert (got.view(np.uint32) == want.view(np.uint32)).all()
        fb.close()
    for o in (dm, ds):
        o.close()
