"""Records listed in the coarser screen bins (4x4 and 16x16 bins large): patches
around the eye whose triangles cover up to the whole view, at frame sizes
around the edges of the levels (no coarse level, level 1 only, both, ragged
last bins), with ordinary and overflowing list capacities. Ids and depth
equal the oracle's bit for bit, and the counters too."""
import numpy as np
import pytest

import oracle
from glimpsw_amd import scene as S
from tests import scenes as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bin_capacity", [0, 2])
@pytest.mark.parametrize("width,height,bin_size", [
    (64, 64, 16),        # 16 bins: no coarse level
    (68, 64, 16),        # 20 bins: level 1, two bins of it
    (512, 512, 16),      # 64 level-1 bins: no level 2
    (516, 512, 16),      # 72 level-1 bins: level 2
    (1284, 964, 8),      # both levels, ragged
    (1284, 964, 16),
    (1284, 964, 32),
    (2044, 1412, 64),
])
def test_large_triangles_match_oracle(gpu_ctx, width, height, bin_size, bin_capacity):
    import glimpsw_amd as g

    print(f"[levels] {width}x{height} bins {bin_size} capacity {bin_capacity}", flush=True)
    sc = T.small_scene(160, seed_offset=7, spread=5.0, near_frac=0.5)
    view = S.make_view(width, height, count=sc.count)
    ofb, octr, _ = oracle.render_frame(sc, view)
    ds = g.Scene(gpu_ctx, sc)
    fb = g.Framebuffer(gpu_ctx, width, height)
    try:
        gpu_ctx.reset_counters()
        fb.clear(0, 0.0)
        fb.draw(ds, view.object_to_clip, sc.count, 0, view.frustum_planes(), g.GLIMP_DRAW_COUNTERS,
                bin_size=bin_size, bin_capacity=bin_capacity)
        ids, depth = fb.read()
        ctr = gpu_ctx.counters()
    finally:
        fb.close()
        ds.close()
    assert (ids == ofb.ids()).all()
    assert (depth.view(np.uint32) == ofb.depth().view(np.uint32)).all()
    assert ctr["fragments_covered"] == octr["fragments_covered"] and ctr["dropped"] == 0
