"""A batch whose views hold no meshlets leaves every view cleared, also at
sizes whose bins read the coarser levels' lists (over 1,024 bins) and in
memory that another batch's counts and lists filled before: eager, and every
replay of its graph with eager draws of the same framebuffers in between."""
import numpy as np
import pytest

from glimpsw_amd import scene as S
from tests import scenes as T

pytestmark = pytest.mark.gpu

SIZES = [(100, 60), (160, 144), (512, 512), (516, 512), (1284, 964)]    # 28 to 4,941 bins of 16 pixels


@pytest.mark.parametrize("bin_size", [8, 16, 64])
def test_views_without_meshlets(gpu_ctx, bin_size):
    import glimpsw_amd as g

    print(f"[empty batch] bins of {bin_size}", flush=True)
    sc = T.small_scene(160, seed_offset=7, spread=5.0, near_frac=0.5)
    views = [S.make_view(w, h, count=sc.count) for w, h in SIZES]
    shape = {"bin_size": bin_size, "bin_capacity": 1024, "raster_threads": 256}
    ds = g.Scene(gpu_ctx, sc)
    fbs = [g.Framebuffer(gpu_ctx, w, h) for w, h in SIZES]
    try:
        full = g.Batch(gpu_ctx, [(ds, fb, v) for fb, v in zip(fbs, views)], shape=shape)
        full.launch()
        assert all((fb.read()[0] != 0).any() for fb in fbs)
        full.close()

        empty = [(ds, fb, S.View(v.width, v.height, v.proj, v.view, v.object_to_clip, 0, 0))
                 for fb, v in zip(fbs, views)]
        b = g.Batch(gpu_ctx, empty, shape=shape, clear_color=7, clear_depth=0.25)
        for graph in (False, True, True, True):
            b.launch(graph=graph)
            for fb in fbs:
                ids, depth = fb.read()
                assert (ids == 7).all() and (depth == np.float32(0.25)).all()
            for fb, v in zip(fbs, views):
                fb.clear(0, 0.0)
                fb.draw(ds, v.object_to_clip, sc.count, 0, v.frustum_planes())
        b.close()
    finally:
        for fb in fbs:
            fb.close()
        ds.close()
