"""Draws with the default list capacity under stream capture, after one draw
of the largest frame: a smaller frame's lists fit in what that draw allocated
(memory cannot be allocated while a stream is captured). Every replay, with
eager draws of the context between them, gives the eager draw's keys."""
import numpy as np
import pytest

from glimpsw_amd import scene as S
from tests import scenes as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("large,small", [
    ((640, 480), (320, 240)),          # 1,200 and 300 bins
    ((1280, 960), (660, 400)),         # 4,800 and 1,050 bins: both with coarser bins
])
def test_smaller_frame_captured(large, small):
    import torch
    import glimpsw_amd as g

    print(f"[capture] {large} then {small}", flush=True)
    sc = T.small_scene(512, seed_offset=9, spread=6.0, near_frac=0.1)
    ctx = g.Context(0)
    ds = g.Scene(ctx, sc)
    views = [S.make_view(*size, count=sc.count) for size in (large, small)]
    fbs = [g.Framebuffer(ctx, v.width, v.height) for v in views]

    def frame(i, stream=None):
        fbs[i].clear(0, 0.0)
        fbs[i].draw(ds, views[i].object_to_clip, sc.count, 0, views[i].frustum_planes(), stream=stream)

    try:
        frame(0)
        graph = torch.cuda.CUDAGraph()
        stream = torch.cuda.Stream()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
            frame(1, stream)
        got = []
        for _ in range(3):
            graph.replay()
            torch.cuda.synchronize()
            got.append(fbs[1].read())
            frame(0)
            fbs[0].read()
        frame(1)
        ids, depth = fbs[1].read()
        assert (ids != 0).any()
        for gi, gd in got:
            assert (gi == ids).all() and (gd.view(np.uint32) == depth.view(np.uint32)).all()
    finally:
        for fb in fbs:
            fb.close()
        ds.close()
        ctx.close()
