"""Draws that are culled and set up in one kernel (as many meshlets as there
are resident waves, or fewer) and draws that are not, one after another on one
context: ids, depth and counters equal the oracle's bit for bit, so each kind
leaves the shared counters as the other expects them. Some meshlets surround
the eye, so triangles are clipped, and some lie outside the view."""
import numpy as np
import pytest

import oracle
from glimpsw_amd import scene as S
from tests import scenes as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pipeline", ["visibility", "direct"])
@pytest.mark.parametrize("alpha", [False, True])
def test_draw_sizes_in_turn(gpu_ctx, alpha, pipeline):
    import glimpsw_amd as g

    W, H = 320, 240
    make = T.alpha_scene if alpha else T.small_scene
    sc = make(9000, seed_offset=11, spread=6.0, near_frac=0.05)
    ds = g.Scene(gpu_ctx, sc)
    fb = g.Framebuffer(gpu_ctx, W, H)
    flags = g.GLIMP_DRAW_COUNTERS | (g.GLIMP_DRAW_DIRECT if pipeline == "direct" else 0)
    for n in (1, 5, 300, 9000, 63, 64, 5119, 5121, 9000, 2, 4096):
        view = S.make_view(W, H, count=n)
        ofb, octr, _ = oracle.render_frame(sc, view)
        gpu_ctx.reset_counters()
        fb.clear(0, 0.0)
        fb.draw(ds, view.object_to_clip, n, 0, view.frustum_planes(), flags)
        ids, depth = fb.read()
        ctr = gpu_ctx.counters()
        print(f"[draws] {n} meshlets: {ctr['triangles_clipped']} clipped", flush=True)
        assert (ids == ofb.ids()).all()
        assert (depth.view(np.uint32) == ofb.depth().view(np.uint32)).all()
        for k in ("triangles_processed", "triangles_rasterized", "triangles_clipped"):
            assert ctr[k] == octr[k], k
    fb.close()
    ds.close()


@pytest.mark.parametrize("size,meshlets", [((16, 16), 3000), ((64, 48), 9000), ((180, 156), 1), ((180, 156), 9000)])
def test_default_list_capacity(gpu_ctx, size, meshlets):
    """Small frames of many meshlets: thousands of records in a bin, drawn
    with the default list capacity and with one that overflows."""
    import glimpsw_amd as g

    W, H = size
    sc = T.small_scene(meshlets, seed_offset=12, spread=6.0, near_frac=0.02)
    view = S.make_view(W, H, count=meshlets)
    ofb, _, _ = oracle.render_frame(sc, view)
    ds = g.Scene(gpu_ctx, sc)
    fb = g.Framebuffer(gpu_ctx, W, H)
    for cap in (0, 128):
        print(f"[draws] {W}x{H}, {meshlets} meshlets, capacity {cap}", flush=True)
        fb.clear(0, 0.0)
        fb.draw(ds, view.object_to_clip, meshlets, 0, view.frustum_planes(), 0, bin_capacity=cap)
        ids, depth = fb.read()
        assert (ids == ofb.ids()).all()
        assert (depth.view(np.uint32) == ofb.depth().view(np.uint32)).all()
    fb.close()
    ds.close()


@pytest.mark.parametrize("meshlets", [8, 640, 641, 1280, 1281, 2560, 2561])
def test_split_meshlets(gpu_ctx, meshlets):
    """Meshlets binned in eight parts and fewer, with ragged record counts and
    with triangles of one pixel to the whole frame."""
    import glimpsw_amd as g

    W, H = 644, 360
    sc = T.ragged(T.small_scene(meshlets, seed_offset=13, spread=8.0, near_frac=0.1))
    view = S.make_view(W, H, count=meshlets)
    ofb, octr, _ = oracle.render_frame(sc, view)
    ds = g.Scene(gpu_ctx, sc)
    fb = g.Framebuffer(gpu_ctx, W, H)
    for cap in (0, 3):
        print(f"[draws] {meshlets} meshlets, capacity {cap}", flush=True)
        gpu_ctx.reset_counters()
        fb.clear(0, 0.0)
        fb.draw(ds, view.object_to_clip, meshlets, 0, view.frustum_planes(), g.GLIMP_DRAW_COUNTERS, bin_capacity=cap)
        ids, depth = fb.read()
        ctr = gpu_ctx.counters()
        assert (ids == ofb.ids()).all()
        assert (depth.view(np.uint32) == ofb.depth().view(np.uint32)).all()
        assert ctr["fragments_covered"] == octr["fragments_covered"] and ctr["dropped"] == 0
    fb.close()
    ds.close()
