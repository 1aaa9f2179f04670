"""Frames of few screen bins and many meshlets, on both sides of the sizes at
which a draw's default lists change (2, 4 and 24 bins, two bin rows, 512
meshlets a bin), so that most records are drawn from the bins or most from the
overflow list. All three pipelines, two draws on one clear; layers equal the
oracle's bit for bit."""
import pytest

import oracle
from glimpsw_amd import scene as S
from tests import scenes as T

pytestmark = pytest.mark.gpu

PIPELINES = {"visbuffer": (0, oracle.PIPELINE_VISBUFFER, 2), "overdraw": (2, oracle.PIPELINE_OVERDRAW, 2),
             "deferred": (1, oracle.PIPELINE_DEFERRED, 3)}


@pytest.fixture(scope="module")
def scene():
    return T.normal_mapped_scene(2200, seed_offset=13, spread=5.0, near_frac=0.01)


@pytest.mark.parametrize("pipeline", list(PIPELINES))
@pytest.mark.parametrize("width,height,count", [
    (16, 16, 90),
    (32, 16, 2200),
    (32, 32, 2048),          # 4 bins: long lists up to 2,048 meshlets
    (32, 32, 2049),
    (92, 52, 2200),          # 24 bins
    (92, 48, 2200),          # 18 bins
    (336, 32, 2200),         # two rows of 21 bins
    (336, 36, 2200),         # three
])
def test_layers_match_oracle(gpu_ctx, scene, pipeline, width, height, count):
    import glimpsw_amd as g

    print(f"[tiny frames] {pipeline} {width}x{height} meshlets {count}", flush=True)
    kind = PIPELINES[pipeline]
    assert (g.GLIMP_PIPELINE_DEFERRED, g.GLIMP_PIPELINE_OVERDRAW) == (1, 2)
    view = S.make_view(width, height, count=scene.count)
    b = oracle.SceneBinding(scene)
    ofb = oracle.OracleFramebuffer(width, height, layers=kind[2])
    ofb.clear(0x00030002, 0.0)
    ds = g.Scene(gpu_ctx, scene)
    fb = g.Framebuffer(gpu_ctx, width, height)
    try:
        fb.clear(0x00030002, 0.0)
        for first, n in ((0, count), (scene.count - 40, 40)):
            bm, _ = oracle.cull(b, view.frustum_planes(), first, n)
            oracle.draw(ofb, b, view.object_to_clip, n, first, bm, pipeline=kind[1])
            fb.draw(ds, view.object_to_clip, n, first, view.frustum_planes(), pipeline=kind[0])
        for k in range(kind[2]):
            got, want = fb.read_layer(k), ofb.pixels(k)
            assert (got == want).all(), (pipeline, k, int((got != want).sum()))
    finally:
        fb.close()
        ds.close()
