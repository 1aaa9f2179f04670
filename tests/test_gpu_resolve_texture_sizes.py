"""The resolve's level and filter choice where a wave's tiles mix textures of
different sizes, aspect ratios and none at all (votes per size), beside scenes
of one size (one vote for the wave): base colour and lit image equal the
oracle's."""
import dataclasses

import numpy as np
import pytest

import oracle
from glimpsw_amd import scene as S
from glimpsw_amd import textures
from tests import scenes as T

pytestmark = pytest.mark.gpu


def _wide(w, h, seed):
    rng = np.random.default_rng(seed)
    return textures.create([rng.integers(0, 1 << 32, size=(h, w), dtype=np.uint32) | np.uint32(0xFF000000)])


@pytest.mark.parametrize("sizes", [[(64, 64)], [(64, 64), (64, 64)], [(16, 16), (512, 512), (128, 128)],
                                   [(256, 64), (64, 256), None], [(4, 4), None, (1024, 1024)]])
@pytest.mark.parametrize("width,height", [(4, 4), (132, 100)])
def test_mixed_texture_sizes(gpu_ctx, sizes, width, height):
    import glimpsw_amd as g

    print(f"[resolve sizes] {sizes} {width}x{height}", flush=True)
    sc = T.small_scene(256, seed_offset=13, spread=5.0, near_frac=0.1)
    texs, mats = [], []
    for i, s in enumerate(sizes):
        mats.append((-1 if s is None else len(texs), False, 255))
        if s is not None:
            texs.append(_wide(*s, seed=i))
    sc = dataclasses.replace(sc, materials=mats, textures=texs,
                             material_id=(np.arange(sc.count) % len(mats)).astype(np.uint32))
    view = S.make_view(width, height, count=sc.count)
    lighting = S.default_lighting(view)
    ds = g.Scene(gpu_ctx, sc)
    fb = g.render_frame(gpu_ctx, ds, view)
    try:
        fb.resolve(ds, view.object_to_clip, g.GLIMP_RESOLVE_ALBEDO)
        albedo = fb.read_color()
        fb.resolve(ds, view.object_to_clip, g.GLIMP_RESOLVE_LIT, lighting)
        lit = fb.read_color()
    finally:
        fb.close()
        ds.close()
    ofb, _, b = oracle.render_frame(sc, view)
    assert (albedo == oracle.resolve_albedo(ofb, b, view.object_to_clip)).all()
    ofb, _, _ = oracle.render_frame(sc, view, b)
    assert (lit == oracle.resolve_lit(ofb, b, view.object_to_clip, lighting)).all()
