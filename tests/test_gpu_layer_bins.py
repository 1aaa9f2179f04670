"""The overdraw and deferred pipelines' screen bins where they can go wrong:
framebuffers smaller than a bin and with ragged last bins, bins without
records after a clear and on top of an earlier draw, triangles over many
bins (the coarser bin lists), and bins with more records than their lists
hold (the overflow passes). Layers equal the oracle's bit for bit."""
import dataclasses

import numpy as np
import pytest

import oracle
from glimpsw_amd import scene as S
from tests import scenes as T

pytestmark = pytest.mark.gpu


def _crowded(n, copies):
    """`copies` small patches on top of each other beside n ordinary ones:
    98 triangles each, half of them facing the camera, all in a few bins."""
    sc = T.normal_mapped_scene(n, seed_offset=11, near_frac=0.1)
    pos = sc.positions.copy()
    bounds = sc.bounds.copy()
    g = (np.arange(8) / 7.0 - 0.5) * 0.12
    for i in range(copies):
        z = -3.0 - 0.01 * i
        pos[i, 0] = np.tile(g, 8) + 0.001 * i
        pos[i, 1] = np.repeat(-g, 8)
        pos[i, 2] = z
        bounds[i] = (0.001 * i, 0.0, z, 0.2)
    return dataclasses.replace(sc, positions=pos, bounds=bounds)


@pytest.mark.parametrize("pipeline", ["overdraw", "deferred"])
@pytest.mark.parametrize("width,height,copies", [(4, 4, 0), (20, 12, 0), (132, 68, 0), (516, 260, 0), (1284, 964, 0),
                                                 (132, 68, 40), (516, 260, 90)])
def test_layers_match_oracle(gpu_ctx, pipeline, width, height, copies):
    import glimpsw_amd as g

    print(f"[layers] {pipeline} {width}x{height} crowd {copies}", flush=True)
    sc = _crowded(128, copies)
    view = S.make_view(width, height, count=sc.count)
    kind = {"overdraw": (g.GLIMP_PIPELINE_OVERDRAW, oracle.PIPELINE_OVERDRAW, 2),
            "deferred": (g.GLIMP_PIPELINE_DEFERRED, oracle.PIPELINE_DEFERRED, 3)}[pipeline]
    # two draws on one clear, the first one leaving many bins empty
    draws = [(0, 8), (8, sc.count - 8)]
    b = oracle.SceneBinding(sc)
    ofb = oracle.OracleFramebuffer(width, height, layers=kind[2])
    ofb.clear(0x00030002, 0.0)
    ds = g.Scene(gpu_ctx, sc)
    fb = g.Framebuffer(gpu_ctx, width, height)
    try:
        fb.clear(0x00030002, 0.0)
        for first, count in draws:
            bm, _ = oracle.cull(b, view.frustum_planes(), first, count)
            oracle.draw(ofb, b, view.object_to_clip, count, first, bm, pipeline=kind[1])
            fb.draw(ds, view.object_to_clip, count, first, view.frustum_planes(), pipeline=kind[0])
        for k in range(kind[2]):
            got, want = fb.read_layer(k), ofb.pixels(k)
            assert (got == want).all(), (pipeline, k, int((got != want).sum()))
    finally:
        fb.close()
        ds.close()
