"""Texel gradients where one texel's run of pixel records crosses many tiles of
256 records: every pixel on one texel, at the numbers of tiles where the wave
takes over from the thread (8 after the first) and where its steps of 64 end,
and a few texels with runs that start in different tiles. Against the FP64
oracle within the suite's 1e-4 and bitwise reproducible."""
import numpy as np
import pytest

import oracle
from glimpsw_amd import diff as D
from glimpsw_amd import scene as S
from tests import scenes as T

pytestmark = pytest.mark.gpu

GRAD_RTOL = 1e-4


@pytest.mark.parametrize("magnify", [0.0, 0.002])
@pytest.mark.parametrize("width,height", [
    (48, 48),          # 9 tiles
    (64, 40),          # 10
    (96, 192),         # 72
    (292, 64),         # 73
    (292, 68),         # 77.6
    (548, 64),         # 137
])
def test_texel_gradients(gpu_ctx, width, height, magnify):
    import torch
    import glimpsw_amd as g

    print(f"[long runs] {width}x{height} magnify {magnify}", flush=True)
    sc = T.fullscreen_grid(width, height)
    view = S.make_view(width, height, count=sc.count)
    chains = D.chains_from_textures(sc.textures)
    rng = np.random.default_rng(9)
    uv = D.vertex_uv(sc) * np.float32(magnify)
    color = rng.uniform(0.5, 1.5, size=(sc.count * 64, 4)).astype(np.float32)
    gout = rng.normal(0, 1, size=(height, width, 4)).astype(np.float32)
    ofb, _, bind = oracle.render_frame(sc, view)
    assert (ofb.depth() > 0).all()
    want = oracle.diff_backward(ofb, bind, view.object_to_clip, chains, chains.data, uv, color,
                                gout.astype(np.float64))[0]
    ds = g.Scene(gpu_ctx, sc)
    fb = g.render_frame(gpu_ctx, ds, view)
    try:
        op = D.DiffResolve(gpu_ctx, fb, ds, view.object_to_clip, chains)
        args = [torch.from_numpy(a).cuda() for a in (chains.data, uv, color, gout)]
        got = op.backward(*args)[0]
        assert torch.equal(got, op.backward(*args)[0])
        err = np.abs(got.cpu().numpy().astype(np.float64) - want)
        print(f"[long runs]   {np.count_nonzero(want.any(axis=1))} texels {err.max() / np.abs(want).max():.2g}", flush=True)
        assert np.linalg.norm(err) <= GRAD_RTOL * np.linalg.norm(want)
        assert err.max() <= GRAD_RTOL * np.abs(want).max()
    finally:
        fb.close()
        ds.close()
