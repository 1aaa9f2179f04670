"""Texture tables whose entries share texels: one range under another width,
row windows of a texture, a range at the array's end under a larger width,
levels inside another texture's level 0, and entries of the very same range.
The backward's texel gradients against the FP64 oracle within the suite's
1e-4, bitwise reproducible."""
import numpy as np
import pytest

import oracle
from glimpsw_amd import diff as D
from glimpsw_amd import scene as S
from glimpsw_amd import textures
from tests import scenes as T

pytestmark = pytest.mark.gpu

GRAD_RTOL = 1e-4

# name: texels, (width, height, levels) and level offsets per texture
TABLES = {
    "other width": (512, [(32, 16, 1), (16, 32, 1), (32, 16, 1)], [[0], [0], [0]]),
    "row windows": (512, [(32, 16, 1), (32, 8, 1), (32, 8, 1)], [[0], [128], [256]]),
    "array end": (520, [(8, 8, 1), (64, 2, 1), (32, 4, 1)], [[456], [392], [392]]),
    "shifted": (640, [(16, 16, 1), (16, 16, 1), (1, 256, 1)], [[0], [7], [300]]),
    "nested levels": (1024, [(32, 32, 3), (16, 16, 2), (16, 16, 1)], [[0, 512, 40], [700, 256], [256]]),
    "same range": (512, [(16, 16, 1), (16, 16, 1), (16, 16, 1)], [[256], [256], [0]]),
}


@pytest.mark.parametrize("magnify", [0.1, 0.3])
@pytest.mark.parametrize("table", list(TABLES))
def test_gradients(gpu_ctx, table, magnify):
    import torch
    import glimpsw_amd as g

    print(f"[shared texels] {table} magnify {magnify}", flush=True)
    rng = np.random.default_rng(5)
    num_texels, sizes, offsets = TABLES[table]
    chains = D.TexelChains(rng.uniform(0, 1, size=(num_texels, 4)).astype(np.float32), sizes, offsets)
    n = 96
    base = T.small_scene(n, seed_offset=21, spread=4.0, near_frac=0.1)
    tex = textures.checker_texture(16)
    sc = S.dataclasses.replace(base, material_id=(np.arange(n) % 3).astype(np.uint32),
                               materials=[(i, False, 255) for i in range(3)], textures=[tex] * 3)
    view = S.make_view(260, 132, count=sc.count)
    # each meshlet's UVs around a point of its own, so most of the texture shows
    uv = D.vertex_uv(sc) * np.float32(magnify) + np.repeat(rng.uniform(0, 1, size=(n, 2)), 64, axis=0).astype(np.float32)
    color = rng.uniform(0.5, 1.5, size=(sc.count * 64, 4)).astype(np.float32)
    gout = rng.normal(0, 1, size=(view.height, view.width, 4)).astype(np.float32)

    ofb, _, bind = oracle.render_frame(sc, view)
    want = oracle.diff_backward(ofb, bind, view.object_to_clip, chains, chains.data, uv, color,
                                gout.astype(np.float64))[0]
    assert np.count_nonzero(want.any(axis=1)) > 100

    ds = g.Scene(gpu_ctx, sc)
    fb = g.render_frame(gpu_ctx, ds, view)
    try:
        op = D.DiffResolve(gpu_ctx, fb, ds, view.object_to_clip, chains)
        args = [torch.from_numpy(a).cuda() for a in (chains.data, uv, color, gout)]
        got = op.backward(*args)[0]
        assert torch.equal(got, op.backward(*args)[0])
        err = np.abs(got.cpu().numpy().astype(np.float64) - want)
        print(f"[shared texels]   {err.max() / np.abs(want).max():.2g}", flush=True)
        assert np.linalg.norm(err) <= GRAD_RTOL * np.linalg.norm(want)
        assert err.max() <= GRAD_RTOL * np.abs(want).max()
    finally:
        fb.close()
        ds.close()
