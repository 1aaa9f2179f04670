"""The backward's runs where they can go wrong: views smaller than a pixel
block, ragged ones, triangles that cover a whole view (a meshlet's vertex
gradients in several parts), more views than one pass over the marked cells
takes, and one texel for every pixel (a run over all record tiles). Gradients
against the FP64 oracle within the suite's 1e-4 and bitwise reproducible."""
import numpy as np
import pytest

import oracle
from glimpsw_amd import diff as D
from glimpsw_amd import scene as S
from tests import scenes as T

pytestmark = pytest.mark.gpu

GRAD_RTOL = 1e-4


@pytest.mark.parametrize("sizes,magnify", [
    ([(4, 4)], 0.02),
    ([(20, 12)], 0.02),
    ([(260, 516)], 0.02),              # 17 x 33 blocks, cells of 2 x 3
    ([(260, 516)], 0.0),               # every pixel samples the same texel
    ([(8, 8)] * 40, 0.02),
    ([(16, 16), (84, 20), (300, 4)], 0.3),
])
def test_gradients(gpu_ctx, sizes, magnify):
    import torch
    import glimpsw_amd as g

    print(f"[diff runs] {sizes[:3]} x{len(sizes)} magnify {magnify}", flush=True)
    sc = T.small_scene(96, seed_offset=21, spread=4.0, near_frac=0.4)
    ds = g.Scene(gpu_ctx, sc)
    views = [S.make_view(w, h, count=sc.count, view=S.view_matrix((0.0, 0.0, 0.0), 0.13 * i, 0.0))
             for i, (w, h) in enumerate(sizes)]
    fbs = [g.render_frame(gpu_ctx, ds, v) for v in views]
    chains = D.chains_from_textures(sc.textures)
    uv = D.vertex_uv(sc) * np.float32(magnify)
    rng = np.random.default_rng(3)
    color = rng.uniform(0.5, 1.5, size=(sc.count * 64, 4)).astype(np.float32)
    texels_t, uv_t, color_t = (torch.from_numpy(a).cuda() for a in (chains.data, uv, color))
    op = D.DiffResolveViews(gpu_ctx, ds, [(fb, v.object_to_clip) for fb, v in zip(fbs, views)], chains)
    gout = torch.from_numpy(rng.normal(0, 1, size=(op.binding.total_pixels, 4)).astype(np.float32)).cuda()
    try:
        grads = op.backward(texels_t, uv_t, color_t, gout)
        again = op.backward(texels_t, uv_t, color_t, gout)
        for a, b in zip(grads, again):
            assert torch.equal(a, b)
        ref = [np.zeros((chains.num_texels, 4)), np.zeros((uv.shape[0], 2)), np.zeros((color.shape[0], 4))]
        for v, part in zip(views, op.split(gout)):
            ofb, _, bind = oracle.render_frame(sc, v)
            g64 = oracle.diff_backward(ofb, bind, v.object_to_clip, chains, chains.data, uv, color,
                                       part.cpu().numpy().astype(np.float64))
            for r, x in zip(ref, g64):
                r += x
        for name, gg, r in zip(("texels", "uv", "color"), grads, ref):
            got = gg.cpu().numpy().astype(np.float64)
            norm = np.linalg.norm(r)
            if norm == 0:
                assert not got.any(), name
                continue
            rel, elem = np.linalg.norm(got - r) / norm, np.abs(got - r).max() / np.abs(r).max()
            print(f"[diff runs]   {name}: {rel:.2g} {elem:.2g}", flush=True)
            assert rel <= GRAD_RTOL and elem <= GRAD_RTOL, (name, rel, elem)
    finally:
        for fb in fbs:
            fb.close()
        ds.close()
