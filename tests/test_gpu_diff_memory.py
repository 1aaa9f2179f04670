"""Device memory of the backward's workspace: a small fit, whose meshlets'
vertex gradients are never split into parts, takes none for the parts' sums."""
import numpy as np
import pytest

from glimpsw_amd import diff as D
from glimpsw_amd import scene as S
from tests import scenes as T

pytestmark = pytest.mark.gpu


def _backward(ctx, sc, size):
    import torch
    import glimpsw_amd as g

    view = S.make_view(*size, count=sc.count)
    chains = D.chains_from_textures(sc.textures)
    ds = g.Scene(ctx, sc)
    fb = g.render_frame(ctx, ds, view)
    try:
        op = D.DiffResolve(ctx, fb, ds, view.object_to_clip, chains)
        args = [torch.from_numpy(a).cuda() for a in
                (chains.data, D.vertex_uv(sc), np.ones((sc.count * 64, 4), np.float32))]
        args.append(torch.ones((size[1], size[0], 4), device="cuda"))
        op.backward(*args)                 # torch's own buffers
        torch.cuda.synchronize()
    finally:
        fb.close()
        ds.close()


def test_small_fit_workspace(gpu_ctx):
    import torch
    import glimpsw_amd as g

    sc = T.small_scene(96, seed_offset=21, spread=4.0, near_frac=0.4)
    _backward(gpu_ctx, sc, (64, 64))       # code and torch's buffers loaded
    ctx = g.Context(0)
    try:
        before = torch.cuda.mem_get_info()[0]
        _backward(ctx, sc, (64, 64))
        used = before - torch.cuda.mem_get_info()[0]
        print(f"[diff memory] 64x64 fit: {used >> 20} MiB", flush=True)
        # 4,096 pixels at about 260 bytes, a draw's scratch of 96 meshlets (4 MiB), allocation granules
        assert used < 32 << 20
    finally:
        ctx.close()
