"""Records of meshlets that spread over more than 1,024 screen bins, listed by
the size of their box: up to 64 bins in the bins themselves, then in bins of
4x4 bins, and those over 64 of these in bins of 16x16. Triangles are placed by
the bins their boxes cover, on both sides of each limit, in views of ragged
bins, of exactly 1,024 bins (no coarser level) and of three and six bin rows or
columns, with lists that hold everything and lists that overflow at every
level. Ids and depth equal the oracle's bit for bit; the (record, bin) pairs
the draw counts show that the boxes are as placed."""
import dataclasses

import numpy as np
import pytest

import oracle
from glimpsw_amd import scene as S
from glimpsw_amd import textures

pytestmark = pytest.mark.gpu

COPIES = 20        # meshlets of the same boxes: more than a level-2 bin holds at capacity 1


def _boxes(bx, by):
    """Bin boxes (x0, y0, x1, y1), inclusive, of one meshlet that spans bx x by bins."""
    X, Y = bx - 1, by - 1
    boxes = [(0, 0, 0, 0), (X, Y, X, Y), (0, 0, X, Y), (0, Y, X, Y), (X, 0, X, Y), (1, 0, X, min(Y, 1))]
    if bx >= 36 and by >= 32:
        boxes += [(3, 2, 10, 9),               # 64 bins: not above the limit
                  (3, 2, 11, 9),               # 72 bins: 3 x 3 of level 1
                  (0, 0, 31, 31),              # 8 x 8 of level 1: not above the limit
                  (0, 0, 32, 31),              # 9 x 8 of level 1: level 2
                  (3, 3, 31, 28)]
    return boxes


def _scene(width, height, bin_size, spans):
    """Clip-space triangles (object_to_clip is the identity) over `spans`, one
    meshlet each and copy."""
    rng = np.random.default_rng(11)
    n = len(spans) * COPIES
    sc = S.build_patches(np.zeros((n, 3)), np.tile(np.eye(3), (n, 1, 1)), np.ones(n), np.zeros(n, np.uint32),
                         [(0, True, 255)], [textures.checker_texture(16)])
    pos = np.zeros((n, 3, 64), np.float32)
    idx = np.zeros_like(sc.indices)
    nt, nv = np.zeros(n, np.uint8), np.zeros(n, np.uint8)
    pairs = 0
    for m in range(n):
        for t, (x0, y0, x1, y1) in enumerate(_boxes(*spans[m % len(spans)])):
            left, top = x0 * bin_size + 1, y0 * bin_size + 1
            right, bottom = min((x1 + 1) * bin_size, width) - 1, min((y1 + 1) * bin_size, height) - 1
            for k, (x, y) in enumerate(((left, top), (right, top), (left, bottom))):
                pos[m, :, 3 * t + k] = (2 * x / width - 1, 2 * y / height - 1, rng.uniform(0.1, 0.9))
                idx[m, k, t] = 3 * t + k
            nt[m], nv[m] = t + 1, 3 * t + 3
            pairs += (x1 - x0 + 1) * (y1 - y0 + 1)
    bounds = np.tile(np.float32([0, 0, 0, 10]), (n, 1))
    return dataclasses.replace(sc, positions=pos, indices=idx, num_triangles=nt, num_vertices=nv, bounds=bounds), pairs


@pytest.mark.parametrize("bin_capacity", [0, 1, 3])
@pytest.mark.parametrize("width,height,bin_size,spans", [
    (324, 292, 8, [(41, 37), (33, 32), (32, 32)]),          # 1,517 bins, meshlets over 1,517, 1,056 and 1,024
    (644, 580, 16, [(41, 37), (33, 32), (32, 32)]),
    (1284, 1156, 32, [(41, 37), (33, 32), (32, 32)]),
    (2564, 2308, 64, [(41, 37), (33, 32), (32, 32)]),
    (512, 512, 16, [(32, 32), (20, 20)]),                   # 1,024 bins: no coarser level
    (2880, 24, 8, [(360, 3), (342, 3), (341, 3)]),          # 1,080, 1,026 and 1,023 bins
    (24, 2880, 8, [(3, 360)]),
    (2880, 96, 16, [(180, 6), (171, 6), (170, 6)]),
])
def test_boxes_by_level(gpu_ctx, width, height, bin_size, spans, bin_capacity):
    import glimpsw_amd as g

    print(f"[coarse bins] {width}x{height} bins of {bin_size} capacity {bin_capacity}", flush=True)
    sc, pairs = _scene(width, height, bin_size, spans)
    clip = np.eye(4, dtype=np.float32).reshape(16)
    ofb = oracle.OracleFramebuffer(width, height)
    ofb.clear(0, 0.0)
    octr, _ = oracle.draw(ofb, oracle.SceneBinding(sc), clip, sc.count)
    ds = g.Scene(gpu_ctx, sc)
    fb = g.Framebuffer(gpu_ctx, width, height)
    try:
        gpu_ctx.reset_counters()
        fb.clear(0, 0.0)
        fb.draw(ds, clip, sc.count, 0, None, g.GLIMP_DRAW_COUNTERS, bin_size=bin_size, bin_capacity=bin_capacity)
        ids, depth = fb.read()
        ctr = gpu_ctx.counters()
    finally:
        fb.close()
        ds.close()
    assert (ids == ofb.ids()).all()
    assert (depth.view(np.uint32) == ofb.depth().view(np.uint32)).all()
    assert ctr["bin_entries"] == pairs and ctr["dropped"] == 0
    for name in ("triangles_processed", "triangles_rasterized", "triangles_clipped", "fragments_covered"):
        assert ctr[name] == octr[name], name
