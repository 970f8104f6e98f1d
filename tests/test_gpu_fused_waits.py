"""Waits of a fused frame for single tiles of the level above, and launches
with such waits from several streams side by side, through the C ABI.

Bar: flow and brightness bitwise the oracle's, and no wait gives up. The
sizes and smoothing counts put the tiles of the two levels in different
proportions: an upper tile that covers many of the level below, upper tiles so
small that one tile waits for a grid of them, a last row and column of one
pixel, levels of a single tile, odd sizes (where the upper-level index is not
x >> 1).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [  # h, w, levels, maxflow, smooth per level
    (272, 512, 2, 4.0, [2, 2]),
    (257, 401, 2, 4.0, [1, 10]),
    (193, 391, 2, 2.0, [12, 1]),
    (195, 290, 3, 4.0, [2, 2, 12]),
    (97, 130, 2, 1.0, [1, 1]),
    (64, 900, 2, 3.0, [3, 6]),
    (300, 66, 2, 3.0, [1, 9]),
]


@pytest.mark.parametrize("h,w,levels,maxflow,smooth", CASES)
def test_tile_waits_on_two_streams_match_oracle(ffo, h, w, levels, maxflow, smooth):
    import flowfilter.gpu.flowfilters as gf
    from flowfilter import synthetic
    print("tile waits", (h, w), levels, maxflow, smooth, flush=True)
    gamma = [10.0, 30.0, 50.0][:levels]
    frames = list(synthetic.blob_affine(h, w, 5, blobs=30, seed=h))
    filters = []
    for _ in range(2):  # each on a stream of its own
        f = gf.PyramidalFlowFilter(h, w, levels)
        f.gamma, f.maxflow, f.smoothIterations = gamma, maxflow, smooth
        filters.append(f)
    o = ffo.PyramidalFlowFilter(h, w, levels)
    o.configure_like(gamma, maxflow, smooth)
    for t, img in enumerate(frames):
        for f in filters:
            f.loadImage(img)
        for f in filters:
            f.compute()
        o.compute(img)
        for k, f in enumerate(filters):
            assert np.array_equal(f.getFlow(), o.downloadFlow()), (t, k)
            assert np.array_equal(f.getImage(), o.downloadImage()), (t, k)
    assert all(f.waitTimeouts() == 0 for f in filters)
