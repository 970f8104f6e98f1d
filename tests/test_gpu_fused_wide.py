"""A frame so wide that its top level has more than 2^16 tiles across: the tiles
of the level below still wait for the ones that they read."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_more_tiles_across_than_16_bits_count(ffo):
    import flowfilter.gpu.flowfilters as gf
    # 12 smoothing iterations leave 10 of a tile's 64 columns
    h, w, smooth = 8, 2 * (10 * 2 ** 16 + 5000), [1, 12]
    print("wide frame", (h, w), flush=True)
    rng = np.random.default_rng(3)
    base = rng.integers(0, 256, (h, w + 3), dtype=np.uint8)
    f = gf.PyramidalFlowFilter(h, w, 2)
    o = ffo.PyramidalFlowFilter(h, w, 2)
    f.gamma, f.maxflow, f.smoothIterations = [10.0, 30.0], 4.0, smooth
    o.configure_like([10.0, 30.0], 4.0, smooth)
    for t in range(3):
        img = np.ascontiguousarray(base[:, t:t + w])
        f.loadImage(img)
        f.compute()
        o.compute(img)
        print("frame", t, flush=True)
        assert np.array_equal(f.getFlow(), o.downloadFlow()), t
    assert f.waitTimeouts() == 0
