"""Several iterations of a stage in one launch (ff_tiles.hip) against the CPU
oracle, bitwise, at sizes on both sides of a tile's edges: images smaller than
a buffer (64 columns, 32 or 64 rows) across or down, one pixel more, whole
tiles and remainders, enough tiles for the taller workgroups, more iterations
than one launch takes; and the inputs that the tile kernels leave to the
single passes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(2, 3), (31, 63), (32, 64), (33, 65), (64, 200), (65, 130), (57, 113), (200, 57), (700, 900)]


def _img(a):
    from flowfilter.gpu.image import GPUImage
    g = GPUImage(a.shape, 4)
    g.upload(np.ascontiguousarray(a))
    return g


def _fields(h, w, seed):
    r = np.random.default_rng(seed)
    f = (r.standard_normal((h, w, 2)) * 2.0).astype(np.float32)
    return f, r.random((h, w), np.float32), r.standard_normal((h, w, 2)).astype(np.float32)


def _same(a, b):
    # (these flows are faster than the scheme is stable for: at some sizes the
    # oracle overflows, and the same pixels must be NaN)
    return np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("h,w", SIZES)
@pytest.mark.parametrize("n", [1, 3, 4, 5, 9])
def test_iterations_match_oracle(ffo, h, w, n):
    from flowfilter.gpu.flowsmoothing import FlowSmoother
    from flowfilter.gpu.propagation import FlowPropagator, FlowPropagatorPayload, LaxWendroffPropagator
    print("tiles", (h, w), n, flush=True)
    f, s, v = _fields(h, w, h * w + n)
    for border in (0, 1, 3):
        p = FlowPropagator(_img(f), n)
        p.border = border
        p.compute()
        assert _same(p.getPropagatedFlow().download(np.float32), ffo.propagate(f, n, border=border)), border
        q = FlowPropagatorPayload(_img(f), _img(s), _img(v), n)
        q.border = border
        q.compute()
        rf, rs, rv = ffo.propagate_payload(f, s, v, n, border=border)
        assert _same(q.getPropagatedFlow().download(np.float32), rf), border
        assert _same(q.getPropagatedScalar().download(np.float32), rs), border
        assert _same(q.getPropagatedVector().download(np.float32), rv), border
    m = FlowSmoother(_img(f), n)
    m.compute()
    assert _same(m.getSmoothedFlow().download(np.float32), ffo.smooth(f, n))
    lw = LaxWendroffPropagator(_img(f), _img(s))
    lw.iterations = n
    lw.compute()
    assert _same(lw.getPropagatedImage().download(np.float32), ffo.lax_wendroff(f, s, n))


@pytest.mark.parametrize("n", [1, 2, 5])
def test_own_output_as_input(ffo, n):
    """A stage whose input is its own output buffer (set after it was made)
    still reads all of it before it is overwritten."""
    from flowfilter.gpu.flowsmoothing import FlowSmoother
    from flowfilter.gpu.propagation import FlowPropagator
    f, _, _ = _fields(70, 150, n)
    p = FlowPropagator(_img(f), n)
    p.border = 1
    p.compute()
    p.invertInputFlow = True
    p.compute()
    assert _same(p.getPropagatedFlow().download(np.float32), ffo.propagate(f, n, border=1, invert=True))
    m = FlowSmoother(_img(f), n)
    m.compute()
    want = m.getSmoothedFlow().download(np.float32)
    m.setInputFlow(m.getSmoothedFlow())
    m.configure()
    m.compute()  # the buffers are new ones: the input is the old output
    assert _same(m.getSmoothedFlow().download(np.float32), ffo.smooth(want, n))
