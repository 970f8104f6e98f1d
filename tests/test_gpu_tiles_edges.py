"""Calls that the tile kernels (ff_tiles.hip) take, at the edges of what they
accept: results that overlap inputs, sizes beyond 32-bit offsets, many
iterations, and what the profile counts of them."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _stream():
    import torch
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _p(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else None


@pytest.mark.parametrize("B,h,w", [(1, 5, 7), (2, 33, 65), (3, 130, 200)])
@pytest.mark.parametrize("acc", [0, 1])
def test_image_model_adjoint_that_overlaps_its_inputs(B, h, w, acc):
    """The result anywhere in the gradients it is computed from is bitwise the
    result beside them: at the start, inside and in the second half of the
    image gradient's, and one row into the brightness'."""
    import torch
    from flowfilter import _native as N
    print("image model adjoint", (B, h, w), acc, flush=True)
    g = torch.Generator(device="cuda").manual_seed(h)
    n = B * h * w
    ga = torch.randn(n, generator=g, device="cuda")
    gg = torch.randn(2 * n, generator=g, device="cuda")
    work = torch.empty(B, 2 * h, w, device="cuda")
    call = lambda a, d, o: N.call("ff_ad_image_model_backward", _p(a), _p(d), _p(o), _p(work), B, h, w, acc, _stream())
    for base, off in (("gg", 0), ("gg", 2 * w), ("gg", n - 1), ("gg", n), ("gg", 2 * n - 2), ("ga", w), ("ga", n - 1)):
        buf = {"ga": torch.cat([ga, ga[:n]]), "gg": torch.cat([gg, gg[:n]])}
        out = buf[base][off:off + n]
        want = out.clone()
        call(ga, gg, want)
        call(buf["ga"][:n], buf["gg"][:2 * n], out)
        assert torch.equal(out, want), (base, off)


@pytest.mark.parametrize("n", [1, 4, 9])
def test_profile_counts_every_launch(n):
    """Launches of several iterations are bracketed and counted one by one,
    under the names that the header lists; the single passes under theirs."""
    from flowfilter import _native as N
    from flowfilter.gpu.flowsmoothing import FlowSmoother
    from flowfilter.gpu.image import GPUImage
    from flowfilter.gpu.propagation import FlowPropagator, FlowPropagatorPayload, LaxWendroffPropagator
    print("profile", n, flush=True)
    h, w = 70, 150

    def img(*shape):
        g = GPUImage(shape, 4)
        g.upload(np.full(shape, 0.25, np.float32))
        return g

    flow, one = img(h, w, 2), img(h, w)
    lw = LaxWendroffPropagator(flow, one)
    lw.iterations = n
    stages = [(FlowPropagator(flow, n), "propagate_tile", 4), (FlowPropagatorPayload(flow, one, flow, n), "propagate_payload_tile", 4),
              (FlowSmoother(flow, n), "smooth_tile", 4), (lw, "lax_wendroff_tile", 8)]
    passes = FlowPropagatorPayload(flow, one, flow, n)
    passes.border = 0
    for st, name, most in stages + [(passes, "propagate_payload_x", 1), (passes, "propagate_payload_y", 1)]:
        N.profile_begin(name)
        st.compute()
        ms, launches = N.profile_end()
        assert launches == -(-n // most) and ms > 0.0, name


def test_rows_of_two_gib(ffo):
    """Rows longer than 32-bit offsets reach run in the single passes, with
    64-bit offsets: bitwise the oracle's on crops at both ends and in the
    middle (their edges left out)."""
    import torch
    from flowfilter.gpu.flowsmoothing import FlowSmoother
    from flowfilter.gpu.image import GPUImage
    from flowfilter.gpu.propagation import FlowPropagator
    h, w = 3, 2 ** 28 + 70
    print("rows of 2 GiB", (h, w), flush=True)
    g = torch.Generator(device="cuda").manual_seed(1)
    img = GPUImage((h, w, 2), 4)
    flow = torch.from_dlpack(img)
    for row in flow:
        row.uniform_(-1.0, 1.0, generator=g)
    torch.cuda.synchronize()
    starts = (0, w // 2 - 100, w - 200)

    def check(got, oracle):
        got = torch.from_dlpack(got)
        for x in starts:
            want = oracle(flow[:, x:x + 200].cpu().numpy())
            inner = slice(0 if x == 0 else 10, 200 if x == starts[-1] else 190)
            assert np.array_equal(got[:, x:x + 200].cpu().numpy()[:, inner], want[:, inner]), x

    p = FlowPropagator(img, 2)
    p.border = 1
    p.compute()
    check(p.getPropagatedFlow(), lambda a: ffo.propagate(a, 2, border=1))
    del p
    m = FlowSmoother(img, 2)
    m.compute()
    check(m.getSmoothedFlow(), lambda a: ffo.smooth(a, 2))


@pytest.mark.parametrize("n", [1, 3, 9])
def test_lax_wendroff_of_its_own_output(ffo, n):
    """A Lax-Wendroff propagator fed its own output buffer (set after it was
    made) reads all of it before it is overwritten, frame after frame."""
    from flowfilter.gpu.image import GPUImage
    from flowfilter.gpu.propagation import LaxWendroffPropagator
    print("own output", n, flush=True)
    rng = np.random.default_rng(n)
    h, w = 70, 150
    f = (rng.standard_normal((h, w, 2)) * 0.3).astype(np.float32)
    a = rng.random((h, w), np.float32)
    flow, img = GPUImage((h, w, 2), 4), GPUImage((h, w), 4)
    flow.upload(f)
    img.upload(a)
    p = LaxWendroffPropagator(flow, img)
    p.iterations = n
    for _ in range(3):
        p.compute()
        a = ffo.lax_wendroff(f, a, n)
        assert np.array_equal(p.getPropagatedImage().download(np.float32), a)
        p.setInputImage(p.getPropagatedImage())
