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


@pytest.mark.parametrize("B,h,w", [(1, 33, 65), (3, 57, 113), (2, 130, 200)])
@pytest.mark.parametrize("n,after", [(1, 0), (2, 1), (3, 2), (4, 2)])
@pytest.mark.parametrize("pay", [False, True])
def test_ad_steps_match_single_passes(B, h, w, n, after, pay):
    """ff_ad_propagate_steps (with the fields in between) and
    ff_ad_smooth_steps on a batch are bitwise the single passes."""
    import ctypes

    import torch
    from flowfilter import _native as N
    print("ad steps", (B, h, w), n, after, pay, flush=True)
    g = torch.Generator(device="cuda").manual_seed(h * n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda") * 0.7
    new = lambda: [torch.empty(B, h, w, 2, device="cuda")] + ([torch.empty(B, h, w, device="cuda"),
                                                             torch.empty(B, h, w, 2, device="cuda")] if pay else [])
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    arg = lambda fs: [p(t) for t in fs] + [None] * (3 - len(fs))
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    dt = ctypes.c_float(1.0 / n)
    fields = [rnd(B, h, w, 2)] + ([rnd(B, h, w), rnd(B, h, w, 2)] if pay else [])
    ref, kept = fields, None
    for k in range(n):
        for axis in (0, 1):
            out = new()
            N.call("ff_ad_propagate_pass", axis, *arg(ref), *arg(out), B, h, w, dt, 3, s)
            ref = out
        if k + 1 == after:
            kept = ref
    mid, out = (new() if after else []), new()
    N.call("ff_ad_propagate_steps", *arg(fields), n, after, *arg(mid), *arg(out), B, h, w, dt, 3, s)
    assert all(torch.equal(a, b) for a, b in zip(ref, out))
    if after:
        assert all(torch.equal(a, b) for a, b in zip(kept, mid))
    sm, got = fields[0], torch.empty_like(fields[0])
    for _ in range(n):
        o = torch.empty_like(sm)
        N.call("ff_ad_smooth_pair", p(sm), p(o), B, h, w, s)
        sm = o
    N.call("ff_ad_smooth_steps", p(fields[0]), p(got), n, B, h, w, s)
    assert torch.equal(sm, got)


@pytest.mark.parametrize("B,h,w", [(2, 1, 1), (1, 2, 4), (3, 5, 3), (1, 31, 63), (2, 33, 65), (1, 61, 60), (3, 130, 122)])
@pytest.mark.parametrize("n", [1, 2, 3])
@pytest.mark.parametrize("second,acc", [(False, 0), (True, 1)])
def test_ad_tile_adjoints(B, h, w, n, second, acc):
    """The smoothing iterations' adjoint is bitwise that many single
    iterations'; the image model's adjoint is the transpose of the image model:
    <g, M x> = <M^T g, x> in float64 sums of float32 results, to 1e-5 of the
    terms' magnitude (a few float32 roundings each)."""
    import ctypes

    import torch
    from flowfilter import _native as N
    print("ad adjoints", (B, h, w), n, second, acc, flush=True)
    g = torch.Generator(device="cuda").manual_seed(h * 7 + n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr()) if t is not None else None
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    a, b = rnd(B, h, w, 2), rnd(B, h, w, 2) if second else None
    base = rnd(B, h, w, 2)
    ref, two = a, b
    for k in range(n):
        last = k == n - 1
        o = base.clone() if last and acc else torch.empty_like(a)
        N.call("ff_ad_smooth_pair_backward", p(ref), p(two), p(o), B, h, w, acc if last else 0, s)
        ref, two = o, None
    got = base.clone() if acc else torch.empty_like(a)
    N.call("ff_ad_smooth_steps_backward", p(a), p(b), p(got), n, B, h, w, acc, s)
    assert torch.equal(ref, got)
    img, ga, gg = rnd(B, h, w), rnd(B, h, w), rnd(B, h, w, 2)
    a0, gr, work = torch.empty_like(img), torch.empty_like(gg), torch.empty(B, 2 * h, w, device="cuda")
    N.call("ff_ad_image_model", p(img), p(a0), p(gr), B, h, w, s)
    out = base[..., 0].contiguous() if acc else torch.empty_like(img)
    start = out.double().clone() if acc else 0.0
    N.call("ff_ad_image_model_backward", p(ga), p(gg), p(out), p(work), B, h, w, acc, s)
    left = (ga.double() * a0.double()).sum() + (gg.double() * gr.double()).sum()
    terms = (out.double() - start) * img.double()
    scale = terms.abs().sum() + (ga.double() * a0.double()).abs().sum() + (gg.double() * gr.double()).abs().sum()
    assert abs(float(left - terms.sum())) <= 1e-5 * float(scale)
    # in place, through the work buffer
    inplace = ga.clone()
    N.call("ff_ad_image_model_backward", p(inplace), p(gg), p(inplace), p(work), B, h, w, 0, s)
    plain = torch.empty_like(img)
    N.call("ff_ad_image_model_backward", p(ga), p(gg), p(plain), p(work), B, h, w, 0, s)
    assert torch.equal(inplace, plain)


@pytest.mark.parametrize("B,h,w,border", [(1, 80, 180, 1), (2, 57, 122, 1), (1, 81, 181, 3), (1, 49, 113, 20),
                                          (1, 120, 240, 2)])
@pytest.mark.parametrize("pay", [False, True])
@pytest.mark.parametrize("special", [False, True])
def test_ad_two_iterations_adjoint(B, h, w, border, pay, special):
    """The adjoint of two propagation iterations in one launch, at sizes with
    workgroups wholly inside the border (and one pixel short of that), is
    bitwise the adjoints of the two iterations, infinite and NaN flows and
    gradients included."""
    import ctypes

    import torch
    from flowfilter import _native as N
    print("ad two iterations", (B, h, w), border, pay, special, flush=True)
    g = torch.Generator(device="cuda").manual_seed(h * 5 + w)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr()) if t is not None else None
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    dt = ctypes.c_float(0.25)
    new = lambda: [rnd(B, h, w, 2), rnd(B, h, w) if pay else None, rnd(B, h, w, 2) if pay else None]
    f, go, mid, gmid, ref = new(), new(), new(), new(), new()
    if special:
        for k, t in enumerate((f[0], go[0])):
            for i, v in enumerate((float("inf"), float("nan"), -float("inf"))):
                t[0, (7 + 17 * i + 31 * k) % h, (5 + 41 * i + 23 * k) % w, i % 2] = v
                t[-1, 0, (60 * i + k) % w, 0] = v
    got = [t.clone() if t is not None else None for t in ref]
    acc = 5  # (added to the flow's and the vector's, the scalar's written)
    N.call("ff_ad_propagate_pair", *map(p, f), None, None, None, *map(p, mid), B, h, w, dt, border, s)
    N.call("ff_ad_propagate_pair_backward", *map(p, mid), None, None, None, *map(p, go), *map(p, gmid), B, h, w, dt,
           border, 0, s)
    N.call("ff_ad_propagate_pair_backward", *map(p, f), None, None, None, *map(p, gmid), *map(p, ref), B, h, w, dt,
           border, acc, s)
    N.call("ff_ad_propagate_quad_backward", *map(p, f), *map(p, go), *map(p, got), B, h, w, dt, border, acc, s)
    for a, b in zip(ref, got):
        if a is not None:
            assert torch.equal(torch.isnan(a), torch.isnan(b))
            assert torch.equal(torch.nan_to_num(a, nan=0.0), torch.nan_to_num(b, nan=0.0))


@pytest.mark.parametrize("B,h,w", [(1, 2, 3), (2, 31, 63), (1, 33, 65), (3, 64, 57), (2, 130, 200), (1, 420, 700)])
@pytest.mark.parametrize("n,K", [(0, 1), (1, 0), (2, 1), (3, 2), (4, 1), (7, 1), (9, 3)])
@pytest.mark.parametrize("delta", [False, True])
def test_ad_level_matches_stages(B, h, w, n, K, delta):
    """A level in one launch is bitwise its stages' own launches: the new state,
    the unsmoothed flow, and what is kept for the adjoints; an infinite and a
    NaN brightness included."""
    import ctypes

    import torch
    from flowfilter import _native as N
    from flowfilter.autograd import FilterSpec, _Level, _propagate
    print("ad level", (B, h, w), n, K, delta, flush=True)
    g = torch.Generator(device="cuda").manual_seed(h + 3 * w + n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr()) if t is not None else None
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    f32 = ctypes.c_float
    dt, border, gamma, maxflow = 1.0 / max(n, 1), 1 + n % 3, 3e-4, 2.5
    hu, wu = max(h // 2, 1), max(w // 2, 1)
    image, flow, bright = rnd(B, h, w).abs(), rnd(B, h, w, 2), rnd(B, h, w).abs()
    bright[0, h // 2, w // 3], bright[-1, h // 3, w // 2] = float("inf"), float("nan")
    dflow, upper = (rnd(B, h, w, 2), rnd(B, hu, wu, 2)) if delta else (None, None)
    maps = FilterSpec(max(h, 2), max(w, 2), 2).levels[0]
    # the stages
    a0, gr = torch.empty_like(image), torch.empty_like(flow)
    N.call("ff_ad_image_model", p(image), p(a0), p(gr), B, h, w, s)
    fields = (flow, bright if delta else None, dflow)
    prop, passes = _propagate(fields, n, dt, border, B, h, w, True, s)
    upd, dn = torch.empty_like(flow), torch.empty_like(flow)
    if delta:
        N.call("ff_ad_delta_update", p(a0), p(gr), p(prop[1]), p(prop[2]), p(upper), p(maps["xmap"]), p(maps["ymap"]),
               p(dn), p(upd), B, h, w, hu, wu, f32(gamma), f32(maxflow), s)
    else:
        N.call("ff_ad_update", p(a0), p(gr), p(bright), p(prop[0]), p(upd), B, h, w, f32(gamma), f32(maxflow), s)
    sm = upd
    for _ in range(K):
        o = torch.empty_like(sm)
        N.call("ff_ad_smooth_pair", p(sm), p(o), B, h, w, s)
        sm = o
    same = lambda a, b: torch.equal(torch.nan_to_num(a, 7e7), torch.nan_to_num(b, 7e7))
    for save in (False, True):
        new = lambda *shape: torch.full(shape, -5.0, device="cuda")
        mids = max((n + 1) // 2 - 1, 0)
        got = dict(flow_out=new(B, h, w, 2), bright_out=new(B, h, w))
        ref = dict(flow_out=sm, bright_out=a0)
        if delta:
            got["dflow_out"], ref["dflow_out"] = new(B, h, w, 2), dn
        else:
            got["flow_upd"], ref["flow_upd"] = new(B, h, w, 2), upd
        if save:
            got["grad"], ref["grad"] = new(B, h, w, 2), gr
            names = ("flow", "scalar", "vector") if delta else ("flow",)
            for k, name in enumerate(names):
                if n and (not delta or k):
                    got["prop_" + name], ref["prop_" + name] = torch.full_like(prop[k], -5.0), prop[k]
                if mids:
                    ref["mid_" + name] = torch.stack([q[1 + k] for q in passes[1:]])
                    got["mid_" + name] = torch.full_like(ref["mid_" + name], -5.0)
        a = _Level(image=image.data_ptr(), flow=flow.data_ptr(), bright=bright.data_ptr())
        if delta:
            a.dflow, a.upper = dflow.data_ptr(), upper.data_ptr()
            a.xmap, a.ymap = maps["xmap"].data_ptr(), maps["ymap"].data_ptr()
        for name, t in got.items():
            setattr(a, name, t.data_ptr())
        N.call("ff_ad_level_forward", ctypes.byref(a), n, K, B, h, w, hu, wu, f32(dt), border, f32(gamma),
               f32(maxflow), s)
        for name in got:
            assert same(ref[name], got[name]), (save, name)


def test_ad_level_refusals():
    """Sizes and iterations that no tile has room for, and outputs that are
    inputs, are errors, not launches."""
    import ctypes

    import torch
    from flowfilter import _native as N
    from flowfilter.autograd import _Level
    ok = lambda *a: N.get_int("ff_ad_level_supported", *a)
    assert ok(64, 64, 8, 2) and ok(64, 64, 0, 0) and ok(64, 64, 29, 1) and ok(64, 64, 2, 14)
    assert not ok(64, 64, 30, 1) and not ok(64, 64, 2, 15) and not ok(20000, 20000, 4, 1) and not ok(64, 64, -1, 1)
    assert not ok(64, 64, 1, 2 ** 30) and not ok(0, 64, 1, 1)
    t = torch.zeros(1, 8, 8, 2, device="cuda")
    a = _Level(*[t.data_ptr()] * 3)
    a.flow_out, a.bright_out = t.data_ptr(), t.data_ptr()
    call = lambda n: N.call("ff_ad_level_forward", ctypes.byref(a), n, 1, 1, 8, 8, 0, 0, ctypes.c_float(1), 1,
                            ctypes.c_float(1), ctypes.c_float(1), None)
    for n in (1, 30):
        with pytest.raises(Exception):
            call(n)


@pytest.mark.parametrize("B,T,h,w", [(1, 2, 1, 1), (2, 3, 3, 2), (1, 4, 5, 63), (2, 2, 16, 64), (1, 3, 17, 65), (1, 2, 90, 200)])
@pytest.mark.parametrize("kind", ["zero", "smooth", "rough"])
def test_photometric_adjoint(B, T, h, w, kind):
    """The photometric term's gradients against the float64 composition's (on
    the CPU): fields whose shares of a sampled pixel all meet, mostly meet, or
    rarely do. A frame pixel's gradient is a sum over the pixels that sample it,
    each share a float32 product within 4e-7 of itself times the terms'
    magnitude (coordinates of up to 200 px carry 1e-5 px of float32 rounding,
    and the differences up to 1): 2e-5 of the largest gradient of its kind, and
    for the flow 1e-3 more where a coordinate is that close to a pixel's edge,
    which only the random fields' 1 in 1e4 pixels are; none of the flows here
    samples a pixel's edge exactly but `zero`, whose coordinates are integers
    (left out for the flow: the derivative there is one-sided)."""
    import torch
    from flowfilter.autograd import photometric_error
    print("photometric adjoint", (B, T, h, w), kind, flush=True)
    g = torch.Generator().manual_seed(h * 100 + w)
    frames = torch.rand(B, T, h, w, generator=g)
    y, x = torch.meshgrid(torch.arange(h), torch.arange(w), indexing="ij")
    if kind == "zero":
        flows = torch.zeros(B, T, h, w, 2)
    elif kind == "smooth":
        flows = torch.stack([0.3 + 0.5 * torch.sin(x / 40.0), -0.4 + 0.5 * torch.cos(y / 30.0)], -1).expand(
            B, T, h, w, 2).contiguous()
    else:
        flows = torch.randn(B, T, h, w, 2, generator=g) * 3.0
    out = []
    for dev, dt in (("cpu", torch.float64), ("cuda", torch.float32)):
        fr = frames.to(dev, dt).requires_grad_()
        fl = flows.to(dev, dt).requires_grad_()
        photometric_error(fr, fl).backward()
        out.append((fr.grad.cpu().double(), fl.grad.cpu().double()))
    (a, b), (c, d) = out
    assert float((a - c).abs().max()) <= 2e-5 * max(float(a.abs().max()), 1.0 / (B * T * h * w))
    if kind != "zero":
        near = (flows.double() - flows.double().round()).abs().amin(-1, keepdim=True) < 1e-4
        bad = ((b - d).abs() > 1e-3 * float(b.abs().max()) + 1e-12) & ~near
        assert not bool(bad.any())


@pytest.mark.parametrize("B,h,w", [(1, 2, 2), (2, 3, 5), (1, 9, 130), (3, 16, 63), (2, 67, 129)])
@pytest.mark.parametrize("inplace", [False, True])
def test_float_pyramid_step(ffo, B, h, w, inplace):
    """The reduction is bitwise the oracle's, and its adjoint, added to what is
    there, its transpose: <g, D x> = <D^T g, x> in float64 sums to 1e-6 of the
    terms' magnitude (weights that are powers of two; a rounding per sum). Also
    with the result in the input's place, and the adjoint's in its input's."""
    import ctypes

    import torch
    from flowfilter import _native as N
    print("pyramid step", (B, h, w), inplace, flush=True)
    g = torch.Generator(device="cuda").manual_seed(h * w)
    rnd = lambda *s: torch.rand(*s, generator=g, device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    img, work = rnd(B, h, w), torch.empty(B, h, w // 2, device="cuda")
    hh, hw = h // 2, w // 2
    n = B * hh * hw
    buf = img.clone()
    half = buf.view(-1)[:n] if inplace else torch.empty(n, device="cuda")
    N.call("ff_ad_down", p(buf), p(half), p(work), B, h, w, s)
    half = half.view(B, hh, hw).clone()
    for b in range(B):
        assert np.array_equal(half[b].cpu().numpy(), ffo.pyramid(img[b].cpu().numpy(), 2)[1])
    gh, base = rnd(B, hh, hw) - 0.5, rnd(B, h, w)
    out = base.clone()
    src = gh.contiguous()
    if inplace:
        out.view(-1)[:n] = gh.view(-1)
        base = out.clone()
        src = out.view(-1)[:n]
    N.call("ff_ad_down_backward", p(src), p(out), p(work), B, h, w, 1, s)
    left = (gh.double() * half.double()).sum()
    right = ((out.double() - base.double()) * img.double()).sum()
    assert abs(float(left - right)) <= 1e-6 * float((gh.abs().double() * half.double()).sum() + base.sum().double())
