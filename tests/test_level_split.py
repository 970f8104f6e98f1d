"""Which iterations of a level of the differentiable window run in the launch of
its image model and update: the rule on the CPU, and on the GPU that the split
changes no bit."""
import pytest

SIZES = [(1, 1, 1), (1, 64, 64), (1, 64, 65), (16, 64, 64), (2, 165, 123), (1, 400, 600), (1, 600, 800),
         (16, 512, 512), (1, 2160, 3840), (4, 4320, 7680)]


@pytest.mark.parametrize("save", [False, True])
def test_halo_is_bounded(save):
    """However many iterations a level has, those in its launch leave a tile of
    at least a quarter of the buffer, unless all its workgroups run at once; and
    they are iterations that the launch takes."""
    from flowfilter import _native as N
    from flowfilter.autograd import _in_launch
    for B, h, w in SIZES:
        for n in (0, 1, 2, 4, 6, 7, 8, 9, 16, 20, 28, 64):
            for K in (0, 1, 2, 3, 4, 5, 8, 10, 12, 14, 40):
                a, b = _in_launch(B, h, w, n, K, save)
                assert 0 <= a <= n and 0 <= b <= K
                inner = 64 - 2 * (max(a, 2) + 2 * b)
                tiles = B * (-(-w // max(inner, 1)) if w > 64 else 1) * (-(-h // max(inner, 1)) if h > 64 else 1)
                assert inner >= 32 or tiles <= 512, (B, h, w, n, K, a, b)
                assert N.get_int("ff_ad_level_supported", h, w, a, b), (B, h, w, n, K, a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("B,h,w,levels", [(1, 60, 64, 1), (2, 130, 200, 2), (1, 700, 900, 2)])
@pytest.mark.parametrize("maxflow,smooth", [(4.0, 5), (9.0, 2), (20.0, 1), (2.0, 12)])
def test_split_levels_match_the_stages(monkeypatch, B, h, w, levels, maxflow, smooth):
    """Flows and gradients of a window are bitwise those of the stages' own
    launches."""
    import torch
    from flowfilter.autograd import FilterSpec, flow_window
    print("split", (B, h, w), levels, maxflow, smooth, flush=True)
    g = torch.Generator(device="cuda").manual_seed(h + smooth)
    frames = torch.rand(B, 3, h, w, generator=g, device="cuda")
    weights = torch.randn(B, 3, h, w, 2, generator=g, device="cuda")
    spec = FilterSpec(h, w, levels, maxflow=maxflow, smooth=smooth)

    def run():
        f = frames.clone().requires_grad_()
        gamma = torch.tensor([10.0, 50.0][:levels], device="cuda", requires_grad=True)
        out = flow_window(f, gamma, spec)
        (out * weights).sum().backward()
        return out.detach(), f.grad, gamma.grad

    assert spec.tiled
    got = run()
    monkeypatch.setattr(FilterSpec, "tiled", False)
    want = run()
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.gpu
def test_window_allocates_no_unused_work_buffers(monkeypatch):
    """The image model's adjoint and the pyramid's reduction use a work buffer
    only where a result overlaps an input, which a window never asks for: none is
    allocated for them (the pyramid's adjoint does use its own)."""
    import torch
    from flowfilter import autograd as A
    shapes, inner = [], A._empty
    monkeypatch.setattr(A, "_empty", lambda *a, **k: shapes.append(a) or inner(*a, **k))
    B, T, h, w = 2, 3, 64, 80
    frames = torch.rand(B, T, h, w, device="cuda", requires_grad=True)
    out = A.flow_window(frames, torch.tensor([10.0, 50.0], device="cuda"), A.FilterSpec(h, w, 2, maxflow=2.0))
    forward, shapes[:] = list(shapes), []
    assert (B, h, w // 2) not in forward and (B, h // 2, w // 2) in forward
    out.sum().backward()
    assert shapes.count((B, h, w // 2)) == T  # the pyramid's adjoint
    assert (B, 2 * h, w) not in shapes and (B, h, w) in shapes
