"""The work that programs give this library, as cases that can be timed and
compared.

A case is a dict of plain values; its "kind" names the path:

* ``frame``: one camera stream. A PyramidalFlowFilter is fed one frame per
  pass and its flow is read; the frame is a device buffer read in place
  (``io`` "place"), a device buffer copied in ("copy"), or a numpy array with
  the flow downloaded to numpy ("host", the loop of the reference's notebook).
  ``tight`` rows have a pitch of exactly the width, as torch tensors have;
  others are padded to 256 bytes.
* ``batch``: many camera streams advanced together by a BatchedFlowFilter.
* ``stages``: a filter level put together by hand from the stage classes on a
  float image: image model, propagation, update and smoothing, with the plain
  update, or with payloads and the delta update of a lower pyramid level.
* ``rotation``: image prediction from a camera's rotation.
* ``window``: the differentiable filter over a window of frames, forward only
  or forward and backward with its training loss.

``prepare`` makes the inputs from the seed (band-limited texture under a
smooth motion within the filter's maxflow, in u8 levels) and the filter with a
few frames behind it, as a running program has it; ``run`` is one pass.
"""
import math
import os
import random
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "optical-flow-filter_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

WARM_FRAMES = 3   # frames a prepared filter has seen
CYCLE = 6         # frames of a stream's cycle: 4 frames, back and forth


# ------------------------------------------------------------------- cases

def listed():
    return [
        # the smallest camera stream of a batch, alone: launches and latency
        dict(name="frame_320x240_1", kind="frame", h=240, w=320, levels=1, gamma="20", maxflow=4.0, smooth="1",
             io="place", tight=False),
        # the reference notebook's loop: numpy frames in, numpy flow out
        dict(name="frame_640x480_2_host", kind="frame", h=480, w=640, levels=2, gamma="10,50", maxflow=4.0,
             smooth="2,4", io="host", tight=True),
        # the benchmark's workload
        dict(name="frame_2048x1088_2", kind="frame", h=1088, w=2048, levels=2, gamma="10,50", maxflow=4.0,
             smooth="2,2", io="place", tight=False),
        # odd sizes at every level, frames of a torch program (tight rows)
        dict(name="frame_1917x1079_3", kind="frame", h=1079, w=1917, levels=3, gamma="10,20,40", maxflow=4.0,
             smooth="1,2,2", io="place", tight=True),
        # the largest single stream: fast motion, a deep pyramid
        dict(name="frame_3840x2160_4", kind="frame", h=2160, w=3840, levels=4, gamma="10,20,30,50", maxflow=8.0,
             smooth="2,2,2,2", io="copy", tight=False),
        # a multi-camera server
        dict(name="batch_64", kind="batch", streams=64, layout=3, maxflow=4.0, scale=1.0),
        # a level wired by hand from the stage classes, on a float image
        dict(name="stages_1280x720", kind="stages", h=720, w=1280, payload=False, iterations=4, gamma=20.0,
             maxflow=4.0, smooth=2),
        # image prediction of a rotating camera
        dict(name="rotation_2048x1088", kind="rotation", h=1088, w=2048, iterations=4),
        # fine-tuning on small crops: many short launches
        dict(name="window_2x4x165x123_3", kind="window", h=123, w=165, batch=2, frames=4, levels=3, gamma="10,20,40",
             maxflow=4.0, smooth="2,1,1", checkpoint=2, grad=True),
        # training on crops
        dict(name="window_16x8x512x512_2", kind="window", h=512, w=512, batch=16, frames=8, levels=2, gamma="10,50",
             maxflow=4.0, smooth="2,2", checkpoint=4, grad=True),
        # training on whole 4K frames
        dict(name="window_1x8x3840x2160_3", kind="window", h=2160, w=3840, batch=1, frames=8, levels=3,
             gamma="10,20,50", maxflow=8.0, smooth="2,2,2", checkpoint=4, grad=True),
        # evaluation of a trained filter: no gradients
        dict(name="window_1x8x1920x1080_eval", kind="window", h=1080, w=1920, batch=1, frames=8, levels=2,
             gamma="10,50", maxflow=6.0, smooth="2,2", checkpoint=4, grad=False),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, most):
    """A frame size of camera shape between lo and hi rows, at most `most`
    pixels; half of them not a multiple of anything."""
    h = _log_uniform(rng, lo, hi)
    w = int(h * rng.choice([1.0, 4.0 / 3.0, 16.0 / 9.0, 2.0]))
    if rng.random() < 0.5:
        h, w = max(8 * (h // 8), lo), max(8 * (w // 8), lo)
    else:
        w += rng.randrange(8)
    while h * w > most:
        h, w = h * 7 // 8, w * 7 // 8
    return h, w


def _per_level(rng, levels, lo, hi, whole):
    pick = (lambda: rng.randint(lo, hi)) if whole else (lambda: round(rng.uniform(lo, hi), 1))
    return ",".join(str(pick()) for _ in range(levels))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "batch", "stages", "rotation", "window", "window"])
    if kind == "frame":
        h, w = _size(rng, 120, 2160, 3840 * 2160)
        levels = rng.randint(1, 4 if h >= 480 else 3)
        return dict(kind=kind, h=h, w=w, levels=levels, gamma=_per_level(rng, levels, 5.0, 50.0, False),
                    maxflow=rng.choice([1.0, 2.0, 3.0, 4.0, 4.0, 6.5, 8.0]),
                    smooth=_per_level(rng, levels, 1, 3, True), io=rng.choice(["place", "place", "copy", "host"]),
                    tight=rng.random() < 0.5)
    if kind == "batch":
        return dict(kind=kind, streams=_log_uniform(rng, 2, 48), layout=rng.randrange(1 << 20),
                    maxflow=rng.choice([2.0, 4.0]), scale=round(rng.uniform(0.6, 1.0), 3))
    if kind == "stages":
        h, w = _size(rng, 120, 2160, 3840 * 2160)
        return dict(kind=kind, h=h, w=w, payload=rng.random() < 0.5, iterations=rng.randint(1, 8),
                    gamma=round(rng.uniform(5.0, 50.0), 1), maxflow=rng.choice([2.0, 4.0, 8.0]),
                    smooth=rng.randint(1, 4))
    if kind == "rotation":
        h, w = _size(rng, 120, 2160, 3840 * 2160)
        return dict(kind=kind, h=h, w=w, iterations=rng.randint(1, 8))
    batch, frames = _log_uniform(rng, 1, 16), rng.randint(3, 8)
    h, w = _size(rng, 96, 1080, min(1920 * 1080, 40_000_000 // (batch * frames)))
    levels = rng.randint(1, 3)
    return dict(kind=kind, h=h, w=w, batch=batch, frames=frames, levels=levels,
                gamma=_per_level(rng, levels, 5.0, 50.0, False), maxflow=rng.choice([2.0, 3.0, 4.0, 8.0]),
                smooth=_per_level(rng, levels, 1, 2, True), checkpoint=rng.choice([1, 2, 4]),
                grad=rng.random() < 0.75)


def _floats(text):
    return [float(v) for v in text.split(",")]


def _ints(text):
    return [int(v) for v in text.split(",")]


# Resolutions of a batch's camera streams (320x240 to 1920x1080).
_STREAMS = ((240, 320), (480, 640), (720, 1280), (1080, 1920))


def _layout(case):
    """The streams of a batch: size, levels, gains and smoothing of each."""
    rng = random.Random("batch %d" % case["layout"])
    out = []
    for _ in range(case["streams"]):
        h, w = rng.choice(_STREAMS)
        h, w = int(h * case["scale"]), int(w * case["scale"])
        levels = rng.randint(1, 3)
        out.append(dict(h=h, w=w, levels=levels, gamma=[round(rng.uniform(5.0, 50.0), 1) for _ in range(levels)],
                        maxflow=case["maxflow"], smooth=[rng.randint(1, 2) for _ in range(levels)]))
    return out


# ------------------------------------------------------------------ inputs

def _gen(seed, device):
    return torch.Generator(device=device).manual_seed(int(seed) & 0x7fffffffffff)


def _lowpass(x, sigma):
    ky = torch.fft.fftfreq(x.shape[-2], device=x.device)[:, None]
    kx = torch.fft.rfftfreq(x.shape[-1], device=x.device)[None, :]
    g = torch.exp(-2.0 * (math.pi * sigma) ** 2 * (kx * kx + ky * ky))
    return torch.fft.irfft2(torch.fft.rfft2(x) * g, s=x.shape[-2:])


def _sequence(h, w, count, reach, seed, device="cuda"):
    """`count` frames [count, h, w] of u8 levels: low-passed noise carried by
    a translation plus a rotation about the centre, at most `reach` pixels a
    frame; and that motion [h, w, 2]."""
    g = _gen(seed, device)
    pad = int(math.ceil(reach * count)) + 4
    th, tw = -(-(h + 2 * pad) // 32) * 32, -(-(w + 2 * pad) // 32) * 32
    tex = _lowpass(torch.randn(th, tw, generator=g, device=device), 2.5)
    tex = 128.0 + 52.0 * tex / tex.std()
    p = torch.rand(3, generator=g, device=device) * 2.0 - 1.0
    ys = torch.arange(h, device=device, dtype=torch.float32)[:, None]
    xs = torch.arange(w, device=device, dtype=torch.float32)[None, :]
    spin = 0.5 * reach * p[2] / (0.5 * math.hypot(h, w))
    v = torch.stack([0.5 * reach * p[0] / math.sqrt(2) - spin * (ys - 0.5 * h) + 0.0 * xs,
                     0.5 * reach * p[1] / math.sqrt(2) + spin * (xs - 0.5 * w) + 0.0 * ys], -1)
    frames = []
    for t in range(count):
        gx = 2.0 * (xs + pad - t * v[..., 0]) / (tw - 1) - 1.0
        gy = 2.0 * (ys + pad - t * v[..., 1]) / (th - 1) - 1.0
        f = torch.nn.functional.grid_sample(tex[None, None], torch.stack([gx, gy], -1)[None], mode="bilinear",
                                            padding_mode="border", align_corners=True)[0, 0]
        f = f + 1.5 * torch.randn(h, w, generator=g, device=device)
        frames.append(f.round().clamp(0, 255).to(torch.uint8))
    return torch.stack(frames), v


def _turn(i):
    """Frame of step i when a stream's frames run back and forth."""
    k = i % CYCLE
    return k if k <= CYCLE // 2 else CYCLE - k


def _stream_frames(h, w, maxflow, seed):
    return _sequence(h, w, CYCLE // 2 + 1, 0.6 * maxflow, seed)[0]


# ---------------------------------------------------------------- programs

def _filter(gf, spec):
    f = gf.PyramidalFlowFilter(spec["h"], spec["w"], spec["levels"])
    one = spec["levels"] == 1
    f.gamma = spec["gamma"][0] if one else spec["gamma"]
    f.maxflow = spec["maxflow"]
    f.smoothIterations = spec["smooth"][0] if one else spec["smooth"]
    return f


def _frame_spec(case):
    return dict(h=case["h"], w=case["w"], levels=case["levels"], gamma=_floats(case["gamma"]),
                maxflow=case["maxflow"], smooth=_ints(case["smooth"]))


def _pitched(frames, tight):
    """Frames as device buffers: [count, h, pitch] u8 and the row pitch."""
    w = frames.shape[2]
    pitch = w if tight else -(-w // 256) * 256
    buf = torch.zeros(frames.shape[0], frames.shape[1], pitch, dtype=torch.uint8, device=frames.device)
    buf[:, :, :w] = frames
    return buf, pitch


def prepare(case, seed):
    import flowfilter.gpu.flowfilters as gf
    kind = case["kind"]
    state = dict(kind=kind, step=0)
    if kind == "frame":
        spec = _frame_spec(case)
        frames = _stream_frames(case["h"], case["w"], case["maxflow"], seed)
        f = _filter(gf, spec)
        state.update(io=case["io"], filter=f, flow=f.getFlowDevice())
        if case["io"] == "host":
            state["frames"] = [x for x in frames.cpu().numpy()]
        else:
            buf, pitch = _pitched(frames, case["tight"])
            state.update(buffer=buf, pitch=pitch, at=[buf[i].data_ptr() for i in range(len(buf))])
    elif kind == "batch":
        specs = _layout(case)
        bufs = [_pitched(_stream_frames(s["h"], s["w"], s["maxflow"], seed * 1009 + k), False)
                for k, s in enumerate(specs)]
        batch = gf.BatchedFlowFilter([_filter(gf, s) for s in specs])
        state.update(batch=batch, views=[], buffers=bufs,
                     pitches=[p for _, p in bufs],
                     at=[[b[_turn(i)].data_ptr() for b, _ in bufs] for i in range(CYCLE)])
    elif kind == "stages":
        _prepare_stages(case, seed, state)
    elif kind == "rotation":
        _prepare_rotation(case, seed, state)
    elif kind == "window":
        _prepare_window(case, seed, state)
    torch.cuda.synchronize()
    if kind in ("frame", "batch", "stages"):
        for _ in range(WARM_FRAMES):
            run(state)
    if kind == "batch":
        # a filter's flow alternates between two buffers, so a program with
        # many streams takes both views of each once
        for _ in range(2):
            run(state)
            state["views"].append([torch.from_dlpack(f.getFlowDevice()) for f in state["batch"]])
    torch.cuda.synchronize()
    return state


def _prepare_stages(case, seed, state):
    from flowfilter.gpu.flowsmoothing import FlowSmoother
    from flowfilter.gpu.image import GPUImage
    from flowfilter.gpu.imagemodel import ImageModel
    from flowfilter.gpu.propagation import FlowPropagator, FlowPropagatorPayload
    from flowfilter.gpu.update import DeltaFlowUpdate, FlowUpdate
    h, w, n = case["h"], case["w"], case["iterations"]
    frames = _stage_frames(case, seed)
    image = GPUImage((h, w), 4)
    model = ImageModel(image)
    flow, old = GPUImage((h, w, 2), 4), GPUImage((h, w), 4)
    gamma = case["gamma"] / 255.0 ** 2
    # wired in a circle, as the filters are: the propagation reads the
    # smoothed flow of the frame before, the update the propagated flow
    flow = GPUImage((h, w, 2), 4)
    flow.clear()
    if case["payload"]:
        upper, old = GPUImage((h // 2, w // 2, 2), 4), GPUImage((h, w), 4)
        upper.upload(_stage_upper(case, seed).cpu().numpy())
        update = DeltaFlowUpdate(upper, flow, old, model.getImageConstant(), model.getImageGradient(), gamma,
                                 case["maxflow"])
        smoother = FlowSmoother(update.getUpdatedFlow(), case["smooth"])
        prop = FlowPropagatorPayload(smoother.getSmoothedFlow(), update.getUpdatedImage(),
                                     update.getUpdatedDeltaFlow(), n)
        update.setInputDeltaFlow(prop.getPropagatedVector())
        update.setInputImageOld(prop.getPropagatedScalar())
        update.getUpdatedDeltaFlow().clear()
        state["upper"] = upper
    else:
        update = FlowUpdate(flow, model.getImageConstant(), model.getImageGradient(), gamma, case["maxflow"])
        smoother = FlowSmoother(update.getUpdatedFlow(), case["smooth"])
        prop = FlowPropagator(smoother.getSmoothedFlow(), n)
        update.setInputFlow(prop.getPropagatedFlow())
    update.getUpdatedImage().clear()
    smoother.getSmoothedFlow().clear()
    state.update(image=image, frames=frames, at=[frames[i].data_ptr() for i in range(len(frames))], pitch=w * 4,
                 stages=[model, prop, update, smoother], flow=smoother.getSmoothedFlow())


def _stage_frames(case, seed):
    frames, _ = _sequence(case["h"], case["w"], CYCLE // 2 + 1, 0.6 * case["maxflow"], seed)
    return (frames.to(torch.float32) / 255.0).contiguous()


def _stage_upper(case, seed):
    """A coarser level's flow: smooth, half the level's motion."""
    h, w = case["h"] // 2, case["w"] // 2
    u = _lowpass(torch.randn(2, h, w, generator=_gen(seed + 1, "cuda"), device="cuda"), 12.0)
    return (0.15 * case["maxflow"] * u / u.std()).permute(1, 2, 0).contiguous()


def _rotation_inputs(case, seed):
    frames, _ = _sequence(case["h"], case["w"], 1, 1.0, seed)
    p = torch.rand(3, generator=_gen(seed + 2, "cpu")) * 2.0 - 1.0
    scale = 2.0 / (case["w"] * 4.0 / 4.8)  # about two pixels
    return (frames[0].to(torch.float32) / 255.0).contiguous(), [float(v) * scale for v in p]


_LENS = (4.0, 3.6, 4.8)  # focal length, sensor height and width in mm


def _prepare_rotation(case, seed, state):
    from flowfilter.gpu.camera import createPerspectiveCamera
    from flowfilter.gpu.image import GPUImage
    from flowfilter.gpu.rotation import RotationalFlowImagePredictor
    h, w = case["h"], case["w"]
    frame, spin = _rotation_inputs(case, seed)
    image = GPUImage((h, w), 4)
    image.upload(frame.cpu().numpy())
    predictor = RotationalFlowImagePredictor(createPerspectiveCamera(_LENS[0], h, w, _LENS[1], _LENS[2]), image)
    predictor.iterations = case["iterations"]
    state.update(image=image, predictor=predictor, spin=spin, predicted=predictor.getPredictedImage(),
                 field=predictor.getOpticalFlow())


def _window_inputs(case, seed):
    both = [_sequence(case["h"], case["w"], case["frames"], 0.5 * case["maxflow"], seed * 131 + b)
            for b in range(case["batch"])]
    frames = torch.stack([f for f, _ in both]).to(torch.float32) / 255.0
    return frames.contiguous(), torch.stack([v for _, v in both]).contiguous()


def _prepare_window(case, seed, state):
    import flowfilter.autograd as ag
    frames, truth = _window_inputs(case, seed)
    spec = ag.FilterSpec(case["h"], case["w"], case["levels"], maxflow=case["maxflow"], smooth=_ints(case["smooth"]))
    gamma = torch.tensor(_floats(case["gamma"]), device="cuda")
    state.update(ag=ag, frames=frames, truth=truth, spec=spec, gamma=gamma, checkpoint=case["checkpoint"],
                 grad=case["grad"])


def run(state):
    kind = state["kind"]
    if kind == "frame":
        f, i = state["filter"], _turn(state["step"])
        state["step"] += 1
        if state["io"] == "host":
            f.loadImage(state["frames"][i])
            f.compute()
            return f.getFlow()
        if state["io"] == "place":
            f.setImageDevice(state["at"][i], state["pitch"])
        else:
            f.loadImageDevice(state["at"][i], state["pitch"])
        f.compute()
        return torch.from_dlpack(state["flow"])
    if kind == "batch":
        batch = state["batch"]
        batch.setImagesDevice(state["at"][state["step"] % CYCLE], state["pitches"])
        state["step"] += 1
        batch.compute()
        views = state["views"]
        return views[(state["step"] - WARM_FRAMES - 1) % 2] if len(views) == 2 else None
    if kind == "stages":
        i = _turn(state["step"])
        state["step"] += 1
        state["image"].uploadDevice(state["at"][i], state["pitch"])
        for stage in state["stages"]:
            stage.compute()
        return torch.from_dlpack(state["flow"])
    if kind == "rotation":
        predictor = state["predictor"]
        predictor.setAngularVelocity(*state["spin"])
        predictor.compute()
        return [torch.from_dlpack(state["predicted"]), torch.from_dlpack(state["field"])]
    ag = state["ag"]
    if not state["grad"]:
        with torch.no_grad():
            return ag.flow_window(state["frames"], state["gamma"], state["spec"], state["checkpoint"])
    frames = state["frames"].detach().requires_grad_(True)
    gamma = state["gamma"].detach().requires_grad_(True)
    flows = ag.flow_window(frames, gamma, state["spec"], state["checkpoint"])
    loss = ag.flow_loss(frames, flows, state["truth"])
    g_frames, g_gamma = torch.autograd.grad(loss, (frames, gamma))
    return dict(loss=loss.detach(), flows=flows.detach(), g_frames=g_frames, g_gamma=g_gamma)


# -------------------------------------------------------------------- work

def _level_iterations(levels, maxflow):
    """Propagation iterations of each level: ceil of its maxflow, halved from
    level to level."""
    out, m = [], np.float32(maxflow)
    for l in range(levels):
        out.append(max(1, int(math.ceil(float(m)))))
        if l < levels - 1:
            m = np.float32(m / np.float32(2.0))
    return out


# Operations per pixel: an upwind pass of one field (a difference, a product
# and a sum) and its speed; the image model's five 5-tap sums; the solve; one
# smoothing iteration of a vector.
_OPS_FIELD, _OPS_SPEED, _OPS_MODEL, _OPS_SOLVE, _OPS_SMOOTH = 3, 3, 50, 32, 40


def _filter_work(spec):
    """Bytes: each level's state (flow, brightness, on delta levels the delta
    flow) read and written once, the frame read once, the level above read
    once."""
    nbytes = flops = 0
    h, w = spec["h"], spec["w"]
    its = _level_iterations(spec["levels"], spec["maxflow"])
    nbytes += h * w
    for l in range(spec["levels"]):
        n, top = h * w, l == spec["levels"] - 1
        nbytes += n * (24 if top else 40)
        if not top:
            nbytes += (h // 2) * (w // 2) * 8 * (2 if l == spec["levels"] - 2 else 1)
        fields = 2 if top else 5
        flops += n * (2 * its[l] * (_OPS_FIELD * fields + _OPS_SPEED) + _OPS_MODEL + _OPS_SOLVE +
                      _OPS_SMOOTH * spec["smooth"][l])
        h, w = h // 2, w // 2
    return nbytes, flops


def work(case):
    kind = case["kind"]
    if kind == "frame":
        b, f = _filter_work(_frame_spec(case))
        if case["io"] == "host":
            b += 8 * case["h"] * case["w"]  # the flow goes to the host too
        return dict(bytes=b, flops=f)
    if kind == "batch":
        both = [_filter_work(s) for s in _layout(case)]
        return dict(bytes=sum(b for b, _ in both), flops=sum(f for _, f in both))
    if kind == "stages":
        n, fields = case["h"] * case["w"], 5 if case["payload"] else 2
        return dict(bytes=n * (4 + (40 if case["payload"] else 24) + (2 if case["payload"] else 0)),
                    flops=n * (2 * case["iterations"] * (_OPS_FIELD * fields + _OPS_SPEED) + _OPS_MODEL + _OPS_SOLVE +
                               _OPS_SMOOTH * case["smooth"]))
    if kind == "rotation":
        n = case["h"] * case["w"]
        return dict(bytes=n * 16, flops=n * (16 + 2 * 9 * case["iterations"]))
    n = case["batch"] * case["frames"] * case["h"] * case["w"]
    spec = dict(h=case["h"], w=case["w"], levels=case["levels"], maxflow=case["maxflow"], smooth=_ints(case["smooth"]))
    f = _filter_work(spec)[1] * case["batch"] * case["frames"]
    return dict(bytes=n * (16 if case["grad"] else 12), flops=f * (3 if case["grad"] else 1))


# ------------------------------------------- the same values in 64 bits

def _shift(t, dim, k):
    n = t.shape[dim]
    return t.index_select(dim, (torch.arange(n, device=t.device) + k).clamp(0, n - 1))


def _taps(t, dim, weights):
    return sum(c * _shift(t, dim, k - 2) for k, c in enumerate(weights) if c)


_BINOMIAL = (0.0625, 0.25, 0.375, 0.25, 0.0625)
_DERIVATIVE = (-0.125, -0.25, 0.0, 0.25, 0.125)


def _model64(img):
    sy, sx = _taps(img, -2, _BINOMIAL), _taps(img, -1, _BINOMIAL)
    return _taps(sy, -1, _BINOMIAL), (_taps(sy, -1, _DERIVATIVE), _taps(sx, -2, _DERIVATIVE))


def _advect64(fields, n, border=3):
    """n upwind iterations (along x, then y) of fields [u, v, payloads...]."""
    h, w = fields[0].shape[-2:]
    inside = torch.zeros(h, w, dtype=torch.bool, device=fields[0].device)
    inside[border:max(h - border, border), border:max(w - border, border)] = True
    for _ in range(n):
        for axis, dim in ((0, -1), (1, -2)):
            a, b = _shift(fields[axis], dim, -1), _shift(fields[axis], dim, 1)
            speed = torch.where(b.abs() > a.abs(), b, a) / n
            back = speed >= 0
            fields = [torch.where(inside, t - speed * torch.where(back, t - _shift(t, dim, -1), _shift(t, dim, 1) - t),
                                  t) for t in fields]
    return fields


def _solve64(g, dY, f, gamma):
    c = (dY - g[0] * f[0] - g[1] * f[1]) / (gamma + g[0] * g[0] + g[1] * g[1])
    return f[0] + c * g[0], f[1] + c * g[1]


def _smooth64(f, k):
    for _ in range(k):
        f = [_taps(_taps(t, -1, (0.2,) * 5), -2, (0.2,) * 5) for t in f]
    return f


def _map(n, nu, device):
    """Which pixel of a level of nu pixels pixel x of n reads."""
    if n <= 1:
        return torch.zeros(n, dtype=torch.long, device=device)
    x = np.arange(n, dtype=np.float32) / np.float32(n - 1)
    return torch.from_numpy(np.clip(np.floor(x * np.float32(nu)).astype(np.int64), 0, nu - 1)).to(device)


def _upper64(f, h, w):
    ym, xm = _map(h, f[0].shape[-2], f[0].device), _map(w, f[0].shape[-1], f[0].device)
    return [t.index_select(-2, ym).index_select(-1, xm) for t in f]


def _halve(img, dim, whole):
    i = 2 * torch.arange(img.shape[dim] // 2, device=img.device)
    n = img.shape[dim]
    m, z, p = (img.index_select(dim, (i + k).clamp(0, n - 1)) for k in (-1, 0, 1))
    return (2 * z + m + p) // 4 if whole else 0.5 * z + 0.25 * (m + p)


def _frame64(spec, state, pyramid, gamma):
    """One frame of the filter. state: per level (flow, brightness, delta
    flow), or None before the first frame; gamma in the update's units."""
    top = spec["levels"] - 1
    its = _level_iterations(spec["levels"], spec["maxflow"])
    models = [_model64(p) for p in pyramid]
    if state is None:
        z = [torch.zeros_like(m[0]) for m in models]
        state = [([z[l], z[l]], models[l][0], [z[l], z[l]]) for l in range(top + 1)]
    new = [None] * (top + 1)
    a0, g = models[top]
    f = _advect64(state[top][0], its[top])
    m = spec["maxflow"] / 2.0 ** top
    raw = [t.clamp(-m, m) for t in _solve64(g, state[top][1] - a0, f, gamma[top])]
    new[top] = (_smooth64(raw, spec["smooth"][top]), a0, None, raw)
    for l in range(top):
        a0, g = models[l]
        p = _advect64(list(state[l][0]) + [state[l][1]] + list(state[l][2]), its[l])
        ml = spec["maxflow"] / 2.0 ** l
        d = [t.clamp(-0.5 * ml, 0.5 * ml) for t in _solve64(g, p[2] - a0, p[3:], gamma[l])]
        up = _upper64(raw if l == top - 1 else state[l + 1][0], *a0.shape[-2:])
        flow = [(x + 2.0 * y).clamp(-ml, ml) for x, y in zip(d, up)]
        new[l] = (_smooth64(flow, spec["smooth"][l]), a0, d)
    return new


def _stream64(spec, frames, host=False, count=WARM_FRAMES + 1):
    """Flow after `count` frames. The device flow of a
    single level is the update's, before the smoothing; the downloaded one
    is the smoothed."""
    state = None
    gamma = [v / 255.0 ** 2 for v in spec["gamma"]]
    for i in range(count):
        levels = [frames[_turn(i)].to(torch.int64)]
        for _ in range(spec["levels"] - 1):
            levels.append(_halve(_halve(levels[-1], -1, True), -2, True))
        state = _frame64(spec, state, [x.double() / 255.0 for x in levels], gamma)
    return torch.stack(state[0][3 if spec["levels"] == 1 and not host else 0], -1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "frame":
        host = case["io"] == "host"
        out = _stream64(_frame_spec(case), _stream_frames(case["h"], case["w"], case["maxflow"], seed), host)
        return out.cpu().numpy() if host else out
    if kind == "batch":
        return [_stream64(s, _stream_frames(s["h"], s["w"], s["maxflow"], seed * 1009 + k), count=WARM_FRAMES + 3)
                for k, s in enumerate(_layout(case))]
    if kind == "stages":
        return _stages64(case, seed)
    if kind == "rotation":
        return _rotation64(case, seed)
    return _window64(case, seed)


def _stages64(case, seed):
    frames = _stage_frames(case, seed).double()
    gamma, m = case["gamma"] / 255.0 ** 2, case["maxflow"]
    zero = torch.zeros_like(frames[0])
    flow, old, delta = [zero, zero], zero, [zero, zero]
    if case["payload"]:
        up = _upper64([t.double() for t in _stage_upper(case, seed).unbind(-1)], case["h"], case["w"])
    for i in range(WARM_FRAMES + 1):
        a0, g = _model64(frames[_turn(i)])
        if case["payload"]:
            p = _advect64(list(flow) + [old] + list(delta), case["iterations"])
            delta = [t.clamp(-0.5 * m, 0.5 * m) for t in _solve64(g, p[2] - a0, p[3:], gamma)]
            flow = [(x + 2.0 * y).clamp(-m, m) for x, y in zip(delta, up)]
        else:
            f = _advect64(flow, case["iterations"])
            flow = [t.clamp(-m, m) for t in _solve64(g, old - a0, f, gamma)]
        old = a0
        flow = _smooth64(flow, case["smooth"])
    return torch.stack(flow, -1)


def _rotation64(case, seed):
    h, w, n = case["h"], case["w"], case["iterations"]
    frame, (wx, wy, wz) = _rotation_inputs(case, seed)
    ax, ay = _LENS[0] * (w - 1) / _LENS[2], _LENS[0] * (h - 1) / _LENS[1]
    x = torch.arange(w, device="cuda", dtype=torch.float64)[None, :] - 0.5 * (w - 1)
    y = torch.arange(h, device="cuda", dtype=torch.float64)[:, None] - 0.5 * (h - 1)
    px, py = x / ax, y / ay
    cz = wx * py - wy * px
    u, v = ax * (wy - wz * py) - x * cz, ay * (wz * px - wx) - y * cz
    img = frame.double()
    for _ in range(n):
        for dim, s in ((-2, v), (-1, u)):
            a, b, r = _shift(img, dim, -1), _shift(img, dim, 1), s / n
            img = img - 0.5 * r * (b - a) + 0.5 * r * r * (a - 2.0 * img + b)
    return [img, torch.stack([u, v], -1)]


def _window64(case, seed):
    its = _level_iterations(case["levels"], case["maxflow"])
    pixels = case["batch"] * case["frames"] * case["h"] * case["w"]
    if pixels * (60 * its[0] + 90) * 8 > 90e9:
        return None  # autograd's saved tensors in 64 bits would not fit
    frames, truth = _window_inputs(case, seed)
    spec = dict(levels=case["levels"], maxflow=case["maxflow"], smooth=_ints(case["smooth"]))
    frames = frames.double().requires_grad_(case["grad"])
    gamma = torch.tensor(_floats(case["gamma"]), device="cuda", dtype=torch.float64, requires_grad=case["grad"])
    with torch.set_grad_enabled(case["grad"]):
        state, out = None, []
        for t in range(case["frames"]):
            levels = [frames[:, t]]
            for _ in range(case["levels"] - 1):
                levels.append(_halve(_halve(levels[-1], -1, False), -2, False))
            state = _frame64(spec, state, levels, [g / 255.0 ** 2 for g in gamma])
            out.append(torch.stack(state[0][0], -1))
        flows = torch.stack(out, 1)
        if not case["grad"]:
            return flows
        loss = ((flows[:, 1:] - truth.double()[:, None]) ** 2).mean() + 0.1 * _photometric64(frames, flows)
        g_frames, g_gamma = torch.autograd.grad(loss, (frames, gamma))
    return dict(loss=loss.detach(), flows=flows.detach(), g_frames=g_frames, g_gamma=g_gamma)


def _photometric64(frames, flows):
    """Mean squared difference of frame t and frame t-1 sampled bilinearly at
    x - flow, coordinates clamped into the image."""
    B, T, h, w = frames.shape
    f = flows[:, 1:]
    sx = (torch.arange(w, device=f.device, dtype=f.dtype) - f[..., 0]).clamp(0, w - 1)
    sy = (torch.arange(h, device=f.device, dtype=f.dtype)[:, None] - f[..., 1]).clamp(0, h - 1)
    x0, y0 = sx.detach().floor(), sy.detach().floor()
    ax, ay = sx - x0, sy - y0
    x0, y0 = x0.long(), y0.long()
    x1, y1 = (x0 + 1).clamp(max=w - 1), (y0 + 1).clamp(max=h - 1)
    prev = frames[:, :-1].reshape(B, T - 1, h * w)

    def at(yy, xx):
        return prev.gather(2, (yy * w + xx).reshape(B, T - 1, h * w)).reshape(B, T - 1, h, w)

    v = (1 - ay) * ((1 - ax) * at(y0, x0) + ax * at(y0, x1)) + ay * ((1 - ax) * at(y1, x0) + ax * at(y1, x1))
    return ((frames[:, 1:] - v) ** 2).mean()
