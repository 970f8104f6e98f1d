"""Order of fused launches on several streams: the bookkeeping on the CPU (also
that of set-up once per device), and on the GPU what it counts against what the
launches did."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("program", ["launch_order", "per_device"])
def test_bookkeeping(tmp_path, program):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / program)
    subprocess.check_call([gxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread",
                           "-I" + os.path.join(ROOT, "optical-flow-filter_amd", "csrc"),
                           os.path.join(ROOT, "tests", "cpp", program + ".cpp"), "-o", exe])
    subprocess.check_call([exe], timeout=60)


def _pyr(h, w, levels=2):
    import flowfilter.gpu.flowfilters as gf
    f = gf.PyramidalFlowFilter(h, w, levels)
    f.gamma, f.maxflow, f.smoothIterations = [10.0, 30.0, 50.0, 50.0][:levels], 4.0, [2] * levels
    return f


def _frames(h, w, n, seed):
    from flowfilter import synthetic
    return list(synthetic.blob_affine(h, w, n, blobs=30, seed=seed))


def _order_state():
    from flowfilter import _native as N
    v = [ctypes.c_uint() for _ in range(3)]
    N.call("ff_wait_order_state", *[ctypes.byref(x) for x in v])
    return [x.value for x in v]


def _hip_runtime():
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    return ctypes.CDLL(path)


@pytest.mark.gpu
def test_an_earlier_error_does_not_upset_the_count(ffo):
    """An error that an earlier HIP call of the thread left behind is reported
    by compute(), though its launch ran: the launch stays counted, and frames
    of two streams after it are right. With launches replayed from a graph (4
    levels) and launched directly."""
    hip = _hip_runtime()
    h, w = 272, 512
    frames = _frames(h, w, 6, 4)
    for levels in (2, 4):
        print("earlier error", levels, flush=True)
        fs = [_pyr(h, w, levels) for _ in range(2)]
        for f in fs:
            for img in frames[:4]:
                f.loadImage(img)
                f.compute()
            f.elapsedTime()
        before = _order_state()
        assert before[0] == before[1] and (before[0] != 0 or levels == 4)
        fs[0].loadImage(frames[4])
        assert hip.hipSetDevice(1000) != 0  # (an invalid argument, refused on the host)
        try:
            fs[0].compute()
        except Exception as e:
            print("reported:", e, flush=True)
        hip.hipGetLastError()
        after = _order_state()
        assert after[0] == after[1]
        for f in fs[1:]:
            f.loadImage(frames[4])
            f.compute()
        # (the first filter's frame may have been taken back with its error: it
        # starts anew)
        fresh = _pyr(h, w, levels)
        o = ffo.PyramidalFlowFilter(h, w, levels)
        o.configure_like([10.0, 30.0, 50.0, 50.0][:levels], 4.0, [2] * levels)
        for t, img in enumerate(frames):
            o.compute(img)
            fresh.loadImage(img)
            fresh.compute()
            if t == 5:
                fs[1].loadImage(img)
                fs[1].compute()
        for f in (fs[1], fresh):
            assert np.array_equal(f.getFlow(), o.downloadFlow())
            assert f.waitTimeouts() == 0
        after = _order_state()
        assert after[0] == after[1]


@pytest.mark.gpu
def test_timeouts_of_replayed_frames_are_reported():
    """Frames of four levels are replayed from a graph: a wait in a replay that
    gives up (forced by the test hook) is an error of the next check, also
    after an earlier check has read the count."""
    from flowfilter import errors
    h, w = 1088, 2048
    f = _pyr(h, w, 4)
    assert f.graphs
    frames = _frames(h, w, 2, 4)
    step = lambda t: (f.loadImage(frames[t % 2]), f.compute())
    for t in range(4):
        step(t)
    f.elapsedTime()
    f.setWaitTest(4)
    for t in range(8):  # records the graphs, then replays them
        print("replayed frame", t, flush=True)
        step(t)
        with pytest.raises(errors.FilterError, match="spin limit"):
            f.elapsedTime()
    f.setWaitTest(0)
    step(0)
    f.elapsedTime()


def _backlog(stream, seconds):
    """About that much work on a torch stream, of one wave."""
    import torch
    e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    with torch.cuda.stream(stream):
        for _ in range(2):  # (the first loads the kernel)
            e[0].record()
            torch.cuda._sleep(10 ** 7)
            e[1].record()
            e[1].synchronize()
        ms = e[0].elapsed_time(e[1])
        print("10^7 cycles of it: %.2f ms" % ms, flush=True)
        torch.cuda._sleep(int(10 ** 7 * min(seconds * 1e3 / ms, 1e3)))


def _two_filters(ffo, h, w):
    """Two filters that have taken turns, one of them on a torch stream, and
    the oracle after the same frames."""
    import torch
    side = torch.cuda.Stream()
    a, b = _pyr(h, w), _pyr(h, w)
    a.stream = side.cuda_stream
    o = ffo.PyramidalFlowFilter(h, w, 2)
    o.configure_like([10.0, 30.0], 4.0, [2, 2])
    frames = _frames(h, w, 6, 9)
    for img in frames[:4]:
        for f in (a, b):
            f.loadImage(img)
            f.compute()
        o.compute(img)
    a.getFlow(), b.getFlow()
    return side, a, b, o, frames


@pytest.mark.gpu
def test_a_launch_behind_a_backlog_is_waited_for(ffo):
    """A filter's launch is queued behind a second of other work of its stream:
    a launch of a filter on another stream comes after it, however long that
    takes."""
    import time

    import torch
    h, w = 272, 512
    side, a, b, o, frames = _two_filters(ffo, h, w)
    own = torch.cuda.ExternalStream(b.stream)
    for t, img in enumerate(frames[4:]):
        print("backlog", t, flush=True)
        for f in (a, b):
            f.loadImage(img)
        _backlog(side, 1.0)
        busy = torch.cuda.Event()
        busy.record(side)
        a.compute()
        b.compute()
        time.sleep(0.6)
        assert not busy.query(), "the backlog is too short for this test"
        assert not own.query()
        o.compute(img)
        for f in (a, b):
            assert np.array_equal(f.getFlow(), o.downloadFlow())
            assert f.waitTimeouts() == 0
    st = _order_state()
    assert st[0] == st[1]


@pytest.mark.gpu
def test_a_wait_for_another_streams_launch_that_gives_up_is_an_error(ffo):
    """Forced by the test hook (a few polls, for a count that no launch
    reaches): the wait is counted and reported, the next launch finds the
    device idle, and the other filter's frames stay right."""
    from flowfilter import errors
    h, w = 272, 512
    side, a, b, o, frames = _two_filters(ffo, h, w)
    gave_up = _order_state()[2]
    img = frames[4]
    b.loadImage(img)
    b.compute()  # (in a state of its own from here on)
    b.elapsedTime()
    n = b.waitTimeouts()
    b.setWaitTest(4)
    b.compute()
    with pytest.raises(errors.FilterError, match="spin limit"):
        b.elapsedTime()
    alone = b.waitTimeouts() - n  # of a launch without another before it
    for f in (a, b):
        f.loadImage(img)
    _backlog(side, 0.2)
    a.compute()
    b.compute()
    with pytest.raises(errors.FilterError, match="spin limit"):
        b.elapsedTime()
    assert b.waitTimeouts() - n == 2 * alone + 1
    b.setWaitTest(0)
    o.compute(img)
    assert np.array_equal(a.getFlow(), o.downloadFlow())
    for f in (b, a):
        f.loadImage(frames[5])
        f.compute()
    b.elapsedTime()
    o.compute(frames[5])
    assert np.array_equal(a.getFlow(), o.downloadFlow())
    assert a.waitTimeouts() == 0
    st = _order_state()
    assert st[0] == st[1] and st[2] == gave_up + 1


@pytest.mark.gpu
def test_backlogs_on_streams_that_share_hardware_queues(ffo):
    """More filters on streams of their own than the process has hardware
    queues, while other streams, which share those queues, hold half a second of
    work each: no wait gives up and every flow is the oracle's."""
    import torch
    h, w = 272, 512
    fs = [_pyr(h, w) for _ in range(10)]
    o = ffo.PyramidalFlowFilter(h, w, 2)
    o.configure_like([10.0, 30.0], 4.0, [2, 2])
    gave_up = _order_state()[2]
    others = [torch.cuda.Stream() for _ in range(6)]
    for t, img in enumerate(_frames(h, w, 6, 21)):
        if t in (3, 5):
            print("backlogs at frame", t, flush=True)
            for s in others:
                _backlog(s, 0.5)
        for f in fs:
            f.loadImage(img)
        for f in fs:
            f.compute()
        o.compute(img)
    for k, f in enumerate(fs):
        assert np.array_equal(f.getFlow(), o.downloadFlow()), k
        assert f.waitTimeouts() == 0, k
    st = _order_state()
    assert st[0] == st[1] and st[2] == gave_up
