"""Which way a solve takes (one launch, one launch lost and taken again, or
separate passes), and that every way gives the same bits."""
import ctypes

import numpy as np
import pytest

from yetanotherslam_amd import native
from yetanotherslam_amd import rgbdfusion as rf
from yetanotherslam_amd import synth

from helpers import to_dev

pytestmark = pytest.mark.gpu


def _pipeline(w=320, h=240, n=8, ctx=None, mode=rf.TRACK_RGBD):
    """A pipeline and its frames on the device."""
    p = synth.params(width=w, height=h, theta0=0.7)
    p.noise_k, p.step = 0.0002, 0.004
    pl = rf.DensePipeline(w, h, synth.intrinsics(p), rf.map_params(1 << 16, 1 << 13, 0.01, 0.04),
                          rf.tracker_params(3, (10, 5, 3), mode, (0.1, 0.1, 1.0, 1.0)), ctx=ctx)
    return pl, [tuple(to_dev(x) for x in synth.frame(p, t)[:2]) for t in range(n)]


def _poses(pl):
    return np.stack([pl.pose(i)[0] for i in range(pl.num_frames())])


def test_steps_beside_a_capture(gpu):
    """Pipelines on streams of their own step while another stream's work is
    captured in the global mode: the capture stands, and so do the poses."""
    import torch
    streams = [torch.cuda.Stream() for _ in range(2)]
    pls = []
    for s in streams:
        with torch.cuda.stream(s):
            pls.append(_pipeline(ctx=rf.Context()))
    ref, frames = _pipeline()
    for f in frames[:6]:
        ref.step(*f)
    want = _poses(ref)
    for pl, fr in pls:
        for f in fr[:3]:
            pl.step(*f)
    x = torch.zeros(1024, device="cuda")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, capture_error_mode="global"):
        x.add_(1.0)
        for k in range(3, 6):
            for pl, fr in pls:
                pl.step(*fr[k])
        x.add_(1.0)
    for k in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert float(x[0]) == 2.0 * (k + 1)
    for pl, _ in pls:
        assert np.array_equal(_poses(pl), want)


DEFAULT_TICKS = 2000000


def _ticks(h, ticks):
    native.call("yas_tracker_set_wait_ticks", h, ticks)


def _routes(h):
    r = (ctypes.c_int * 3)()
    native.call("yas_tracker_solve_routes", h, r)
    return list(r)  # in one launch, lost, passes


def _tracker(w, h, mode, iters=(10, 5, 3), ctx=None):
    p = synth.params(width=w, height=h, theta0=0.7)
    p.noise_k, p.step = 0.0002, 0.004
    trk = rf.RGBDTracking(w, h, synth.intrinsics(p), len(iters), iters, mode, (0.1, 0.1, 1.0, 1.0), ctx=ctx)
    keep = []
    for t in range(2):
        d, c = synth.frame(p, t)[:2]
        z = to_dev(d.astype(np.float32) * np.float32(0.001))
        g = to_dev(c.astype(np.float32) @ np.array([0.299, 0.587, 0.114], np.float32))
        keep.append((z, g))
        (trk.SetReferenceDepth, trk.SetTrackingDepth)[t](z)
        (trk.SetReferenceImage, trk.SetTrackingImage)[t](g)
    trk._keep = keep
    _ticks(trk.h, DEFAULT_TICKS)  # whatever other tests left
    return trk


def _solve(trk):
    T, st = trk.GetTransform(swap=False)
    return T, (st.good, st.icp_inliers, st.rgb_inliers, np.float32(st.last_error).tobytes())


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("w,h,iters", [(32, 24, (4,)), (164, 124, (4, 2, 2)), (644, 484, (3, 2, 1)), (1280, 968, (2, 1))])
def test_a_solve_is_one_launch_and_a_lost_one_is_taken_again(gpu, w, h, iters, mode):
    trk = _tracker(w, h, mode, iters)
    T, st = _solve(trk)
    assert _routes(trk.h) == [1, 0, 0]
    if w == 32:  # one workgroup waits for itself alone
        return
    _ticks(trk.h, 0)
    Tl, sl = _solve(trk)
    assert _routes(trk.h) == [1, 1, 0]
    _ticks(trk.h, DEFAULT_TICKS)
    T2, s2 = _solve(trk)
    assert _routes(trk.h) == [2, 1, 0]
    assert np.array_equal(T, Tl) and np.array_equal(T, T2) and st == sl == s2


def test_a_stream_beside_a_busy_one_takes_the_passes(gpu):
    import torch
    s = [torch.cuda.Stream() for _ in range(2)]
    trks = []
    for q in s:
        with torch.cuda.stream(q):
            trks.append(_tracker(320, 240, 2, ctx=rf.Context()))
    with torch.cuda.stream(s[0]):
        pl, fr = _pipeline(ctx=trks[0].ctx)
    want = _solve(trks[1])
    x = torch.zeros(1 << 26, device="cuda")
    torch.cuda.synchronize()
    pl.step(*fr[0])
    with torch.cuda.stream(s[0]):
        for _ in range(600):  # some 60 ms, then a solve
            x.add_(1.0)
    pl.step(*fr[1])
    got = _solve(trks[1])
    assert _routes(trks[1].h) == [1, 0, 1]
    torch.cuda.synchronize()
    again = _solve(trks[1])
    assert _routes(trks[1].h) == [2, 0, 1]
    for g in (got, again):
        assert np.array_equal(g[0], want[0]) and g[1] == want[1]


@pytest.mark.parametrize("mode", [0, 2])
def test_queued_solves_that_are_lost_are_rescued(gpu, mode):
    """A pipeline with the bound at 0 in some frames: the rescue that follows
    each queued solve takes those, with the same bits, and no others."""
    lost = (2, 3, 6)
    ref, frames = _pipeline(mode=mode)
    pl, _ = _pipeline(mode=mode, n=1)
    h = ctypes.c_void_p()
    native.call("yas_pipeline_tracker", pl.h, ctypes.byref(h))
    for i, f in enumerate(frames):
        ref.step(*f)
        _ticks(h, 0 if i in lost else DEFAULT_TICKS)
        pl.step(*f)
        assert np.array_equal(pl.pose(i)[0], ref.pose(i)[0]) and pl.pose(i)[1] == ref.pose(i)[1], i
    assert _routes(h) == [len(frames) - 1 - len(lost), len(lost), 0]


def test_many_coarse_iterations_are_no_time_out(gpu):
    """Workgroups without work on the coarse level wait for all of its
    iterations together, far longer than the bound that holds for one."""
    trk = _tracker(320, 240, 2, (1, 6000))
    T, st = _solve(trk)
    assert _routes(trk.h) == [1, 0, 0]
    _ticks(trk.h, 0)
    Tl, sl = _solve(trk)
    assert _routes(trk.h) == [1, 1, 0]
    assert np.array_equal(T, Tl) and st == sl


def test_after_a_lost_solve_come_passes(gpu):
    """A solve that waits in vain is not tried again each time: 64 solves are
    separate passes, 128 after the next loss, and 64 again once one completes."""
    trk = _tracker(164, 124, 0, (2, 1, 1))
    T, st = _solve(trk)
    done, lost, passes = 1, 0, 0

    def solve(n=1):
        for _ in range(n):
            got = _solve(trk)
            assert np.array_equal(got[0], T) and got[1] == st

    _ticks(trk.h, 0)
    for n in (64, 128):
        solve(1 + n)
        lost, passes = lost + 1, passes + n
        assert _routes(trk.h) == [done, lost, passes]
    _ticks(trk.h, DEFAULT_TICKS)
    solve(3)
    done += 3
    assert _routes(trk.h) == [done, lost, passes]
    _ticks(trk.h, 0)
    solve(1 + 64 + 1)
    assert _routes(trk.h) == [done, lost + 2, passes + 64]


@pytest.mark.parametrize("wait", [True, False])
def test_after_a_rescued_frame_come_passes(gpu, wait):
    """The same where the solves are queued: the loss is known once the frame
    has run, and frames queued before that are rescued too."""
    ref, frames = _pipeline()
    pl, _ = _pipeline(n=1)
    h = ctypes.c_void_p()
    native.call("yas_pipeline_tracker", pl.h, ctypes.byref(h))
    _ticks(h, 0)
    for i, f in enumerate(frames):
        ref.step(*f)
        pl.step(*f)
        if wait:
            pl.pose(i)
    assert np.array_equal(_poses(pl), _poses(ref))
    done, lost, passes = _routes(h)
    assert done == 0 and lost + passes == len(frames) - 1 and lost >= 1
    if wait:
        assert lost == 1
    for i in range(8):
        pl.step(*frames[6 - i % 2])
        pl.pose(len(frames) + i)
    assert _routes(h)[1] == lost  # still by passes, once, however many were lost together


def test_overlapping_solves_of_large_images_take_the_passes(gpu):
    """Two cameras whose frames are enqueued without waiting: a one-launch
    solve on every CU would hold up the other camera, so neither takes it while
    their solves overlap, nor for 32 solves after; the poses are the same."""
    import torch
    size = dict(w=640, h=480)
    streams = [torch.cuda.Stream() for _ in range(2)]
    ref, frames = _pipeline(**size)
    pls, hs = [], []
    for q in streams:
        with torch.cuda.stream(q):
            pls.append(_pipeline(n=1, ctx=rf.Context(), **size)[0])
        h = ctypes.c_void_p()
        native.call("yas_pipeline_tracker", pls[-1].h, ctypes.byref(h))
        hs.append(h)
    for f in frames:
        ref.step(*f)
    want = _poses(ref)
    _ticks(hs[0], DEFAULT_TICKS)  # whatever other tests left
    x = torch.zeros(1 << 26, device="cuda")
    torch.cuda.synchronize()
    for pl in pls:
        pl.step(*frames[0])
    for i in (1, 2):  # waited for one after the other: no overlap
        for pl in pls:
            pl.step(*frames[i])
            pl.pose(i)
    assert [_routes(h) for h in hs] == [[2, 0, 0]] * 2
    for q in streams:
        with torch.cuda.stream(q):
            for _ in range(600):  # some 60 ms
                x.add_(1.0)
    for f in frames[3:]:
        for pl in pls:
            pl.step(*f)
    torch.cuda.synchronize()
    n = len(frames) - 3
    # the first of all finds no other solve
    assert [_routes(h) for h in hs] == [[3, 0, n - 1], [2, 0, n]]
    for pl in pls:
        assert np.array_equal(_poses(pl), want)
    for i in range(33):  # alone again
        assert _routes(hs[0]) == [3, 0, n - 1 + i]
        pls[0].step(*frames[(6, 7)[i % 2]])
        pls[0].pose(len(frames) + i)
    assert _routes(hs[0]) == [4, 0, n - 1 + 32]
