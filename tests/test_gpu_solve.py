"""The tracker's one-launch solve: the same bits as the launch-per-pass solve
whatever the size (one workgroup or 256, one to three rounds of pixel slots
a thread, a level without iterations), whether its workgroups meet or the
rescue takes the solve, and when another stream holds the one-launch path.

The launch-per-pass code itself is checked against the oracle elsewhere; here
it runs as the rescue, forced by a wait bound of 0."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DEFAULT_TICKS = 2000000


def _tracker(w, h, mode, iters=(10, 5, 3), ctx=None):
    import torch
    from oracle import pyoracle as po
    from yetanotherslam_amd import rgbdfusion as rf
    from yetanotherslam_amd import synth
    p = synth.params(width=w, height=h, theta0=0.7)
    p.noise_k, p.step = 0.0002, 0.004
    K = synth.intrinsics(p)
    fr = [synth.frame(p, t) for t in range(2)]
    z = [torch.from_numpy(po.depth_u16_to_f32(f[0])).cuda() for f in fr]
    g = [torch.from_numpy((f[1].astype(np.float32) @ np.array([0.299, 0.587, 0.114], np.float32))).cuda() for f in fr]
    torch.cuda.synchronize()
    trk = rf.RGBDTracking(w, h, K, len(iters), iters, mode, (0.1, 0.1, 1.0, 1.0), ctx=ctx)
    trk.SetReferenceImage(g[0])
    trk.SetReferenceDepth(z[0])
    trk.SetTrackingImage(g[1])
    trk.SetTrackingDepth(z[1])
    trk._keep = (z, g)
    return trk


def _set_ticks(trk, ticks):
    from yetanotherslam_amd import native
    f = native.lib().yas_tracker_set_wait_ticks
    f.argtypes = [ctypes.c_void_p, ctypes.c_ulonglong]
    assert f(trk.h, ticks) == 0


def _solve(trk, init=None):
    T, st = trk.GetTransform(init=init, swap=False)
    return T, (st.good, st.icp_inliers, st.rgb_inliers, np.float32(st.last_error).tobytes())


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("w,h,iters", [
    (32, 24, (4,)),            # one workgroup
    (36, 28, (3, 2)),          # 1008 pixels: the last slot partly past the image
    (164, 124, (4, 2, 2)),     # 20 workgroups, short of four slots a thread
    (320, 240, (3, 0, 2)),     # a level without iterations
    (644, 484, (3, 2, 1)),     # 256 workgroups, a second round for some wavefronts
    (1280, 968, (2, 1)),       # more rounds than LDS keeps residuals for
])
def test_one_launch_solve_equals_passes(gpu, w, h, iters, mode):
    trk = _tracker(w, h, mode, iters)
    T, st = _solve(trk)
    T2, st2 = _solve(trk)  # the next solve's epochs
    assert np.array_equal(T, T2) and st == st2
    _set_ticks(trk, 0)
    Tr, sr = _solve(trk)
    assert np.array_equal(T, Tr), (T, Tr)
    assert st == sr
    _set_ticks(trk, DEFAULT_TICKS)
    T3, st3 = _solve(trk)  # after a rescue
    assert np.array_equal(T, T3) and st == st3


def test_one_launch_solve_after_nan_update(gpu):
    """A NaN pose: the same status by both routes, and the next solve is sound."""
    from yetanotherslam_amd.native import YasError  # noqa: F401
    trk = _tracker(320, 240, 2)
    T, st = _solve(trk)
    bad = np.eye(4)
    bad[0, 3] = np.nan
    a = _solve(trk, bad)
    _set_ticks(trk, 0)
    b = _solve(trk, bad)
    _set_ticks(trk, DEFAULT_TICKS)
    assert np.array_equal(a[0], b[0], equal_nan=True) and a[1] == b[1]
    T2, st2 = _solve(trk)
    assert np.array_equal(T, T2) and st == st2


def test_solves_on_two_streams(gpu):
    """Two trackers on streams of their own, each enqueued while the other's
    stream is busy: one of them takes the passes, with the same bits."""
    import torch
    from yetanotherslam_amd import rgbdfusion as rf
    ctxs, trks = [], []
    for _ in range(2):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            ctxs.append((s, rf.Context()))
            trks.append(_tracker(320, 240, 2, ctx=ctxs[-1][1]))
    want = [_solve(t) for t in trks]
    assert np.array_equal(want[0][0], want[1][0])
    x = torch.zeros(1 << 26, device="cuda")
    torch.cuda.synchronize()
    for _ in range(3):
        for i in (0, 1):
            with torch.cuda.stream(ctxs[1 - i][0]):
                for _ in range(20):
                    x.add_(1.0)  # the other stream is busy
            got = _solve(trks[i])
            assert np.array_equal(got[0], want[i][0]) and got[1] == want[i][1]
    torch.cuda.synchronize()
