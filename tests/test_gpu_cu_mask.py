"""A context on a stream that may use a part of the CUs: launches are sized
for those, a solve whose workgroups they do not hold at once takes the separate
passes, and every result has the same bits."""
import ctypes

import numpy as np
import pytest

from yetanotherslam_amd import native
from yetanotherslam_amd import rgbdfusion as rf
from yetanotherslam_amd import synth

from helpers import to_dev

pytestmark = pytest.mark.gpu


def _hip():
    native.lib()
    with open("/proc/self/maps") as fh:
        return ctypes.CDLL(next(l.split()[-1] for l in fh if "libamdhip64" in l))


def _work(ctx, w, h):
    p = synth.params(width=w, height=h, theta0=0.7)
    p.noise_k, p.step = 0.0002, 0.004
    K = synth.intrinsics(p)
    m = rf.MapStruct(K.astype(np.float32), 1 << 16, 1 << 13, 0.01, 0.04, ctx=ctx)
    rc = rf.RayTraceEngine(w, h, K, ctx=ctx)
    trk = rf.RGBDTracking(w, h, K, 3, (4, 2, 2), rf.TRACK_RGBD, (0.1, 0.1, 1.0, 1.0), ctx=ctx)
    keep = []
    for t in range(2):
        d, c = synth.frame(p, t)[:2]
        raw, z = to_dev(d), to_dev(d.astype(np.float32) * np.float32(0.001))
        g = to_dev(c.astype(np.float32) @ np.array([0.299, 0.587, 0.114], np.float32))
        keep += [raw, z, g]
        m.FuseU16(raw, np.eye(4))
        (trk.SetReferenceDepth, trk.SetTrackingDepth)[t](z)
        (trk.SetReferenceImage, trk.SetTrackingImage)[t](g)
    rc.RayTrace(m, np.eye(4))
    T, st = trk.GetTransform(swap=False)
    r = (ctypes.c_int * 3)()
    native.call("yas_tracker_solve_routes", trk.h, r)
    mesh = rf.canonical_mesh(rf.MeshEngine(1 << 20, ctx=ctx).Meshify(m))
    return [rc.GetVMap(), T, np.array([st.good, st.icp_inliers, st.rgb_inliers]), mesh[3], mesh[4]], list(r)


@pytest.mark.parametrize("w,h", [(160, 120), (320, 240)])
def test_results_on_64_cus(gpu, w, h):
    import torch
    hip = _hip()
    want, routes = _work(rf.default_context(), w, h)
    assert routes == [1, 0, 0]
    mask = (ctypes.c_uint32 * 2)(0xFFFFFFFF, 0xFFFFFFFF)
    s = ctypes.c_void_p()
    assert hip.hipExtStreamCreateWithCUMask(ctypes.byref(s), ctypes.c_uint32(2), mask) == 0
    with torch.cuda.stream(torch.cuda.ExternalStream(s.value)):
        ctx = rf.Context()
        got, routes = _work(ctx, w, h)
        torch.cuda.synchronize()
    # 19 workgroups, and 75 of which each takes a CU
    assert routes == ([1, 0, 0] if w == 160 else [0, 0, 1])
    for a, b in zip(got, want):
        assert np.array_equal(np.asarray(a).view(np.uint32), np.asarray(b).view(np.uint32))
