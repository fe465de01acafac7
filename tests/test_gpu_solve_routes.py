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
