"""A pipeline past its first 1024 frames: poses, outcomes and statistics of
the frames before are kept when their arrays grow."""
import ctypes

import numpy as np
import pytest

from yetanotherslam_amd import native
from yetanotherslam_amd import rgbdfusion as rf
from yetanotherslam_amd import synth

from helpers import to_dev

pytestmark = pytest.mark.gpu


def _stats(pl, n):
    out = (ctypes.c_int * (8 * n))()
    native.call("yas_pipeline_frame_stats", pl.h, 0, n, out)
    return np.array(out).reshape(n, 8)


def test_what_is_known_of_1024_frames_is_kept(gpu):
    p = synth.params(width=64, height=48, theta0=0.7)
    p.step = 0.002
    fr = [tuple(to_dev(x) for x in synth.frame(p, t)[:2]) for t in range(4)]
    pl = rf.DensePipeline(64, 48, synth.intrinsics(p), rf.map_params(1 << 14, 1 << 11, 0.02, 0.08),
                          rf.tracker_params(3, (2, 1, 1), rf.TRACK_DEPTH))
    for i in range(1024):
        pl.step(*fr[(0, 1, 2, 3, 2, 1)[i % 6]])
    poses = [pl.pose(i) for i in range(1024)]
    stats = _stats(pl, 1024)
    for i in range(1024, 1030):
        pl.step(*fr[(0, 1, 2, 3, 2, 1)[i % 6]])
    assert pl.num_frames() == 1030 and stats[:, 0].min() > 0
    for i, (T, ok) in enumerate(poses):
        got = pl.pose(i)
        assert np.array_equal(got[0], T) and got[1] == ok
    assert np.array_equal(_stats(pl, 1030)[:1024], stats)
    assert all(np.isfinite(pl.pose(i)[0]).all() for i in range(1024, 1030))
