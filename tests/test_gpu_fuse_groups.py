"""Allocation by workgroups of 32x32 pixels: the oracle's volume where a
workgroup finds more new blocks than its list holds and where the image ends
inside a tile; uint16 depth fused without a converted image; and Reset, which
clears only what a map holds, also after its pool overflowed."""
import numpy as np
import pytest

from oracle import pyoracle as po
from yetanotherslam_amd import rgbdfusion as rf
from yetanotherslam_amd import synth

from helpers import assert_bits_equal, to_dev

pytestmark = pytest.mark.gpu


def _scene(w, h, n=2):
    p = synth.params(width=w, height=h, theta0=0.7)
    return synth.intrinsics(p), [synth.frame(p, t)[0] for t in range(n)], synth.relative_poses(p, n)


def _same(gm, om):
    kg, sg, wg = gm.export_sorted()
    ko, so, wo = om.export()
    assert np.array_equal(kg, ko), (len(kg), len(ko))
    assert_bits_equal(sg, so.astype(np.float32), "sdf")
    assert np.array_equal(wg, wo.astype(np.float32))


@pytest.mark.parametrize("w,h,voxel,trunc", [
    (33, 31, 0.002, 0.20),    # walks of some 13 blocks a pixel: over 512 new blocks in a tile
    (64, 32, 0.02, 0.06),     # whole tiles, few blocks
    (95, 65, 0.01, 0.04),     # both ends inside a tile
])
def test_fused_blocks_equal_the_oracle_s(gpu, w, h, voxel, trunc):
    K, depth, T = _scene(w, h)
    gm = rf.MapStruct(K.astype(np.float32), 1 << 18, 1 << 16, voxel, trunc)
    gu = rf.MapStruct(K.astype(np.float32), 1 << 18, 1 << 16, voxel, trunc)
    om = po.OracleMap(voxel, trunc)
    for d, t in zip(depth, T):
        z = po.depth_u16_to_f32(d)
        gm.Fuse(to_dev(z), t)
        gu.FuseU16(to_dev(d), t)
        om.fuse(z, K, t)
    if voxel < 0.005:
        assert gm.stats().num_allocated > 2 * 512
    _same(gm, om)
    _same(gu, om)
    assert gm.stats().reserved == gu.stats().reserved  # walk steps


@pytest.mark.parametrize("fmt", [0, 1, 2])
@pytest.mark.parametrize("blocks", [1 << 14, 256])  # 256: the pool overflows
def test_reset_then_fuse_equals_a_new_map(gpu, fmt, blocks):
    K, depth, T = _scene(160, 120)
    K = K.astype(np.float32)
    a = rf.MapStruct(K, 1 << 15, blocks, 0.01, 0.04, voxel_format=fmt)
    for d, t in zip(depth, T):
        a.FuseU16(to_dev(d), t)
    assert bool(a.stats().flags & 1) == (blocks == 256)
    a.Reset()
    st = a.stats()
    assert (st.num_allocated, st.num_visible, st.flags, st.reserved) == (0, 0, 0, 0)
    assert a.CheckNumVisibleBlocks(160, 120, T[0]) == 0
    # a far smaller scene than the first, so that leftovers would show
    near = np.full((120, 160), 400, np.uint16)
    b = rf.MapStruct(K, 1 << 15, 1 << 14, 0.01, 0.04, voxel_format=fmt)
    if blocks == 256:
        near[:, 40:] = 0
    for m in (a, b):
        m.FuseU16(to_dev(near), np.eye(4))
    assert a.stats().flags == 0
    for x, y in zip(a.export_sorted(), b.export_sorted()):
        assert np.array_equal(np.asarray(x).view(np.uint32), np.asarray(y).view(np.uint32))
    rc = rf.RayTraceEngine(160, 120, K)
    views = []
    for m in (a, b):
        rc.RayTrace(m, np.eye(4))
        views.append(rc.GetVMap())
    assert np.array_equal(views[0].view(np.uint32), views[1].view(np.uint32))
