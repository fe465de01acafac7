"""The ray cast's skips over absent space against the oracle's sample by
sample: volumes wider than the occupancy grid's repeat, rays that start far
from any block and graze edges, coordinates large enough that additions round
coarsely, grids of cells in two chunks and too wide for chunks, and every
voxel format."""
import numpy as np
import pytest

from oracle import pyoracle as po
from yetanotherslam_amd import rgbdfusion as rf
from yetanotherslam_amd import synth

from helpers import assert_bits_equal, to_dev

pytestmark = pytest.mark.gpu

FMTS = {"i16": (rf.VOXEL_I16_U8, po.VOX_REF), "f32": (rf.VOXEL_F32_F32, po.VOX_F32), "f16": (rf.VOXEL_F16_U16, po.VOX_F16)}


def _pose(shift, yaw):
    T = np.eye(4)
    c, s = np.cos(yaw), np.sin(yaw)
    T[:3, :3] = [[c, 0, s], [0, 1, 0], [-s, 0, c]]
    T[:3, 3] = shift
    return T


def _with_intrinsics(m, K, Kr, tmp_path):
    """The volume with other intrinsics, which decide what is visible (the
    oracle takes a ray cast's own): by way of its file."""
    path = tmp_path / "v.yas"
    m.SaveToFile(path)
    data = bytearray(path.read_bytes())
    at = data.index(K.tobytes(), 0, 224)
    data[at:at + 16] = Kr.tobytes()
    path.write_bytes(bytes(data))
    return rf.MapStruct.ReadFromFile(path)


@pytest.mark.parametrize("w,h,voxel,trunc,fmt,shift,yaw,origin", [
    (320, 240, 0.008, 0.024, "f32", (0, 0, -1.0), 0.0, 0.0),      # starts a metre before the volume
    (320, 240, 0.008, 0.024, "i16", (0.8, 0.1, -0.5), -0.7, 0.0),  # across it, past silhouettes
    (160, 120, 0.002, 0.008, "f16", (0.1, 0, 0), 0.2, 0.0),       # 2 mm: the grid repeats every 2 m
    (160, 120, 0.01, 0.03, "f32", (0, 0, 0), 0.1, 900.0),         # 90000 voxels from the origin
    (160, 120, 0.01, 0.03, "f32", (0, 0, 0), 0.1, 9000.0),        # 900000 voxels
    (1280, 960, 0.01, 0.03, "f32", (0.2, 0, -0.3), -0.2, 0.0),    # two chunks of cells
    (480, 360, 0.01, 0.03, "i16", (-0.2, 0, -0.2), 0.3, 0.0),     # 32 rays a wavefront (64, 16 and 8 above)
    (77832, 8, 0.02, 0.06, "f32", (0, 0, -0.3), 0.0, 0.0),        # 9729 columns of cells
])
def test_ray_cast_equals_the_oracle(gpu, w, h, voxel, trunc, fmt, shift, yaw, origin, tmp_path):
    p = synth.params(width=160, height=120, theta0=0.7)
    K = synth.intrinsics(p)
    base = np.eye(4)
    base[0, 3] = origin
    gfmt, ofmt = FMTS[fmt]
    gm = rf.MapStruct(K.astype(np.float32), 1 << 18, 1 << 16, voxel, trunc, voxel_format=gfmt)
    om = po.OracleMap(voxel, trunc, voxfmt=ofmt)
    for t, T in enumerate(synth.relative_poses(p, 3)):
        z = po.depth_u16_to_f32(synth.frame(p, t)[0])
        gm.Fuse(to_dev(z), base @ T)
        om.fuse(z, K, base @ T)
    assert gm.stats().flags == 0 and gm.stats().num_allocated == om.num_blocks()
    Kr = (K * [w / 160, h / 120, w / 160, h / 120]).astype(np.float32)
    T = base @ _pose(shift, yaw)
    rc = rf.RayTraceEngine(w, h, Kr)
    rc.RayTrace(_with_intrinsics(gm, K.astype(np.float32), Kr, tmp_path), T)
    want, zmin, zmax = om.raycast(w, h, Kr.astype(np.float64), T)
    got = rc.GetVMap().reshape(h, w, 4)
    hit = want[..., 3] > 0
    assert hit.sum() > 100 and np.array_equal(got[..., 3] > 0, hit)
    assert_bits_equal(got[hit], want[hit].astype(np.float32), "vertices")


def test_visibility_is_by_the_map_s_intrinsics(gpu):
    """A ray caster with intrinsics of its own: the visible blocks are those
    that CheckNumVisibleBlocks counts, by the map's."""
    p = synth.params(width=160, height=120, theta0=0.7)
    K = synth.intrinsics(p).astype(np.float32)
    m = rf.MapStruct(K, 1 << 16, 1 << 14, 0.01, 0.03)
    m.FuseU16(to_dev(synth.frame(p, 0)[0]), np.eye(4))
    rc = rf.RayTraceEngine(160, 120, K * np.float32([3, 3, 1, 1]))
    T = _pose((0.1, 0, -0.2), 0.2)
    rc.RayTrace(m, T)
    own = rf.RayTraceEngine(160, 120, K)
    n = rc.GetNumVisibleBlock()
    own.RayTrace(m, T)
    assert n == own.GetNumVisibleBlock() == m.CheckNumVisibleBlocks(160, 120, T) > 100
