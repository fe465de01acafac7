"""A map file with fewer buckets than blocks: the blocks that find no slot are
in no table, and saving, hibernation, integration and Reset touch no slot for
them.  After Reset the map is as good as a new one of its sizes."""
import numpy as np
import pytest

from yetanotherslam_amd import rgbdfusion as rf
from yetanotherslam_amd import synth

from helpers import to_dev

pytestmark = pytest.mark.gpu

PROBE_LIMIT = 2  # stats().flags


@pytest.mark.parametrize("fmt", [rf.VOXEL_I16_U8, rf.VOXEL_F32_F32, rf.VOXEL_F16_U16])
def test_reset_of_a_table_too_small_for_its_blocks(gpu, fmt, tmp_path):
    p = synth.params(width=160, height=120, theta0=0.7)
    K = synth.intrinsics(p).astype(np.float32)
    depth = to_dev(synth.frame(p, 0)[0])
    m = rf.MapStruct(K, 1 << 14, 1 << 12, 0.02, 0.06, voxel_format=fmt)
    m.FuseU16(depth, np.eye(4))
    path = tmp_path / "full.yas"
    m.SaveToFile(path)
    data = bytearray(path.read_bytes())
    n = int(np.frombuffer(data, np.int32, 1, 24)[0])
    buckets = n // 2 + 1
    data[16:20] = np.int32(buckets).tobytes()
    path.write_bytes(bytes(data))

    a = rf.MapStruct.ReadFromFile(path)
    st = a.stats()
    assert n > 300 and st.num_allocated == n and st.flags & PROBE_LIMIT
    voxels = a.export_sorted()
    a.SaveToFile(tmp_path / "again.yas")  # gathers the blocks' summaries
    a.Hibernate()
    a.ReActivate()
    for x, y in zip(a.export_sorted(), voxels):
        assert np.array_equal(np.asarray(x).view(np.uint32), np.asarray(y).view(np.uint32))
    a.FuseU16(depth, np.eye(4))  # stores the blocks' summaries
    a.Reset()
    st = a.stats()
    assert (st.num_allocated, st.num_visible, st.flags) == (0, 0, 0)

    near = np.zeros((120, 160), np.uint16)
    near[40:80, 60:100] = 400
    b = rf.MapStruct(K, buckets, 1 << 12, 0.02, 0.06, voxel_format=fmt)
    for x in (a, b):
        x.FuseU16(to_dev(near), np.eye(4))
        assert x.stats().flags == 0 and x.stats().num_allocated > 0
    for x, y in zip(a.export_sorted(), b.export_sorted()):
        assert np.array_equal(np.asarray(x).view(np.uint32), np.asarray(y).view(np.uint32))
