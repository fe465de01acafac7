"""Marching cubes over volumes of random voxels, where the emission passes'
lists of a block's triangles and vertices run from empty to filled several
times over, blocks miss some of their neighbours, and voxels hold zeros and
values of magnitude 1e-6: cases, counts and triangles equal the oracle's, and
the indexed form's vertices are those of the owned edges, in order."""
import numpy as np
import pytest

from oracle import pyoracle as po
from yetanotherslam_amd import rgbdfusion as rf
from yetanotherslam_amd import synth

from helpers import assert_bits_equal, to_dev

pytestmark = pytest.mark.gpu

FMTS = [(rf.VOXEL_I16_U8, po.VOX_REF), (rf.VOXEL_F32_F32, po.VOX_F32), (rf.VOXEL_F16_U16, po.VOX_F16)]


def _raw(fmt, rng, n, observed):
    """n blocks of raw voxels: signs at random, some zeros and tiny values."""
    s = rng.uniform(0.01, 1.0, (n, 512)).astype(np.float32) * rng.choice([-1, 1], (n, 512)).astype(np.float32)
    pick = rng.random((n, 512))
    s[pick < 0.05] = 0.0
    s[(pick >= 0.05) & (pick < 0.10)] = 5e-7
    s[(pick >= 0.10) & (pick < 0.12)] = -0.0
    w = (rng.random((n, 512)) < observed).astype(np.float32) * 3
    if fmt == rf.VOXEL_F32_F32:
        return np.stack([s, w], -1).astype(np.float32).view(np.uint8).reshape(n, -1)
    if fmt == rf.VOXEL_I16_U8:
        lo = (s * 32767).astype(np.int16).view(np.uint16)
    else:
        lo = s.astype(np.float16).view(np.uint16)
    return (lo.astype(np.uint32) | (w.astype(np.uint32) << 16)).view(np.uint8).reshape(n, -1)


def _volume(tmp_path, fmt, observed):
    """A saved map's file with its voxels replaced, read back."""
    p = synth.params(width=64, height=48, theta0=0.7)
    K = synth.intrinsics(p).astype(np.float32)
    m = rf.MapStruct(K, 1 << 14, 1 << 12, 0.02, 0.06, voxel_format=fmt)
    m.FuseU16(to_dev(synth.frame(p, 0)[0]), np.eye(4))
    path = tmp_path / "noise.yas"
    m.SaveToFile(path)
    m.close()
    data = bytearray(path.read_bytes())
    n = int(np.frombuffer(data, np.int32, 1, 24)[0])
    rec = np.frombuffer(data, np.int32, 4 * n, 224).reshape(n, 4).copy()
    raw = _raw(fmt, np.random.default_rng(7), n, observed)
    rec[:, 3] = 0
    data[224:224 + 16 * n] = rec.tobytes()
    data[224 + 16 * n:] = raw.tobytes()
    path.write_bytes(bytes(data))
    return rf.MapStruct.ReadFromFile(path), n


def _owned_vertices(keys, sdf, wt, voxel):
    """Vertices of the owned edges by block, voxel and axis, float32."""
    lo = keys.min(0)
    dim = (keys.max(0) - lo + 2) * 8
    s = np.zeros(dim[::-1], np.float32)  # [z, y, x]
    o = np.zeros(dim[::-1], bool)
    for k, a, b in zip(keys - lo, sdf, wt):
        at = tuple(slice(8 * k[i], 8 * k[i] + 8) for i in (2, 1, 0))
        s[at], o[at] = a.reshape(8, 8, 8), b.reshape(8, 8, 8) != 0
    out, per_block = [], []
    l = np.arange(512)
    x, y, z = l & 7, (l >> 3) & 7, l >> 6
    for k in keys:
        kx, ky, kz = 8 * (k - lo)
        v1, o1 = s[kz + z, ky + y, kx + x], o[kz + z, ky + y, kx + x]
        pos = np.stack([8 * k[0] + x, 8 * k[1] + y, 8 * k[2] + z], -1).astype(np.float32)
        verts, has = np.zeros((512, 3, 3), np.float32), np.zeros((512, 3), bool)
        for a, (dx, dy, dz) in enumerate(((1, 0, 0), (0, 1, 0), (0, 0, 1))):
            v2, o2 = (g[kz + z + dz, ky + y + dy, kx + x + dx] for g in (s, o))
            has[:, a] = o1 & o2 & ((v1 < 0) != (v2 < 0))
            with np.errstate(divide="ignore", invalid="ignore"):
                t = (np.float32(0) - v1) / (v2 - v1)
            t = np.where(np.abs(v1 - v2) < 1e-6, np.float32(0), t)
            t = np.where(np.abs(v2).astype(np.float64) < 1e-6, np.float32(1), t)
            t = np.where(np.abs(v1).astype(np.float64) < 1e-6, np.float32(0), t)
            p = pos.copy()
            p[:, a] = p[:, a] + t
            verts[:, a] = p * np.float32(voxel)
        out.append(verts[has])
        per_block.append(int(has.sum()))
    return np.concatenate(out), per_block


@pytest.mark.parametrize("fmt,ofmt", FMTS, ids=["i16u8", "f32", "f16u16"])
@pytest.mark.parametrize("observed", [1.0, 0.9, 0.3])
def test_random_volume(gpu, tmp_path, fmt, ofmt, observed):
    m, n = _volume(tmp_path, fmt, observed)
    keys, sdf, wt = m.export_sorted()
    om = po.OracleMap(0.02, 0.06, voxfmt=ofmt)
    om.import_blocks(keys, sdf, wt)
    mo = om.mesh()
    me = rf.MeshEngine(5 * 512 * n)  # the most a volume can hold
    soup = me.Meshify(m, with_cases=True)
    ks, counts, cases, tris, normals = rf.canonical_mesh(soup)
    np.testing.assert_array_equal(mo["keys"], ks)
    np.testing.assert_array_equal(mo["cases"], cases)
    np.testing.assert_array_equal(mo["counts"], counts)
    assert soup["num_triangles"] == len(mo["tris"])
    assert_bits_equal(mo["tris"], tris, "vertices")
    assert_bits_equal(mo["normals"], normals, "normals")
    if observed == 1.0:
        assert counts.max() > 2 * 512  # a block's triangle list is emptied and filled again
    pool = {tuple(k): i for i, k in enumerate(map(tuple, keys))}
    order = [pool[tuple(k)] for k in soup["keys"]]
    V, per_block = _owned_vertices(soup["keys"], sdf[order], wt[order], np.float32(0.02))
    ix = me.MeshifyIndexed(m)
    assert ix["num_vertices"] == len(V) and ix["num_triangles"] == len(mo["tris"])
    assert_bits_equal(ix["vertices"], V, "owned vertices")
    # corner by corner the soup's: an edge's point from either end, a few
    # roundings of a coordinate of at most 2^9 voxels apart
    np.testing.assert_allclose(ix["vertices"][ix["triangles"]].reshape(-1, 9), soup["tris"], rtol=0,
                               atol=4 * 2.0 ** -15 * 0.02)
    m.close()


@pytest.mark.parametrize("indexed", [False, True])
def test_one_engine_over_volumes_of_different_size(gpu, indexed):
    """The engine's records are sized by the volumes before: one that fits,
    one that outgrows them, a small one after it and an empty one all give
    what an engine of their own gives."""
    p = synth.params(width=160, height=120, theta0=0.7)
    K = synth.intrinsics(p).astype(np.float32)
    gt = synth.relative_poses(p, 6)
    maps = []
    for n in (1, 6, 1, 0):
        m = rf.MapStruct(K, 1 << 15, 1 << 13, 0.01, 0.04)
        for t in range(n):
            m.FuseU16(to_dev(synth.frame(p, 3 * t)[0]), gt[t])
        maps.append(m)
    nb = [m.stats().num_allocated for m in maps]
    assert nb[1] > 1.25 * nb[0] > 0 and nb[3] == 0
    me = rf.MeshEngine(2_000_000)
    for m in [maps[3]] + maps:
        own = rf.MeshEngine(2_000_000)
        a, b = ((e.MeshifyIndexed(m) if indexed else e.Meshify(m, with_cases=True)) for e in (me, own))
        assert a.keys() == b.keys()
        for k in a:
            assert np.array_equal(a[k], b[k]), k
        own.close()
