"""What a mesh engine keeps from its creation and from one extraction to the
next, on streams of its own and over volumes of different sizes."""
import numpy as np
import pytest

from yetanotherslam_amd import rgbdfusion as rf
from yetanotherslam_amd import synth

from helpers import to_dev

pytestmark = pytest.mark.gpu


def _room(voxel=0.01, blocks=1 << 14, ctx=None, w=160, h=120):
    p = synth.params(width=w, height=h, theta0=0.7)
    K = synth.intrinsics(p).astype(np.float32)
    m = rf.MapStruct(K, 8 * blocks, blocks, voxel, 4 * voxel, ctx=ctx)
    m.FuseU16(to_dev(synth.frame(p, 0)[0]), np.eye(4))
    return m


def _same(a, b):
    assert a["num_triangles"] == b["num_triangles"] > 100 and a["num_vertices"] == b["num_vertices"]
    assert np.array_equal(a["triangles"], b["triangles"])
    assert np.array_equal(a["vertices"].view(np.uint32), b["vertices"].view(np.uint32))


def test_engine_made_while_the_null_stream_is_busy(gpu):
    """Its scan's counter is cleared in order with its own stream, whatever
    waits on the null stream."""
    import torch
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        ctx = rf.Context()
        m = _room(ctx=ctx)
        torch.cuda.synchronize()
        want = rf.MeshEngine(1 << 19, ctx=ctx).MeshifyIndexed(m)
        for _ in range(4):
            with torch.cuda.stream(torch.cuda.default_stream()):
                torch.cuda._sleep(20_000_000)
            e = rf.MeshEngine(1 << 19, ctx=ctx)
            for _ in range(2):
                _same(e.MeshifyIndexed(m), want)
        torch.cuda.synchronize()


def test_first_extraction_takes_the_records_it_needs(gpu):
    """Device memory of an engine's first extraction: 2096 bytes a block and
    little more; an engine that outgrows its records gets the same mesh."""
    import torch
    p = synth.params(width=320, height=240, theta0=0.7)
    K = synth.intrinsics(p).astype(np.float32)
    big = rf.MapStruct(K, 1 << 18, 1 << 17, 0.004, 0.3)
    big.FuseU16(to_dev(synth.frame(p, 0)[0]), np.eye(4))
    n = big.stats().num_allocated
    assert n > 40000 and big.stats().flags == 0
    small = _room()
    used = []
    for _ in range(2):
        e = rf.MeshEngine(1 << 21)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        mesh = e.MeshifyIndexed(big)
        used.append(free - torch.cuda.mem_get_info()[0])
        e.close()
    assert min(used) <= 2096 * n + (6 << 20), (used, n)
    e = rf.MeshEngine(1 << 21)
    _same(e.MeshifyIndexed(small), rf.MeshEngine(1 << 21).MeshifyIndexed(small))
    _same(e.MeshifyIndexed(big), mesh)
    _same(e.MeshifyIndexed(small), rf.MeshEngine(1 << 21).MeshifyIndexed(small))
