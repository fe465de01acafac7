"""Every pyramid level formed in one launch equals the levels formed one by
one with the stand-alone image operations, bit for bit: one to five levels,
sizes with whole and partial tiles, padded rows, and the pipeline's form that
reads the camera's images."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ops(torch, w, h, levels, gray, z, K):
    """Levels by the stand-alone entry points: (intensity, gx, gy, inverse depth, vertices) per level."""
    from yetanotherslam_amd import rgbdfusion as rf
    from yetanotherslam_amd.native import call
    ctx = rf.default_context().h
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    out = []
    g = gray.contiguous()
    inv = torch.zeros((h, w), device="cuda")
    call("yas_depth_to_invdepth", ctx, p(z), z.stride(0) * 4, p(inv), 4 * w, w, h)
    for l in range(levels):
        if l:
            w2, h2 = w // 2, h // 2
            g2 = torch.zeros((h2, w2), device="cuda")
            call("yas_pyrdown_gauss", ctx, p(g), 4 * w, w, h, p(g2), 4 * w2)
            i2 = torch.zeros((h2, w2), device="cuda")
            call("yas_pyrdown_depth", ctx, p(inv), 4 * w, p(i2), 4 * w2, w2, h2)
            w, h, g, inv = w2, h2, g2, i2
        gx, gy = torch.zeros((h, w), device="cuda"), torch.zeros((h, w), device="cuda")
        call("yas_image_gradient", ctx, p(g), 4 * w, p(gx), p(gy), 4 * w, w, h)
        v = torch.zeros((h, w, 4), device="cuda")
        Kl = (np.asarray(K, np.float64) / (1 << l)).astype(np.float32)
        call("yas_compute_vertex_map", ctx, p(inv), 4 * w, p(v), 16 * w, w, h, Kl.ctypes.data_as(ctypes.c_void_p), 3.0)
        nrm = torch.zeros((h, w, 4), device="cuda")
        call("yas_compute_normal_map", ctx, p(v), 16 * w, p(nrm), 16 * w, w, h)
        out.append([a.cpu().numpy() for a in (g, gx, gy, inv, v, nrm)])
    return out


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


@pytest.mark.parametrize("w,h,levels", [(32, 32, 1), (36, 28, 2), (68, 60, 3), (128, 96, 4), (176, 80, 5), (324, 244, 3)])
def test_levels_equal_the_separate_operations(gpu, w, h, levels):
    import torch
    from yetanotherslam_amd import rgbdfusion as rf
    rng = np.random.default_rng(w * 1000 + h)
    gray = torch.from_numpy((rng.random((h, w + 8)) * 255).astype(np.float32)).cuda()[:, :w]
    zn = (0.1 + 4.0 * rng.random((h, w + 4))).astype(np.float32)
    zn[rng.random(zn.shape) < 0.1] = 0.0
    zn[3, 5] = np.nan
    z = torch.from_numpy(zn).cuda()[:, :w]
    K = np.array([0.8 * w, 0.82 * w, w / 2 - 0.5, h / 2 - 0.5], np.float32).astype(np.float64)
    t = rf.RGBDTracking(w, h, K, levels, [2] * levels, rf.TRACK_RGBD)
    t.SetTrackingImage(gray)
    t.SetTrackingDepth(z)
    t.SetReferenceImage(gray)
    t.SetReferenceDepth(z)
    want = _ops(torch, w, h, levels, gray, z, K)
    for l in range(levels):
        for which, ref in ((0, 0), (1, 0), (2, 1), (3, 2), (4, 3), (5, 3), (6, 4), (8, 4), (7, 5), (9, 5)):
            assert np.array_equal(_bits(t.level(which, l)), _bits(want[l][ref])), (l, which)
    # a model: level l holds every 2^l-th vertex, its last row and column empty
    vmap = torch.from_numpy(want[0][4]).cuda()
    t.SetReferenceModel(vmap)
    v = want[0][4]
    for l in range(levels):
        if l:
            v = v[::2, ::2].copy()
            v[-1], v[:, -1] = (0, 0, 0, -1), (0, 0, 0, -1)
        assert np.array_equal(_bits(t.level(8, l)), _bits(v)), l


@pytest.mark.parametrize("levels,gray_mode", [(3, 0), (3, 1), (5, 0)])
def test_pipeline_levels_equal_the_tracker_s(gpu, levels, gray_mode):
    import torch
    from yetanotherslam_amd import rgbdfusion as rf
    from yetanotherslam_amd import synth
    w, h = 176, 144
    p = synth.params(width=w, height=h, theta0=0.7)
    K = synth.intrinsics(p)
    fr = [synth.frame(p, t)[:2] for t in range(2)]
    pl = rf.DensePipeline(w, h, K, rf.map_params(1 << 14, 1 << 13, 0.01, 0.04),
                          rf.tracker_params(levels, [2] * levels, rf.TRACK_RGBD), gray_mode=gray_mode)
    dev = [(torch.from_numpy(d.view(np.int16)).cuda(), torch.from_numpy(c).cuda()) for d, c in fr]
    for d, c in dev:
        pl.step(d, c)
    # after the step the frame's levels are the reference ones
    ctx = rf.default_context().h
    z, g = torch.empty((h, w), device="cuda"), torch.empty((h, w), device="cuda")
    rf.call("yas_depth_u16_to_f32", ctx, dev[1][0].data_ptr(), 2 * w, z.data_ptr(), 4 * w, w, h, 1000.0)
    rf.call("yas_rgb_to_intensity", ctx, dev[1][1].data_ptr(), 3 * w, g.data_ptr(), 4 * w, w, h, gray_mode)
    K32 = np.asarray(K, np.float32).astype(np.float64)
    t = rf.RGBDTracking(w, h, K32, levels, [2] * levels, rf.TRACK_RGBD)
    t.SetTrackingImage(g)
    t.SetTrackingDepth(z)
    for l in range(levels):
        for mine, theirs in ((0, 1), (2, 2), (3, 3), (4, 5), (6, 8)):
            assert np.array_equal(_bits(t.level(mine, l)), _bits(pl.tracker_level(theirs, l))), (l, mine)
