"""What a user has the dense RGB-D path do, as cases that can be timed and
compared: every case makes its inputs from a seed (prepare), runs one pass
through the package's public entry points (run) and says what a pass cannot
do without (work).  The kinds of work:

inputs    a camera frame's images made ready for tracking: depth to metres,
          colour to intensity, the intensity and depth pyramids
track     one frame tracked against a model: its pyramids, the model's, the
          Gauss-Newton solve (Tracking::TrackRGBD without the volume)
raycast   a view of a volume rendered to a vertex map
fuse      a submap started over from a few posed depth images, then viewed
pipeline  consecutive frames of one camera, each ray-cast, tracked and fused
serve     several cameras' frames at once, through the server
batch     several submaps fused together from posed frames, each then viewed
mesh      marching cubes: the indexed mesh left on the device, or the
          triangle soup copied to the host

Volumes are the synthetic room (or, for large meshes, a wavy wall) seen by a
moving camera with sensor noise, as in the benchmark and the tests.

exact() restates the image operations and the tracker in 64 bits.  It has no
value for what a ray caster, a volume or a mesh returns: there single
comparisons of rounded numbers (a block's cell, a sample's voxel, a sign)
decide whether a pixel, a block or a triangle exists at all.
"""
import ctypes
import math
import os
import struct
import tempfile

import numpy as np
import torch

from yetanotherslam_amd import native, synth
from yetanotherslam_amd import rgbdfusion as rf
from yetanotherslam_amd import workloads

FORMATS = {"f32": rf.VOXEL_F32_F32, "f16": rf.VOXEL_F16_U16, "i16": rf.VOXEL_I16_U8}
MODES = {"depth": rf.TRACK_DEPTH, "rgb": rf.TRACK_RGB, "rgbd": rf.TRACK_RGBD}
ITERS = (10, 5, 3)
WEIGHTS = (0.1, 0.1, 1.0, 1.0)


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest calls: a thumbnail-sized frame's images, all launches
        {"name": "inputs 160x120", "kind": "inputs", "width": 160, "height": 120},
        # the benchmark's frame
        {"name": "inputs 640x480", "kind": "inputs", "width": 640, "height": 480},
        # geometry-only odometry at half resolution
        {"name": "track 320x240 depth", "kind": "track", "width": 320, "height": 240, "mode": "depth"},
        # the benchmark's tracker on one frame, called as FullSystem calls it
        {"name": "track 640x480 rgbd", "kind": "track", "width": 640, "height": 480, "mode": "rgbd"},
        # the model view that a frame is tracked against
        {"name": "raycast 640x480 5mm f32", "kind": "raycast", "width": 640, "height": 480, "voxel": 0.005,
         "format": "f32", "frames": 12},
        # a large view of a compact volume, for display
        {"name": "raycast 1280x960 5mm f16", "kind": "raycast", "width": 1280, "height": 960, "voxel": 0.005,
         "format": "f16", "frames": 8},
        # a keyframe's submap from the frames that follow it, at a size that is no multiple of a tile
        {"name": "fuse 633x475 5mm f32 x8", "kind": "fuse", "width": 633, "height": 475, "voxel": 0.005,
         "format": "f32", "frames": 8, "u16": True},
        # the headline: one camera, ICP and photometric, 5 mm, float storage
        {"name": "pipeline 640x480 5mm f32", "kind": "pipeline", "width": 640, "height": 480, "voxel": 0.005,
         "format": "f32", "mode": "rgbd", "chunk": 8},
        # a lighter robot: half resolution, coarser and compact volume, geometry only
        {"name": "pipeline 320x240 8mm f16", "kind": "pipeline", "width": 320, "height": 240, "voxel": 0.008,
         "format": "f16", "mode": "depth", "chunk": 8},
        # many cameras of two resolutions on one GPU
        {"name": "serve 12 mixed f32", "kind": "serve", "streams": 12, "width": 640, "height": 480, "mixed": True,
         "voxel": 0.005, "format": "f32", "rounds": 3},
        # an offline reconstruction's mesh, indexed, kept on the device for drawing
        {"name": "mesh indexed wall f32", "kind": "mesh", "form": "indexed", "wall": 3, "voxel": 0.005,
         "format": "f32", "width": 640, "height": 480, "frames": 0},
        # a submap's triangles for the viewer, on the host
        {"name": "mesh soup room i16", "kind": "mesh", "form": "soup", "wall": 0, "voxel": 0.01, "format": "i16",
         "width": 320, "height": 240, "frames": 3},
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _size(rng, lo, hi, step):
    """An image size between lo and hi pixels wide, in steps of `step` pixels, from square to wide."""
    w = max(step, int(round(_log_uniform(rng, lo, hi) / step)) * step)
    h = max(step, int(round(w * rng.uniform(0.55, 0.95) / step)) * step)
    return w, h


def draw(rng):
    kind = rng.choice(["inputs", "track", "track", "raycast", "raycast", "fuse", "fuse", "pipeline", "pipeline", "serve",
                       "batch", "mesh", "mesh"])
    voxel = round(rng.uniform(0.005, 0.012), 4)
    fmt = rng.choice(["f32", "f32", "f16", "i16"])
    mode = rng.choice(["depth", "rgb", "rgbd", "rgbd"])
    if kind == "inputs":
        w, h = _size(rng, 96, 1280, 4)
        return {"kind": kind, "width": w, "height": h}
    if kind == "track":
        w, h = _size(rng, 96, 960, 4)
        return {"kind": kind, "width": w, "height": h, "mode": mode}
    if kind == "raycast":
        w, h = _size(rng, 160, 1280, 8)
        return {"kind": kind, "width": w, "height": h, "voxel": voxel, "format": fmt, "frames": rng.randint(1, 12)}
    if kind == "fuse":
        w, h = _size(rng, 160, 800, 1)
        return {"kind": kind, "width": w, "height": h, "voxel": voxel, "format": fmt, "frames": rng.randint(1, 10),
                "u16": rng.random() < 0.5}
    if kind == "pipeline":
        w, h = _size(rng, 160, 640, 8)
        return {"kind": kind, "width": w, "height": h, "voxel": voxel, "format": fmt,
                "mode": rng.choice(["depth", "rgbd"]), "chunk": rng.randint(2, 8)}
    if kind == "serve":
        w, h = _size(rng, 160, 480, 16)
        return {"kind": kind, "streams": rng.randint(2, 12), "width": w, "height": h, "mixed": rng.random() < 0.5,
                "voxel": voxel, "format": fmt, "rounds": rng.randint(1, 3)}
    if kind == "batch":
        return {"kind": kind, "maps": rng.randint(2, 8), "steps": rng.randint(4, 12), "voxel": voxel, "format": fmt}
    form = rng.choice(["indexed", "soup"])
    if form == "soup":
        voxel = max(voxel, 0.008)
    return {"kind": "mesh", "form": form, "wall": rng.choice([0, 0, 1, 2]) if form == "indexed" else 0, "voxel": voxel,
            "format": fmt, "width": 640 if form == "indexed" else 320, "height": 480 if form == "indexed" else 240,
            "frames": rng.randint(1, 4)}


# ------------------------------------------------------------------ inputs
def _camera(w, h, seed, mode="rgbd"):
    """The room of this seed and a camera starting somewhere on its path.
    Tracking by geometry alone needs normals, so its sensor is filtered and
    its camera slower (3 mm a frame instead of 2 cm): on raw noisy depth
    hardly any pixel's normal is usable."""
    p = synth.params(width=w, height=h, seed=seed % 1000003, noise_seed=seed % 1000003 + 1,
                     theta0=(seed * 0.6180339887) % 1.0 * 2 * math.pi)
    if mode == "depth":
        p.noise_k, p.step = 0.0, 0.003
    return p


def _dev(a):
    if a.dtype == np.uint16:
        a = a.view(np.int16)
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _metres(depth_u16):
    return depth_u16.astype(np.float32) * np.float32(1.0 / 1000.0)


def _gray(rgb):
    c = rgb.astype(np.float32)
    return np.float32(0.299) * c[..., 0] + np.float32(0.587) * c[..., 1] + np.float32(0.114) * c[..., 2]


def _frames(p, n):
    return [synth.frame(p, t)[:2] for t in range(n)]


def _pow2(n):
    return 1 << max(10, math.ceil(math.log2(n)))


def _blocks(voxel, frames, w, h):
    """Pool for a volume of the room seen by `frames` frames: about 11000
    blocks in view at 5 mm, some more with each further frame."""
    per_view = 11000 * (0.005 / voxel) ** 2 * max(1.0, h / w / 0.75)
    return _pow2(per_view * (1.5 + 0.05 * frames) * 1.3)


def _map(p, case, nblocks):
    K = synth.intrinsics(p).astype(np.float32)
    return rf.MapStruct(K, 8 * nblocks, nblocks, case["voxel"], 4 * case["voxel"], voxel_format=FORMATS[case["format"]])


class _Device:
    """A device buffer of the library as an array that torch can take.  The
    tensor made of it holds this object, and with it the buffer's owner."""

    def __init__(self, owner, ptr, shape, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": kind, "data": (ptr, False), "version": 2}


def _view(owner, ptr, shape, kind="<f4"):
    if 0 in shape:
        return torch.zeros(shape, dtype=torch.float32 if kind == "<f4" else torch.int32, device="cuda")
    return torch.as_tensor(_Device(owner, ptr, shape, kind), device="cuda")


def _back_and_forth(i, n):
    """Frame i of a camera that goes along its n frames and back, again and again."""
    i %= 2 * (n - 1)
    return i if i < n else 2 * (n - 1) - i


def _tracker(p, w, h, mode="rgbd"):
    return rf.RGBDTracking(w, h, synth.intrinsics(p), len(ITERS), ITERS, MODES[mode], WEIGHTS)


def _prepare_inputs(case, seed):
    w, h = case["width"], case["height"]
    p = _camera(w, h, seed)
    d, c, _ = synth.frame(p, 0)
    s = {"depth": _dev(d), "rgb": _dev(c), "z": torch.empty((h, w), device="cuda"),
         "gray": torch.empty((h, w), device="cuda"), "trk": _tracker(p, w, h)}
    out = []
    for lvl in range(len(ITERS)):
        for which in (0, 2, 3, 4, 6):  # intensity, its gradients, inverse depth, vertices
            ptr, pitch, lw, lh = ctypes.c_void_p(), ctypes.c_size_t(), ctypes.c_int(), ctypes.c_int()
            native.call("yas_tracker_level", s["trk"].h, which, lvl, ctypes.byref(ptr), ctypes.byref(pitch),
                        ctypes.byref(lw), ctypes.byref(lh))
            out.append(_view(s["trk"], ptr.value, (lh.value, lw.value) + ((4,) if which == 6 else ())))
    s["levels"] = out
    return s


def _run_inputs(s):
    h, w = s["z"].shape
    ctx = s["trk"].ctx.h
    native.call("yas_depth_u16_to_f32", ctx, s["depth"].data_ptr(), 2 * w, s["z"].data_ptr(), 4 * w, w, h, 1000.0)
    native.call("yas_rgb_to_intensity", ctx, s["rgb"].data_ptr(), 3 * w, s["gray"].data_ptr(), 4 * w, w, h, 0)
    s["trk"].SetTrackingImage(s["gray"])
    s["trk"].SetTrackingDepth(s["z"])
    return [s["z"], s["gray"]] + s["levels"]


def _track_images(case, seed):
    """Two successive frames, and the smooth surface that a ray cast would
    give for the first one's camera, as a vertex map."""
    w, h = case["width"], case["height"]
    p = _camera(w, h, seed, case["mode"])
    (d0, c0), (d1, c1) = _frames(p, 2)
    q = _camera(w, h, seed, case["mode"])
    q.noise_k, q.dropout = 0.0, 0.0
    z = _metres(synth.frame(q, 0)[0])
    K = synth.intrinsics(p).astype(np.float32)
    u, v = np.meshgrid(np.arange(w, dtype=np.float32), np.arange(h, dtype=np.float32))
    ok = (z > 0.2) & (z < 3.0)
    vmap = np.stack([z * (u - K[2]) / K[0], z * (v - K[3]) / K[1], z, np.ones_like(z)], -1)
    vmap[~ok] = (0.0, 0.0, 0.0, -1.0)
    return p, _gray(c0), _metres(d0), _gray(c1), _metres(d1), vmap.astype(np.float32)


def _prepare_track(case, seed):
    p, g0, z0, g1, z1, vmap = _track_images(case, seed)
    trk = _tracker(p, case["width"], case["height"], case["mode"])
    s = {"trk": trk, "gray": _dev(g1), "z": _dev(z1), "model": _dev(vmap), "gray0": _dev(g0), "z0": _dev(z0)}
    trk.SetReferenceImage(s["gray0"])
    trk.SetReferenceDepth(s["z0"])
    return s


def _run_track(s):
    trk = s["trk"]
    trk.SetTrackingImage(s["gray"])
    trk.SetTrackingDepth(s["z"])
    trk.SetReferenceModel(s["model"])
    T, st = trk.GetTransform(swap=False)
    return [T, st.icp_inliers, st.rgb_inliers]


def _prepare_raycast(case, seed):
    w, h, n = case["width"], case["height"], case["frames"]
    p = _camera(w, h, seed)
    gt = synth.relative_poses(p, n + 1)
    m = _map(p, case, _blocks(case["voxel"], n, w, h))
    for t, (d, _) in enumerate(_frames(p, n)):
        m.FuseU16(_dev(d), gt[t])
    rc = rf.RayTraceEngine(w, h, synth.intrinsics(p))
    return {"map": m, "rc": rc, "T": gt[n], "out": _view(rc, rc.vmap_ptr()[0], (h, w, 4))}


def _run_raycast(s):
    s["rc"].RayTrace(s["map"], s["T"])
    return s["out"]


def _prepare_fuse(case, seed):
    w, h, n = case["width"], case["height"], case["frames"]
    p = _camera(w, h, seed)
    fr = [d for d, _ in _frames(p, n)]
    vw, vh = max(8, w // 2 // 8 * 8), max(8, h // 2 // 8 * 8)
    Kv = synth.intrinsics(p) * 0.5
    rc = rf.RayTraceEngine(vw, vh, Kv)
    return {"map": _map(p, case, _blocks(case["voxel"], n, w, h)), "rc": rc, "T": synth.relative_poses(p, n),
            "depth": [_dev(d if case["u16"] else _metres(d)) for d in fr], "u16": case["u16"],
            "out": _view(rc, rc.vmap_ptr()[0], (vh, vw, 4))}


def _run_fuse(s):
    m = s["map"]
    m.Reset()
    for d, T in zip(s["depth"], s["T"]):
        if s["u16"]:
            m.FuseU16(d, T)
        else:
            m.Fuse(d, T)
    s["rc"].RayTrace(m, s["T"][-1])
    return s["out"]


WARM = 4


def _prepare_pipeline(case, seed):
    w, h, n = case["width"], case["height"], WARM + case["chunk"]
    p = _camera(w, h, seed, case["mode"])
    nb = _blocks(case["voxel"], 2 * n, w, h)
    mp = rf.map_params(8 * nb, nb, case["voxel"], 4 * case["voxel"], FORMATS[case["format"]])
    pl = rf.DensePipeline(w, h, synth.intrinsics(p), mp, rf.tracker_params(len(ITERS), ITERS, MODES[case["mode"]], WEIGHTS))
    rc, ptr = ctypes.c_void_p(), ctypes.c_void_p()
    native.call("yas_pipeline_raycaster", pl.h, ctypes.byref(rc))
    native.call("yas_raycaster_vmap", rc, ctypes.byref(ptr), None)
    s = {"pl": pl, "fr": [(_dev(d), _dev(c)) for d, c in _frames(p, n)], "next": 0, "chunk": case["chunk"],
         "out": _view(pl, ptr.value, (h, w, 4))}
    for _ in range(WARM):
        pl.step(*s["fr"][s["next"]])
        s["next"] += 1
    return s


def _run_pipeline(s):
    """The camera's next frames: their poses, and the model view that the last one was tracked against."""
    pl, first = s["pl"], s["next"]
    for i in range(first, first + s["chunk"]):
        pl.step(*s["fr"][_back_and_forth(i, len(s["fr"]))])
    s["next"] = first + s["chunk"]
    got = [pl.pose(i) for i in range(first, first + s["chunk"])]
    return [np.stack([T for T, _ in got]), np.array([int(ok) for _, ok in got]), s["out"]]


def _prepare_serve(case, seed):
    w, h, n = case["width"], case["height"], case["streams"]
    small = (max(160, w // 2 // 8 * 8), max(120, h // 2 // 8 * 8))
    span = 8
    sv = rf.Server(w, h, n, rf.tracker_params(len(ITERS), ITERS, rf.TRACK_RGBD, WEIGHTS), FORMATS[case["format"]])
    fr, sid = {}, []
    for size in {(w, h), small if case["mixed"] else (w, h)}:
        p = _camera(*size, seed)
        fr[size] = [(_dev(d), _dev(c)) for d, c in _frames(p, span + n)]
    for i in range(n):
        size = small if case["mixed"] and i % 2 else (w, h)
        p = _camera(*size, seed)
        nb = _blocks(case["voxel"], 2 * span, *size)
        mp = rf.map_params(8 * nb, nb, case["voxel"], 4 * case["voxel"], FORMATS[case["format"]])
        sid.append((sv.add_stream(*size, synth.intrinsics(p), mp), size, i))
    sv.prepare()
    s = {"sv": sv, "fr": fr, "sid": sid, "span": span, "next": 0, "rounds": case["rounds"]}
    _run_serve(dict(s, rounds=2))
    s["next"] = 2
    return s


def _run_serve(s):
    sv, want = s["sv"], []
    for r in range(s["rounds"]):
        k = _back_and_forth(s["next"] + r, s["span"])
        for sid, size, start in s["sid"]:
            want.append(sv.submit(sid, *s["fr"][size][start + k]))
        sv.pump()
    s["next"] += s["rounds"]
    sv.drain()
    got = {r["request"]: r for r in sv.poll()}
    return [np.stack([got[q]["pose"] for q in want]), np.array([int(got[q]["tracked"]) for q in want])]


def _prepare_batch(case, seed):
    n, steps = case["maps"], case["steps"]
    maps, depth, poses, casters, outs = [], [[] for _ in range(steps)], [[] for _ in range(steps)], [], []
    seqs = {}
    for size in ((640, 480), (320, 240)):
        p = _camera(*size, seed)
        seqs[size] = (p, [_dev(d) for d, _ in _frames(p, steps + n)])
    for i in range(n):
        size = (640, 480) if (seed + i) % 2 else (320, 240)
        p, fr = seqs[size]
        maps.append(_map(p, case, _blocks(case["voxel"], steps, *size)))
        use = 2 + (seed // 7 + 5 * i) % (steps - 1)  # submaps of different lengths
        T0 = np.linalg.inv(synth.pose(p, i))
        for k in range(steps):
            depth[k].append(fr[i + k] if k < use else None)
            poses[k].append(T0 @ synth.pose(p, i + k))
        q = _camera(320, 240, seed)
        casters.append(rf.RayTraceEngine(320, 240, synth.intrinsics(q)))
        outs.append(_view(casters[-1], casters[-1].vmap_ptr()[0], (240, 320, 4)))
    b = rf.FusionBatch(maps)
    b.plan(depth, poses)
    return {"maps": maps, "batch": b, "casters": casters, "outs": outs, "T": np.eye(4)}


def _run_batch(s):
    for m in s["maps"]:
        m.Reset()
    s["batch"].run()
    for rc, m in zip(s["casters"], s["maps"]):
        rc.RayTrace(m, s["T"])
    return s["outs"]


def _sorted_volume(m):
    """The volume saved and read back with its blocks in order of their
    coordinates: the order in which a fused volume's blocks were allocated
    differs from run to run, and a mesh follows it."""
    fd, path = tempfile.mkstemp(suffix=".yasmap")
    os.close(fd)
    try:
        m.SaveToFile(path)
        raw = np.fromfile(path, np.uint8)
        n = struct.unpack_from("<i", raw, 24)[0]
        head, rec = raw[:224], raw[224:224 + 16 * n].view(np.int32).reshape(n, 4)
        vox = raw[224 + 16 * n:].reshape(n, -1)
        order = np.lexsort((rec[:, 2], rec[:, 1], rec[:, 0]))
        with open(path, "wb") as f:
            head.tofile(f)
            rec[order].tofile(f)
            vox[order].tofile(f)
        return rf.MapStruct.ReadFromFile(path)
    finally:
        os.unlink(path)


def _triangles(case):
    """About as many as the volume's mesh has: a wall's view holds 6400
    blocks at 5 mm, the room's 17000 and more, of some 105 triangles each."""
    blocks = 6600 * case["wall"] ** 2 if case["wall"] else 17000 + 800 * case["frames"]
    return 105 * blocks * (0.005 / case["voxel"]) ** 2


def _prepare_mesh(case, seed):
    w, h = case["width"], case["height"]
    p = _camera(w, h, seed)
    if case["wall"]:
        g, K = case["wall"], synth.intrinsics(p)
        nb = _pow2(9000 * g * g * (0.005 / case["voxel"]) ** 2)
        m = _map(p, case, nb)
        x0, y0 = (seed * 0.7548776662) % 1.0 * 50, (seed * 0.5698402910) % 1.0 * 50
        for i in range(g):
            for j in range(g):
                T = np.eye(4)
                T[0, 3], T[1, 3] = workloads.WALL_STEP[0] * i, workloads.WALL_STEP[1] * j
                m.Fuse(_dev(workloads.wavy_wall_depth(K, x0 + T[0, 3], y0 + T[1, 3], w, h)), T)
    else:
        gt = synth.relative_poses(p, case["frames"])
        nb = _blocks(case["voxel"], case["frames"], w, h)
        m = _map(p, case, nb)
        for t, (d, _) in enumerate(_frames(p, case["frames"])):
            m.FuseU16(_dev(d), gt[t])
    m, most = _sorted_volume(m), _pow2(1.3 * _triangles(case))
    s = {"map": m, "me": rf.MeshEngine(most), "form": case["form"], "n": (ctypes.c_int(), ctypes.c_int())}
    if case["form"] == "soup":
        s["host"] = [np.zeros((most, 9), np.float32), np.zeros((most, 9), np.float32)]
        s["blocks"] = [np.zeros((m.params.num_blocks,) + k, np.int32) for k in ((3,), (), ())]
        return s
    # the engine's buffers, empty: an extraction from an empty volume says where they are
    n, v, t = s["n"], ctypes.c_void_p(), ctypes.c_void_p()
    empty = rf.MapStruct(np.ones(4), 1024, 16, 0.01, 0.04)
    native.call("yas_mesh_extract_indexed", s["me"].h, empty.h, ctypes.byref(n[0]), ctypes.byref(n[1]))
    native.call("yas_mesher_indexed_device", s["me"].h, ctypes.byref(v), ctypes.byref(t))
    s["out"] = [_view(s["me"], v.value, (most, 3)).zero_(), _view(s["me"], t.value, (most, 3), "<i4").zero_()]
    empty.close()
    return s


def _run_mesh(s):
    """The mesh in buffers of the program's or the engine's own, zeros past its end, and how much of them it fills."""
    me, m, (n, k) = s["me"].h, s["map"].h, s["n"]
    if s["form"] == "indexed":
        native.call("yas_mesh_extract_indexed", me, m, ctypes.byref(n), ctypes.byref(k))
        return s["out"] + [n.value, k.value]
    native.call("yas_mesh_extract", me, m, ctypes.byref(n))
    native.call("yas_mesher_download", me, *(a.ctypes.data for a in s["host"]), n.value)
    native.call("yas_mesher_blocks", me, *(a.ctypes.data for a in s["blocks"]), None, len(s["blocks"][0]), ctypes.byref(k))
    return s["host"] + s["blocks"] + [n.value, k.value]


_PREPARE = {"inputs": _prepare_inputs, "track": _prepare_track, "raycast": _prepare_raycast, "fuse": _prepare_fuse,
            "pipeline": _prepare_pipeline, "serve": _prepare_serve, "batch": _prepare_batch, "mesh": _prepare_mesh}
_RUN = {"inputs": _run_inputs, "track": _run_track, "raycast": _run_raycast, "fuse": _run_fuse,
        "pipeline": _run_pipeline, "serve": _run_serve, "batch": _run_batch, "mesh": _run_mesh}


def prepare(case, seed):
    s = _PREPARE[case["kind"]](case, seed)
    s["kind"] = case["kind"]
    return s


def run(state):
    return _RUN[state["kind"]](state)


# ------------------------------------------------------------------ work
def work(case):
    """Each input read once and each output written once; volumes by the
    blocks in view (about 11000 at 5 mm, _blocks) and their voxels' bytes."""
    kind = case["kind"]
    w, h = case.get("width", 320), case.get("height", 240)
    n = w * h
    sv = 8 if case.get("format") == "f32" else 4
    view = 11000 * (0.005 / case.get("voxel", 0.005)) ** 2 * max(1.0, h / w / 0.75)
    levels = 1 + 1 / 4 + 1 / 16
    images = n * (2 + 3) + n * 8 + levels * n * (4 * 4 + 16)
    its = sum(it / 4 ** i for i, it in enumerate(ITERS))
    icp, rgb = case.get("mode", "rgbd") != "rgb", case.get("mode", "rgbd") != "depth"
    solve = its * n * ((48 if icp else 0) + (36 if rgb else 0))
    solve_f = its * n * ((150 if icp else 0) + (180 if rgb else 0))
    cast = view * (512 * sv + 16) + n * 16
    integrate = view * (512 * 2 * sv + 16) + n * 4
    if kind == "inputs":
        return {"bytes": images, "flops": n * 60}
    if kind == "track":
        return {"bytes": images + levels * n * 16 + solve, "flops": solve_f}
    if kind == "raycast":
        return {"bytes": cast, "flops": n * 300}
    if kind == "fuse":
        return {"bytes": case["frames"] * integrate + view * (512 * sv + 16) + n * 4, "flops": case["frames"] * view * 512 * 40}
    if kind == "pipeline":
        return {"bytes": case["chunk"] * (cast + images + solve + integrate),
                "flops": case["chunk"] * (solve_f + n * 300 + view * 512 * 40)}
    if kind == "serve":
        k = case["rounds"] * case["streams"] * (0.7 if case["mixed"] else 1.0)
        return {"bytes": k * (cast + images + solve + integrate), "flops": k * (solve_f + n * 300 + view * 512 * 40)}
    if kind == "batch":
        k = case["maps"] * case["steps"] * 0.5
        return {"bytes": k * integrate + case["maps"] * cast, "flops": k * view * 512 * 40}
    tri = _triangles(case)
    blocks = tri / 105
    return {"bytes": blocks * 729 * sv + tri * (12 + 6 if case["form"] == "indexed" else 72), "flops": blocks * 512 * 20}


# ------------------------------------------------------------------ 64 bits
def _pyr_gauss(a):
    """[1 4 6 4 1]/16 per axis at every second pixel, the border reflected about its pixel."""
    k = np.array([1.0, 4.0, 6.0, 4.0, 1.0]) / 16
    h, w = a.shape
    ry = [np.abs(2 * np.arange(h // 2) + i - 2) for i in range(5)]
    rx = [np.abs(2 * np.arange(w // 2) + i - 2) for i in range(5)]
    ry = [np.where(r >= h, 2 * h - 2 - r, r) for r in ry]
    rx = [np.where(r >= w, 2 * w - 2 - r, r) for r in rx]
    cols = sum(k[i] * a[ry[i]] for i in range(5))
    return sum(k[i] * cols[:, rx[i]] for i in range(5))


def _gradients(a):
    gx, gy = np.zeros_like(a), np.zeros_like(a)
    gx[1:-1, 1:-1] = (a[1:-1, 2:] - a[1:-1, :-2]) * 0.5
    gy[1:-1, 1:-1] = (a[2:, 1:-1] - a[:-2, 1:-1]) * 0.5
    return gx, gy


def _inverse(z):
    ok = (z > 0.2) & (z < 8.0)
    return np.where(ok, 1.0 / np.where(ok, z, 1.0), 0.0)


def _pyr_pick(a):
    """Every second pixel; the last row and column stay empty."""
    o = np.array(a[::2, ::2])
    o[-1], o[:, -1] = 0, 0
    return o


def _vertices(iv, K, cut=3.0):
    h, w = iv.shape
    z = 1.0 / np.where(iv > 0, iv, 1.0)
    ok = (iv > 0) & (z < cut)
    u, v = np.meshgrid(np.arange(w, dtype=np.float64), np.arange(h, dtype=np.float64))
    V = np.stack([z * (u - K[2]) / K[0], z * (v - K[3]) / K[1], z, np.ones_like(z)], -1)
    V[~ok] = (0.0, 0.0, 0.0, -1.0)
    return V


def _normals(V):
    N = np.zeros_like(V)
    N[..., 3] = -1.0
    a, b, c = V[:-1, :-1], V[:-1, 1:], V[1:, :-1]
    n = np.cross(c[..., :3] - a[..., :3], b[..., :3] - a[..., :3])
    q = np.linalg.norm(n, axis=-1, keepdims=True)
    ok = (a[..., 3] > 0) & (b[..., 3] > 0) & (c[..., 3] > 0)
    n = n / np.where(q > 0, q, 1.0)
    N[:-1, :-1][ok] = np.concatenate([n, np.ones_like(q)], -1)[ok]
    return N


def _exact_inputs(case, seed):
    p = _camera(case["width"], case["height"], seed)
    d, c, _ = synth.frame(p, 0)
    z = d.astype(np.float64) / 1000.0
    g = c.astype(np.float64) @ np.array([0.299, 0.587, 0.114])
    out, iv, K = [z, g], _inverse(z), synth.intrinsics(p)
    for lvl in range(len(ITERS)):
        if lvl:
            g, iv = _pyr_gauss(g), _pyr_pick(iv)
        gx, gy = _gradients(g)
        out += [g, gx, gy, iv, _vertices(iv, K / 2 ** lvl)]
    return out


def _bilinear(a, u, v):
    x, y = np.floor(u).astype(np.int64), np.floor(v).astype(np.int64)
    fx, fy = u - x, v - y
    return (a[y, x] * (1 - fx) + a[y, x + 1] * fx) * (1 - fy) + (a[y + 1, x] * (1 - fx) + a[y + 1, x + 1] * fx) * fy


def _se3_exp(xi):
    w = xi[3:]
    th = float(np.linalg.norm(w))
    W = np.array([[0, -w[2], w[1]], [w[2], 0, -w[0]], [-w[1], w[0], 0]])
    if th < 1e-8:
        A, B, C = 1.0, 0.5, 1.0 / 6.0
    else:
        A, B, C = math.sin(th) / th, (1 - math.cos(th)) / th ** 2, (th - math.sin(th)) / th ** 3
    T = np.eye(4)
    T[:3, :3] += A * W + B * W @ W
    T[:3, 3] = (np.eye(3) + B * W + C * W @ W) @ xi[:3]
    return T


def _icp_system(T, V0, N0, V1, N1, K):
    h, w = V0.shape[:2]
    ok = (V0[..., 3] > 0) & (N0[..., 3] > 0)
    p = V0[ok][:, :3] @ T[:3, :3].T + T[:3, 3]
    n = N0[ok][:, :3] @ T[:3, :3].T
    with np.errstate(all="ignore"):
        u = np.floor(K[0] * p[:, 0] / p[:, 2] + K[2] + 0.5)
        v = np.floor(K[1] * p[:, 1] / p[:, 2] + K[3] + 0.5)
    inside = (u >= 0) & (v >= 0) & (u < w) & (v < h)
    p, n, u, v = p[inside], n[inside], u[inside].astype(np.int64), v[inside].astype(np.int64)
    q, m = V1[v, u], N1[v, u]
    ok = (q[:, 3] > 0) & (m[:, 3] > 0) & (np.linalg.norm(p - q[:, :3], axis=1) <= 0.01)
    ok &= np.linalg.norm(np.cross(n, m[:, :3]), axis=1) < math.sin(math.radians(20.0))
    p, n, q = p[ok], n[ok], q[ok][:, :3]
    return np.concatenate([n, np.cross(p, n), np.sum(n * (q - p), axis=1, keepdims=True)], 1)


def _photometric_system(T, iv, g0, g1, gx, gy, K):
    h, w = iv.shape
    y, x = np.nonzero(iv > 0)
    z = 1.0 / iv[y, x]
    p = np.stack([z * (x - K[2]) / K[0], z * (y - K[3]) / K[1], z], 1) @ T[:3, :3].T + T[:3, 3]
    with np.errstate(all="ignore"):
        u, v = K[0] * p[:, 0] / p[:, 2] + K[2], K[1] * p[:, 1] / p[:, 2] + K[3]
    inside = (u > 0) & (v > 0) & (u < w - 1) & (v < h - 1)
    p, u, v, ref = p[inside], u[inside], v[inside], g0[y, x][inside]
    r, a, b = _bilinear(g1, u, v) - ref, _bilinear(gx, u, v), _bilinear(gy, u, v)
    ok = a * a + b * b > 0
    p, r, a, b = p[ok], r[ok], a[ok], b[ok]
    th = 4.685 * math.sqrt(np.sum((r - r.mean()) ** 2) / (len(r) - 1))
    wt = np.where(np.abs(r) > th, th / np.maximum(np.abs(r), 1e-300), 1.0)
    j0, j1 = a * K[0] / p[:, 2], b * K[1] / p[:, 2]
    j2 = -(j0 * p[:, 0] + j1 * p[:, 1]) / p[:, 2]
    J = np.stack([j0, j1, j2, j2 * p[:, 1] - b * K[1], -j2 * p[:, 0] + a * K[0], -j0 * p[:, 1] + j1 * p[:, 0], -r], 1)
    return J, wt


def _exact_track(case, seed):
    p, g0, z0, g1, z1, vmap = _track_images(case, seed)
    K, mode = synth.intrinsics(p), case["mode"]
    g0, g1, iv0, iv1, V0 = (g0.astype(np.float64), g1.astype(np.float64), _inverse(z0.astype(np.float64)),
                            _inverse(z1.astype(np.float64)), vmap.astype(np.float64))
    pyr = []
    for lvl in range(len(ITERS)):
        if lvl:
            g0, g1, iv0, iv1, V0 = _pyr_gauss(g0), _pyr_gauss(g1), _pyr_pick(iv0), _pyr_pick(iv1), _pyr_pick(V0)
            V0[-1, :, 3], V0[:, -1, 3] = -1, -1
        V1 = _vertices(iv1, K / 2 ** lvl)
        pyr.append((V0, _normals(V0), V1, _normals(V1), iv0, g0, g1) + _gradients(g1))
    T = np.eye(4)
    best = T.copy()
    for lvl in range(len(ITERS) - 1, -1, -1):
        V0, N0, V1, N1, iv, a0, a1, gx, gy = pyr[lvl]
        last = math.inf
        for _ in range(ITERS[lvl]):
            H, b, err, count = np.zeros((6, 6)), np.zeros(6), 0.0, 0.0
            if mode != "depth":
                J, wt = _photometric_system(T, iv, a0, a1, gx, gy, K / 2 ** lvl)
                S = (J * wt[:, None]).T @ J
                f = WEIGHTS[0] if mode == "rgbd" else 1.0
                H, b, err, count = H + f * S[:6, :6], b + f * S[:6, 6], S[6, 6], len(J)
            if mode != "rgb":
                J = _icp_system(T, V0, N0, V1, N1, K / 2 ** lvl)
                S = J.T @ J
                f = WEIGHTS[2] if mode == "rgbd" else 1.0
                H, b, err = H + f * S[:6, :6], b + f * S[:6, 6], S[6, 6]
            err = math.sqrt(err) / (count + 6)
            if H.any():
                T = _se3_exp(np.linalg.solve(H, b)) @ T
            if err < last:
                best, last = T.copy(), err
    return [best, None, None]


def exact(case, seed):
    if case["kind"] == "inputs":
        return _exact_inputs(case, seed)
    if case["kind"] == "track":
        return _exact_track(case, seed)
    return None
