"""The work a user of this package has it do, as cases that can be timed and
checked: rendering, training steps, densification and mesh extraction through
the engine's Python entry points (msplat._engine, msplat.device), from the
smallest frame to the 3M-splat training step.

listed() are fixed cases, draw(rng) draws others from the same ranges,
prepare / run are one user's program split into what it keeps and one pass,
work / tolerance say what a pass cannot do without and how far two correct
implementations may be apart, and exact() is the pass in 64 bits, written in
plain torch from the mathematics.

Scenes are synthetic: "blobs" (64 isotropic clusters in [-2, 2]^3), "cube"
(uniform in [-1, 1]^3) and "ball" (40% of the splats in a 0.1-radius ball on
the optical axis: very long tile lists).  Cameras orbit the origin.
"""
from __future__ import annotations

import ctypes as C
import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parents[1] / "msplat-ios_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from msplat import _engine as E  # noqa: E402
from msplat import device as D  # noqa: E402
from msplat import synthetic as S  # noqa: E402

DEV = "cuda:0"
# Every learning rate at the end of a schedule that decayed it a
# hundredfold: however many passes are run, the scene stays the one the case
# describes.
LR_SCALE = 0.01
TRAIN_CAMERAS = 4
CUTOFF_COST = 60e6  # most tile intersections exact() takes on (0.2 us each)


def listed() -> list[dict]:
    return [
        # the smallest call: a thumbnail-sized preview of a small scene
        # without view dependence; launches and latency
        _case("render", "render-16k-256x256", "cube", 16384, 256, 256, 0, -4.0, 0.5),
        # one frame of a viewer whose image stays on the GPU, the size a
        # quarter-resolution capture is trained at
        _case("render", "render-500k-1297x840", "blobs", 500_000, 1297, 840, 3, -4.0, 0.5),
        # one viewer frame brought to host memory as RGBA8
        # (renderFromPoseToBuffer)
        _case("frame", "frame-500k-1920x1080", "blobs", 500_000, 1920, 1080, 3, -4.3, 0.5),
        # the depth, normal, alpha and median maps that mesh and point-cloud
        # export read
        _case("maps", "maps-200k-1297x840", "blobs", 200_000, 1297, 840, 3, -4.0, 0.5),
        # the start of a training run: 1/4-resolution images (the resolution
        # schedule's first level), SH degree 1 active
        _case("train", "train-100k-324x210", "blobs", 100_000, 324, 210, 3, -4.0, 0.5, active=1),
        # the ordinary training step
        _case("train", "train-500k-1297x840", "blobs", 500_000, 1297, 840, 3, -4.0, 0.5),
        # the largest: full-resolution photographs, a scene at its densest
        _case("train", "train-3M-5187x3361", "blobs", 3_000_000, 5187, 3361, 3, -5.0, 0.7),
        # a scene with a dense core: tile lists of up to ~200k entries
        _case("train", "train-ball-1M-1920x1080", "ball", 1_000_000, 1920, 1080, 3, -4.5, 0.5),
        # a program with its own optimizer: per-group gradients, with the
        # distortion regulariser (full outputs in both directions)
        _case("grads", "grads-200k-989x657", "blobs", 200_000, 989, 657, 3, -4.0, 0.5),
        # the 3DGS mode's training step
        _case("train3d", "train3d-500k-1297x840", "blobs", 500_000, 1297, 840, 3, -4.0, 0.5),
        # one densification: classify, append, cull, compact
        dict(name="densify-300k", kind="densify", n=300_000),
        # mesh extraction at the fine setting: 32 depth maps into 300^3
        # voxels of 2 mm, then marching cubes
        dict(name="mesh-300-32x1297x840", kind="mesh", dim=300, views=32, w=1297, h=840),
    ]


def _case(kind, name, scene, n, w, h, degree, mean, std, active=None):
    return dict(name=name, kind=kind, scene=scene, n=n, w=w, h=h, degree=degree, mean=mean, std=std,
                active=degree if active is None else active)


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["render", "render", "frame", "maps", "train", "train", "train", "grads", "train3d", "densify",
                       "mesh"])
    if kind == "densify":
        return dict(kind=kind, n=_log_int(rng, 2_000, 1_500_000))
    if kind == "mesh":
        return dict(kind=kind, dim=_log_int(rng, 40, 300), views=_log_int(rng, 1, 32), w=_log_int(rng, 160, 1920),
                    h=_log_int(rng, 120, 1080))
    while True:
        n = _log_int(rng, 2_000, 2_000_000)
        w = _log_int(rng, 97, 4100)
        h = max(64, int(w * rng.uniform(0.5, 1.2)))
        scene = rng.choice(["blobs", "blobs", "blobs", "cube", "ball"])
        std = round(rng.uniform(0.4, 0.7), 3)
        # splats of a few to a few dozen pixels at any resolution
        mean = round(-4.0 - 0.72 * math.log(max(w, 300) / 1297.0) + rng.uniform(-0.4, 0.3), 3)
        degree = rng.choice([0, 1, 2, 3, 3, 3])
        active = rng.randint(0, degree)
        if scene == "ball" and (n > 1_000_000 or w > 2000):
            continue
        c = dict(kind=kind, scene=scene, n=n, w=w, h=h, degree=degree, mean=mean, std=std, active=active)
        if _intersections(c) < 40e6:
            return c


def _intersections(c) -> float:
    """About the tile intersections of one frame."""
    sigma = math.exp(c["mean"] + 0.5 * c["std"]) * c["w"] / 4.0
    return 0.85 * c["n"] * min((6.0 * sigma + 1.0) / 16.0 + 1.0, c["w"] / 16.0) ** 2


# ---- inputs -----------------------------------------------------------------
def _gen(seed: int):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 2 + 1)
    return g


def _host_inputs(case, seed):
    """The splats (float32, in the package's group order) and the cameras."""
    g = _gen(seed)
    n, deg = case["n"], case["degree"]
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    uni = lambda *s: torch.rand(*s, device=DEV, generator=g)  # noqa: E731
    if case["scene"] == "cube":
        means = 2 * uni(n, 3) - 1
    elif case["scene"] == "ball":
        nb = int(0.4 * n)
        d = rnd(nb, 3)
        d = d / d.norm(dim=1, keepdim=True) * (0.1 * uni(nb, 1) ** (1 / 3))
        means = torch.cat([d, 4 * uni(n - nb, 3) - 2])
    else:
        centres = 4 * uni(64, 3) - 2
        means = centres[torch.randint(64, (n,), device=DEV, generator=g)] + 0.3 * rnd(n, 3)
    scales = case["mean"] + case["std"] * rnd(n, 3 if case["kind"] == "train3d" else 2)
    quats = rnd(n, 4)
    quats = quats / quats.norm(dim=1, keepdim=True)
    fdc = (uni(n, 3) - 0.5) / S.SH_C0
    frest = 0.05 * rnd(n, (deg + 1) ** 2 - 1, 3)
    opac = rnd(n, 1)
    params = [t.float().contiguous().cpu().numpy() for t in (means, scales, quats, fdc, frest, opac)]
    az = float(uni(1)) * 2 * math.pi
    cams = []
    for k in range(TRAIN_CAMERAS):
        a, el = az + 2 * math.pi * k / TRAIN_CAMERAS, math.radians(20.0)
        r = 3.0 if case["scene"] == "cube" else 4.0
        eye = (r * math.cos(el) * math.cos(a), r * math.sin(el), r * math.cos(el) * math.sin(a))
        cams.append(S.Camera(S.look_at(eye), float(case["w"]), float(case["w"]), case["w"] / 2.0, case["h"] / 2.0,
                             case["w"], case["h"]))
    return params, cams


def _photo(case, seed, k):
    """A photograph-like target [H, W, 3]: smooth colour fields with some
    fine texture."""
    g = _gen(1_000_003 * (k + 1) + seed)
    h, w = case["h"], case["w"]
    low = torch.rand(1, 3, max(2, h // 48), max(2, w // 48), device=DEV, generator=g)
    img = torch.nn.functional.interpolate(low, size=(h, w), mode="bilinear", align_corners=True)[0]
    img = img + 0.03 * torch.randn(3, h, w, device=DEV, generator=g)
    return img.clamp(0, 1).permute(1, 2, 0).contiguous()


def _to_engine(t):
    """A device copy of a torch tensor in the engine's memory."""
    t = t.contiguous()
    torch.cuda.synchronize()
    d = E.DeviceArray(tuple(t.shape), np.dtype(str(t.dtype).replace("torch.", "")))
    E.check(E.lib().msplat_hip_copy(d.ptr, t.data_ptr(), d.nbytes))
    E.sync()
    return d


class _View:
    """Device memory of the engine as torch sees it.  torch keeps this object
    for as long as the tensor lives, so `owner`, the DeviceArray the memory
    belongs to (None: a buffer of the engine's own), outlives every view."""

    def __init__(self, ptr, shape, kind, owner):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=kind, data=(ptr, False), version=2)


def _tensor(st, ptr, shape, kind="<f4", owner=None):
    """A torch view of engine memory (kept: a program wraps a buffer once)."""
    key = (ptr, tuple(shape), kind)
    t = st["views"].get(key)
    if t is None:
        if len(st["views"]) > 256:
            st["views"].clear()
        if 0 in key[1]:
            t = torch.empty(shape, device=DEV, dtype=torch.int32 if kind == "<i4" else torch.float32)
        else:
            t = torch.as_tensor(_View(ptr, shape, kind, owner), device=DEV)
        st["views"][key] = t
    return t


def _last(st, name, shape, kind="<f4"):
    ptr, _ = E.last_ptr(name)
    return _tensor(st, ptr, shape, kind)


def _arr(st, a):
    return _tensor(st, a.ptr, a.shape, owner=a)


def prepare(case, seed):
    E.init()
    kind = case["kind"]
    st = dict(case=case, views={})
    if kind == "mesh":
        st.update(_mesh_inputs(case, seed))
    elif kind == "densify":
        st.update(_densify_state(case, seed))
    else:
        params, cams = _host_inputs(case, seed)
        scene = S.Scene(params[0], params[1], params[2], params[5], params[3], params[4], case["degree"], cams)
        ds = D.DeviceScene3D.from_scene(scene) if kind == "train3d" else D.DeviceScene(scene)
        ds.lr = [LR_SCALE * x for x in D.LR_INIT]
        st.update(ds=ds, cams=[ds.camera(c, case["active"]) for c in cams], at=0)
        if kind in ("train", "train3d", "grads"):
            st["gts"] = [_to_engine(_photo(case, seed, k)) for k in range(TRAIN_CAMERAS if kind != "grads" else 1)]
        if kind == "frame":
            st["rgba"] = np.zeros((case["h"], case["w"], 4), np.uint8)
    E.sync()
    torch.cuda.synchronize()
    return st


def _densify_inputs(case, seed):
    """Splats after a training interval: the six groups, both Adam moments and
    the statistics of 100 steps, most splats seen.  A quarter is split (large
    and of high gradient), an eighth duplicated (small and of high gradient),
    and a tenth of each part culled by its opacity."""
    g = _gen(seed)
    n = case["n"]
    c = dict(kind="densify", scene="blobs", n=n, w=1297, h=840, degree=3, mean=-4.6, std=0.5)
    params, _ = _host_inputs(c, seed)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g).cpu().numpy()  # noqa: E731
    m = [1e-6 * rnd(*p.shape) for p in params]
    v = [(1e-6 * rnd(*p.shape)) ** 2 for p in params]
    vis = torch.randint(1, 60, (n,), device=DEV, generator=g).float().cpu().numpy()
    perm = torch.randperm(n, device=DEV, generator=g).cpu().numpy()
    split, dup, rest = np.split(perm, [n // 4, n // 4 + n // 8])
    high = np.zeros(n, bool)
    high[split] = high[dup] = True
    mag = np.exp(np.minimum(np.abs(rnd(n)), 4.0))
    grad = (vis * np.where(high, 0.00021 * mag, 0.00019 / mag) / 648.5).astype(np.float32)
    vis[rest[: len(rest) // 20]] = 0.0
    size = np.abs(params[1] + 4.6)
    params[1] = -4.62 - size
    params[1][split, 0] += 2 * size[split, 0] + 0.03
    params[1] = params[1].astype(np.float32)
    max2d = np.minimum(np.exp(0.7 * rnd(n) - 4.5), 0.049).astype(np.float32)
    op = np.abs(params[5]) - 2.1
    for part in (split, dup, rest):
        op[part[: len(part) // 10]] = -2.3 - np.abs(params[5][part[: len(part) // 10]])
    params[5] = op.astype(np.float32)
    noise = rnd(2 * n, 3)
    return params, m, v, grad, vis, max2d, noise


def _densify_state(case, seed):
    params, m, v, grad, vis, max2d, noise = _densify_inputs(case, seed)
    n = case["n"]
    scene = S.Scene(params[0], params[1], params[2], params[5], params[3], params[4], 3)
    ds = D.CapacityScene(scene, 4 * n)
    for dst, src in ((ds.exp_avg, m), (ds.exp_avg_sq, v)):
        for a, x in zip(dst, src):
            E.check(E.lib().msplat_hip_upload(a.ptr, np.ascontiguousarray(x, np.float32).ctypes.data, x.size * 4))
    for a, x in ((ds.grad_norm, grad), (ds.vis, vis), (ds.max2d, max2d)):
        E.check(E.lib().msplat_hip_upload(a.ptr, x.ctypes.data, x.nbytes))
    ds.stage_samples(noise)
    kept = [E.DeviceArray.from_numpy(np.ascontiguousarray(x, np.float32)) for x in params + m + v]
    return dict(ds=ds, kept=kept)


def _mesh_cameras(case, seed):
    """Cameras on a sphere of radius 1 around an object of radius ~0.2."""
    w, cams = case["w"], []
    for k in range(case["views"]):
        z = 1 - 2 * (k + 0.5) / case["views"]
        phi = k * math.pi * (3 - math.sqrt(5)) + 0.1 * (seed % 61)
        eye = np.array([math.sqrt(1 - z * z) * math.cos(phi), math.sqrt(1 - z * z) * math.sin(phi), z])
        up = np.array([0.0, 0.0, 1.0]) if abs(z) < 0.9 else np.array([1.0, 0.0, 0.0])
        right = np.cross(-eye, up)
        right /= np.linalg.norm(right)
        R = np.stack([right, np.cross(-eye, right), -eye])
        vm = np.eye(4)
        vm[:3, :3] = R
        vm[:3, 3] = -R @ eye
        cams.append((vm.astype(np.float32), np.float32(1.35 * w), np.float32(1.35 * w), np.float32(w / 2),
                     np.float32(case["h"] / 2)))
    return cams


def _mesh_maps(case, seed):
    """Per view the depth and alpha a render of a slightly bumpy opaque ball
    gives (0 and 0 outside it)."""
    h, w = case["h"], case["w"]
    g = _gen(seed)
    radius = 0.17 + 0.06 * float(torch.rand(1, device=DEV, generator=g))
    maps = []
    for vm, fx, fy, cx, cy in _mesh_cameras(case, seed):
        m = torch.tensor(vm, device=DEV, dtype=torch.float64)
        u = (torch.arange(w, device=DEV, dtype=torch.float64) + 0.5 - float(cx)) / float(fx)
        v = (torch.arange(h, device=DEV, dtype=torch.float64) + 0.5 - float(cy)) / float(fy)
        d = torch.stack([u[None].expand(h, w), v[:, None].expand(h, w), torch.ones(h, w, device=DEV).double()], -1)
        d = d @ m[:3, :3]
        eye = -(m[:3, :3].T @ m[:3, 3])
        a, b, c = (d * d).sum(-1), 2 * (d @ eye), float(eye @ eye) - radius * radius
        disc = b * b - 4 * a * c
        hit = disc >= 0
        depth = torch.where(hit, (-b - disc.clamp(min=0).sqrt()) / (2 * a), torch.zeros_like(a))
        depth = depth + torch.where(hit, 0.0005 * torch.randn(h, w, device=DEV, generator=g).double(), 0.0)
        alpha = torch.where(hit, 0.9 + 0.1 * torch.rand(h, w, device=DEV, generator=g).double(), 0.0)
        maps.append((depth.float(), alpha.float()))
    return maps


def _mesh_grid(case):
    """Voxel size and origin: the object and a margin fill the grid."""
    return 0.6 / case["dim"], [-0.3, -0.3, -0.3]


def _mesh_inputs(case, seed):
    dim = case["dim"]
    vs, origin = _mesh_grid(case)
    views = [cam + (_to_engine(d), _to_engine(a)) for cam, (d, a) in zip(_mesh_cameras(case, seed),
                                                                        _mesh_maps(case, seed))]
    most = 12 * dim * dim
    return dict(grid=E.DeviceArray((dim, dim, dim, 2)), tris=E.DeviceArray.zeros((most, 9)), most=most,
                mesh_views=views, vs=vs, origin=origin)


# ---- one pass ---------------------------------------------------------------
def run(st):
    return _RUN[st["case"]["kind"]](st)


def _render_frame(st):
    ds, n = st["ds"], C.c_int64()
    E.check(E.lib().msplat_hip_render(C.byref(st["cams"][0]), C.byref(ds.gaussians), ds.background.ptr, C.byref(n)))


def _run_render(st):
    _render_frame(st)
    return dict(image=_last(st, "out_img", (st["case"]["h"], st["case"]["w"], 3)))


def _run_frame(st):
    _render_frame(st)
    ptr, numel = E.last_ptr("out_img")
    E.check(E.lib().msplat_hip_image_to_rgba8(ptr, numel // 3, st["rgba"].ctypes.data))
    return dict(rgba=st["rgba"])


def _run_maps(st):
    h, w = st["case"]["h"], st["case"]["w"]
    _render_frame(st)
    return dict(image=_last(st, "out_img", (h, w, 3)), depth=_last(st, "out_depth", (h, w)),
                normal=_last(st, "out_normal", (h, w, 3)), alpha=_last(st, "out_alpha", (h, w)),
                median=_last(st, "out_median_depth", (h, w)))


def _run_train(st):
    ds, k = st["ds"], st["at"]
    st["at"] = (k + 1) % TRAIN_CAMERAS
    step = D.train_step3d if st["case"]["kind"] == "train3d" else D.train_step
    loss, _ = step(ds, st["cams"][k], st["gts"][k])
    out = dict(loss=loss, image=_last(st, "out_img", (st["case"]["h"], st["case"]["w"], 3)),
               grad_norm=_arr(st, ds.grad_norm), vis=_arr(st, ds.vis), max2d=_arr(st, ds.max2d))
    for name, p, m in zip(D.GROUPS, ds.params, ds.exp_avg):
        out[name], out["m_" + name] = _arr(st, p), _arr(st, m)
    return out


_GRADS = (("means", "dL_dmean3D"), ("scales", "dL_dscale"), ("quats", "dL_dquat"), ("features_dc", "dL_dfeatures_dc"),
          ("features_rest", "dL_dfeatures_rest"), ("opacities", "dL_dopacity"))


def _run_grads(st):
    ds, case = st["ds"], st["case"]
    loss, n = C.c_float(), C.c_int64()
    inv = float(np.float32(1.0) / np.float32(max(case["w"], case["h"])))
    for a in (ds.grad_norm, ds.vis, ds.max2d):
        a.zero_()
    E.check(E.lib().msplat_hip_train_step(
        C.byref(st["cams"][0]), C.byref(ds.gaussians), ds.background.ptr, st["gts"][0].ptr, 0.8, LAMBDA_DIST, 0.2,
        ds.grad_norm.ptr, ds.vis.ptr, ds.max2d.ptr, inv, None, C.byref(loss), C.byref(n)))
    out = dict(loss=float(loss.value), image=_last(st, "out_img", (case["h"], case["w"], 3)),
               distortion=_last(st, "out_distortion", (case["h"], case["w"])), grad_norm=_arr(st, ds.grad_norm),
               vis=_arr(st, ds.vis), max2d=_arr(st, ds.max2d))
    for (name, buf), p in zip(_GRADS, ds.params):
        out["d_" + name] = _last(st, buf, p.shape)
    return out


def _run_densify(st):
    ds, n = st["ds"], st["case"]["n"]
    # the splats of the training interval, back in the trainer's buffers
    for dst, src in zip(ds.params + ds.exp_avg + ds.exp_avg_sq, st["kept"]):
        E.check(E.lib().msplat_hip_copy(dst.ptr, src.ptr, src.nbytes))
    ds.n = n
    new = ds.densify(None, 648.5)
    out = dict(count=new)
    for k, bufs in (("", ds.params), ("m_", ds.exp_avg), ("v_", ds.exp_avg_sq)):
        for name, a, stride in zip(D.GROUPS, bufs, D.STRIDES):
            out[k + name] = _tensor(st, a.ptr, (new, stride), owner=a)
    return out


def _run_mesh(st):
    case, dim = st["case"], st["case"]["dim"]
    st["grid"].zero_()
    E.tsdf_integrate(st["grid"], st["origin"], st["vs"], st["mesh_views"], 4 * st["vs"], 0.5)
    n, total = C.c_int64(), C.c_int64()
    E.check(E.lib().msplat_hip_marching_cubes(st["grid"].ptr, dim, dim, dim, (C.c_float * 3)(*st["origin"]), st["vs"],
                                              st["most"], st["tris"].ptr, C.byref(n), C.byref(total)))
    return dict(grid=_arr(st, st["grid"]), triangles=_arr(st, st["tris"]), count=total.value)


_RUN = dict(render=_run_render, frame=_run_frame, maps=_run_maps, train=_run_train, train3d=_run_train,
            grads=_run_grads, densify=_run_densify, mesh=_run_mesh)
LAMBDA_DIST = 0.01


# ---- what a pass cannot do without ------------------------------------------
def work(case):
    """Inputs read once and outputs written once; the operations of about 60
    splats composited per covered pixel (40 operations each forward, 90
    backward), 500 per projected splat, SSIM's five 11-tap separable windows
    forward and three backward."""
    kind = case["kind"]
    if kind == "densify":
        row = 59 * 3 * 4
        return dict(bytes=case["n"] * (row + 12) + 1.5 * case["n"] * row, flops=100.0 * case["n"])
    if kind == "mesh":
        v, px = case["dim"] ** 3, case["w"] * case["h"]
        return dict(bytes=8.0 * v + 8.0 * px * case["views"] + 36.0 * 3 * case["dim"] ** 2,
                    flops=30.0 * v * case["views"])
    n, px, d3 = case["n"], case["w"] * case["h"], kind == "train3d"
    floats = 3 * (case["degree"] + 1) ** 2 + 10 + d3
    blended = min(60.0, 0.4 * _intersections(case) * 256.0 / px)
    fwd_bytes, fwd_flops = 4.0 * floats * n, 500.0 * n + 40.0 * blended * px
    if kind == "render":
        return dict(bytes=fwd_bytes + 12.0 * px, flops=fwd_flops)
    if kind == "frame":
        return dict(bytes=fwd_bytes + 4.0 * px, flops=fwd_flops)
    if kind == "maps":
        return dict(bytes=fwd_bytes + 36.0 * px, flops=fwd_flops)
    ssim = 3.0 * px * 2 * 11 * 2 * 8
    flops = 2 * fwd_flops + 90.0 * blended * px + ssim
    if kind == "grads":
        return dict(bytes=2 * fwd_bytes + 24.0 * n + 28.0 * px, flops=flops)
    return dict(bytes=6 * fwd_bytes + 24.0 * n + 24.0 * px, flops=flops)


# About four times the largest error of one pass against exact(), measured on
# the listed cases.  Images: 1.2e-5 to 2.2e-5 (single pixels 0.007), where a
# splat at the alpha threshold falls on the other side.  The maps, and the
# gradients by the surfels' position and rotation, are dominated by a few
# surfels seen edge-on, whose ray-plane intersection is ill-conditioned in 32
# bits: 6e-3 (depth), 4e-3 (m_means), 0.08 (d_means), single values more than
# their root mean square.  Two runs of the same code differ by up to 1e-6
# (single values 4e-3) in the sums that are taken in any order.
_TOLERANCE = dict(
    render=dict(rel=1e-4, max=0.05),
    frame=dict(rel=0.0, differ=1e-3),  # bytes: a value next to a whole number
    maps=dict(rel=0.025, max=0.99),
    train=dict(rel=0.016, max=0.99),
    train3d=dict(rel=1e-4, max=0.06),
    grads=dict(rel=0.03, max=0.99),
    densify=dict(rel=1e-6),
    mesh=dict(rel=2e-3, max=0.99),  # voxels whose pixel is the neighbour's
)


def tolerance(case):
    return _TOLERANCE[case["kind"]]


# ---- the pass in 64 bits ----------------------------------------------------
def exact(case, seed):
    kind = case["kind"]
    if kind == "densify":
        return _exact_densify(case, seed)
    if kind == "mesh":
        return _exact_mesh(case, seed)
    if kind == "frame":
        return None  # bytes
    if _intersections(case) > CUTOFF_COST or (case["scene"] == "ball" and case["n"] > 300_000):
        return None
    params, cams = _host_inputs(case, seed)
    f = _Frame64(case, params, cams[0])
    if kind in ("render", "maps"):
        o = f.composite()
        if kind == "render":
            return dict(image=o["image"])
        return {k: o[k] for k in ("image", "depth", "normal", "alpha", "median")}
    dist = LAMBDA_DIST if kind == "grads" else 0.0
    o = f.composite(distortion=dist != 0.0)
    loss, dimg = _loss64(o["image"], _photo(case, seed, 0).double())
    grads, stats = f.backward(dimg, dist / (case["w"] * case["h"]))
    if dist:
        loss = loss + dist * float(o["distortion"].mean())
        out = dict(loss=loss, image=o["image"], distortion=o["distortion"], **stats)
        out.update({"d_" + k: v for k, v in grads.items()})
        return out
    out = dict(loss=loss, image=o["image"], **stats)
    for name, p, lr in zip(D.GROUPS, params, D.LR_INIT):
        g = grads[name]
        # Adam's first step: both bias corrections undo the moments' scale
        m, v = (1 - D.BETA1) * g, (1 - D.BETA2) * g * g
        step = LR_SCALE * lr * (m / (1 - D.BETA1)) / ((v / (1 - D.BETA2)).sqrt() + D.EPS)
        out["m_" + name] = m
        out[name] = torch.tensor(p, device=DEV).double().reshape(g.shape) - step
    return out


def _rotation(q):
    w, x, y, z = q.unbind(-1)
    return torch.stack([torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y)], -1),
                        torch.stack([2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x)], -1),
                        torch.stack([2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], -1)], -2)


def _sh_basis(d, degree):
    """Real spherical harmonics from their normalisation constants."""
    x, y, z = d.unbind(-1)
    pi = math.pi
    out = [torch.full_like(x, 0.5 / math.sqrt(pi))]
    if degree >= 1:
        c = math.sqrt(3 / (4 * pi))
        out += [-c * y, c * z, -c * x]
    if degree >= 2:
        a, b = 0.5 * math.sqrt(15 / pi), 0.25 * math.sqrt(5 / pi)
        out += [a * x * y, -a * y * z, b * (2 * z * z - x * x - y * y), -a * x * z, 0.5 * a * (x * x - y * y)]
    if degree >= 3:
        a, b = 0.25 * math.sqrt(35 / (2 * pi)), 0.25 * math.sqrt(21 / (2 * pi))
        c, e = 0.5 * math.sqrt(105 / pi), 0.25 * math.sqrt(7 / pi)
        out += [-a * y * (3 * x * x - y * y), c * x * y * z, -b * y * (4 * z * z - x * x - y * y),
                e * z * (2 * z * z - 3 * x * x - 3 * y * y), -b * x * (4 * z * z - x * x - y * y),
                0.5 * c * z * (x * x - y * y), -a * x * (x * x - 3 * y * y)]
    return torch.stack(out, -1)


def _through(value, carrier):
    """`value`, with the derivative of `carrier`."""
    return carrier + (value - carrier).detach()


class _Frame64:
    """One frame in float64: projection, tile lists (16 x 16 pixels, ordered
    by depth), compositing and its gradients by autograd.  The package's own
    conventions: the quaternion's normalisation, the low-pass distance, the
    alpha cap at 0.99 and (3D Gaussians) the clamp of the view position pass
    no derivative of their own, a splat stops contributing below alpha
    1/255, and a pixel stops before its transmittance falls to 1e-4."""

    PAIRS = 12_000_000  # (pixel, splat) pairs evaluated at once

    def __init__(self, case, params, cam):
        self.case, self.d3 = case, case["kind"] == "train3d"
        self.W, self.H = W, H = case["w"], case["h"]
        self.bg = torch.tensor(np.asarray(S.DEFAULT_BG, np.float64), device=DEV)
        c2w = np.asarray(cam.cam_to_world, np.float64)
        R, t = c2w[:3, :3] * np.array([1.0, -1.0, -1.0]), c2w[:3, 3]
        V = np.eye(4)
        V[:3, :3], V[:3, 3] = R.T, -R.T @ t
        n_, f_ = 0.001, 1000.0
        P = np.array([[2 * cam.fx / W, 0, 0, 0], [0, 2 * cam.fy / H, 0, 0],
                      [0, 0, (f_ + n_) / (f_ - n_), -f_ * n_ / (f_ - n_)], [0, 0, 1, 0]])
        V_, PV = (torch.tensor(a, device=DEV) for a in (V, P @ V))
        leaf = [torch.tensor(p, device=DEV).double().requires_grad_() for p in params]
        self.leaf = dict(zip(D.GROUPS, leaf))
        mean, scale, quat, fdc, frest, opac = leaf
        n = mean.shape[0]
        q = quat / quat.detach().norm(dim=1, keepdim=True)
        Rm = _rotation(q)
        hom = torch.cat([mean, torch.ones_like(mean[:, :1])], 1)
        pv = hom @ V_[:3].T
        ok = pv[:, 2] > 0.01
        vp = torch.tensor([[W / 2, 0, 0, cam.cx - 0.5], [0, H / 2, 0, cam.cy - 0.5], [0, 0, 0, 1]], device=DEV).double()
        if self.d3:
            M = Rm * scale.exp()[:, None, :]
            cov = M @ M.transpose(1, 2)
            z = pv[:, 2]
            lx, ly = 1.3 * 0.5 * W / cam.fx, 1.3 * 0.5 * H / cam.fy
            x = _through(z * (pv[:, 0] / z).clamp(-lx, lx), pv[:, 0])
            y = _through(z * (pv[:, 1] / z).clamp(-ly, ly), pv[:, 1])
            zero = torch.zeros_like(z)
            J = torch.stack([torch.stack([cam.fx / z, zero, -cam.fx * x / z ** 2], -1),
                             torch.stack([zero, cam.fy / z, -cam.fy * y / z ** 2], -1)], -2)
            JW = J @ V_[:3, :3]
            c2 = JW @ cov @ JW.transpose(1, 2)
            a, b, c = c2[:, 0, 0] + 0.3, c2[:, 0, 1], c2[:, 1, 1] + 0.3
            det = a * c - b * b
            ok = ok & (det != 0)
            h = hom @ PV.T
            xy = torch.stack([0.5 * W * h[:, 0] / (h[:, 3] + 1e-6) + cam.cx - 0.5,
                              0.5 * H * h[:, 1] / (h[:, 3] + 1e-6) + cam.cy - 0.5], 1)
            mid = 0.5 * (a + c)
            radius = (3 * (mid + (mid * mid - det).clamp(min=0.1).sqrt()).sqrt()).ceil().detach()
            geo = torch.cat([xy, torch.stack([c / det, -b / det, a / det], 1)], 1)
        else:
            s = scale.exp()
            cols = torch.stack([torch.cat([Rm[:, :, 0] * s[:, :1], 0 * mean[:, :1]], 1),
                                torch.cat([Rm[:, :, 1] * s[:, 1:], 0 * mean[:, :1]], 1), hom], 2)
            T = (vp @ PV) @ cols  # rows Tu, Tv, Tw
            with torch.no_grad():
                w9 = torch.tensor([9.0, 9.0, -1.0], device=DEV).double()
                dd = (w9 * T[:, 2] ** 2).sum(1)
                ok = ok & (dd != 0)
                fw = w9 / dd[:, None]
                xy = torch.stack([(fw * T[:, 0] * T[:, 2]).sum(1), (fw * T[:, 1] * T[:, 2]).sum(1)], 1)
                ext = [(xy[:, k] ** 2 - (fw * T[:, k] ** 2).sum(1)).clamp(min=1e-4).sqrt() for k in (0, 1)]
                radius = torch.maximum(torch.maximum(*ext), torch.full_like(dd, 3 * 0.707106)).ceil()
            geo = T.reshape(n, 9)
        dirs = mean - torch.tensor(t, device=DEV)
        dirs = dirs / dirs.norm(dim=1, keepdim=True)
        act = case["active"]
        basis = _sh_basis(dirs, act)
        coef = torch.cat([fdc[:, None], frest.reshape(n, -1, 3)], 1)[:, : (act + 1) ** 2]
        rgb = ((basis[:, :, None] * coef).sum(1) + 0.5).clamp(min=0)
        # what the pixels see of a splat, all differentiable but xy (2DGS)
        self.attr = torch.cat([geo, Rm[:, :, 2], opac.sigmoid(), rgb], 1)
        self.K = geo.shape[1]
        with torch.no_grad():
            TX, TY = (W + 15) // 16, (H + 15) // 16
            lo = [((xy[:, k] - radius) / 16).trunc().clamp(0, m) for k, m in ((0, TX), (1, TY))]
            hi = [((xy[:, k] + radius) / 16 + 1).trunc().clamp(0, m) for k, m in ((0, TX), (1, TY))]
            nx, ny = (hi[0] - lo[0]).clamp(min=0), (hi[1] - lo[1]).clamp(min=0)
            ok = ok & (nx * ny > 0)
            self.ok, self.radius, self.depth, self.xy = ok, radius, pv[:, 2].detach(), xy.detach()
            idx = torch.nonzero(ok)[:, 0]
            idx = idx[torch.argsort(self.depth[idx], stable=True)]
            cnt = (nx * ny)[idx].long()
            ids = torch.repeat_interleave(idx, cnt)
            pos = torch.arange(ids.numel(), device=DEV) - torch.repeat_interleave(cnt.cumsum(0) - cnt, cnt)
            wide = nx[ids].long()
            tile = (lo[1][ids].long() + pos // wide) * TX + lo[0][ids].long() + pos % wide
            order = torch.argsort(tile, stable=True)
            self.ids, self.len = ids[order], torch.bincount(tile, minlength=TX * TY)
            self.start = self.len.cumsum(0) - self.len
            self.TX, self.tiles = TX, TX * TY

    def _chunks(self):
        """Groups of (tiles, pixels of a tile) of at most PAIRS pairs."""
        order = torch.argsort(self.len, descending=True)
        lens = self.len[order].tolist()
        at = 0
        while at < len(lens):
            longest = max(1, lens[at])
            per = max(1, self.PAIRS // (256 * longest))
            tiles = order[at: at + per]
            step = 256
            while step > 1 and longest * step * len(tiles) > self.PAIRS:
                step //= 2
            for p in range(0, 256, step):
                yield tiles, longest, torch.arange(p, p + step, device=DEV)
            at += per

    def _pixels(self, tiles, longest, lane, attr, want, full):
        """Composites `lane` pixels of `tiles`: per-pixel sums [B, P, .]."""
        k = torch.arange(longest, device=DEV)
        live = k[None] < self.len[tiles][:, None]
        gid = self.ids[(self.start[tiles][:, None] + k[None]).clamp(max=max(0, self.ids.numel() - 1))]
        px = ((tiles % self.TX)[:, None] * 16 + lane[None] % 16).double()
        py = ((tiles // self.TX)[:, None] * 16 + lane[None] // 16).double()
        q = attr[gid]
        if want:
            q = q.detach().requires_grad_()
        a = q[:, :, None, :]
        X, Y = px[:, None, :], py[:, None, :]
        K = self.K
        opa, rgb, nrm = a[..., K + 3], q[..., K + 4:], q[..., K:K + 3]
        depth = None
        if self.d3:
            dx, dy = a[..., 0] - X, a[..., 1] - Y
            rho = a[..., 2] * dx * dx + 2 * a[..., 3] * dx * dy + a[..., 4] * dy * dy
            keep = rho.detach() >= 0
        else:
            kk = [X * a[..., 6 + i] - a[..., i] for i in range(3)]
            ll = [Y * a[..., 6 + i] - a[..., 3 + i] for i in range(3)]
            rz = kk[0] * ll[1] - kk[1] * ll[0]
            u = (kk[1] * ll[2] - kk[2] * ll[1]) / rz
            v = (kk[2] * ll[0] - kk[0] * ll[2]) / rz
            c = self.xy[gid][:, :, None]
            r2 = 2 * ((c[..., 0] - X) ** 2 + (c[..., 1] - Y) ** 2)
            r3 = u * u + v * v
            low = ~(r3.detach() <= r2)
            rho = torch.where(low, r2, r3)
            uu, vv = torch.where(low, u.detach(), u), torch.where(low, v.detach(), v)
            depth = uu * a[..., 6] + vv * a[..., 7] + a[..., 8]
            keep = (rz.detach() != 0) & ~(depth.detach() < 0.2)
        raw = opa * (-0.5 * rho).exp()
        alpha = _through(raw.clamp(max=0.99), raw)
        keep = keep & ~(alpha.detach() < 1 / 255) & live[:, :, None]
        alpha = torch.where(keep, alpha, 0.0)
        logs = torch.log1p(-alpha)
        after = logs.cumsum(1)
        on = (after.detach().exp() > 1e-4) & keep
        alpha, logs = torch.where(on, alpha, 0.0), torch.where(on, logs, 0.0)
        after = logs.cumsum(1)
        before = (after - logs).exp()
        w = alpha * before
        Tend = after[:, -1].exp()
        out = dict(w=w, T=Tend, image=torch.einsum("blp,blc->bpc", w, rgb) + Tend[..., None] * self.bg)
        if full:
            depth = torch.where(on, depth, 1.0)
            m = 100.0 / 99.8 * (1 - 0.2 / depth)
            m = torch.where(on, m, 0.0)
            wm, wmm = (w * m), (w * m * m)
            A = 1 - before
            out["distortion"] = (w * (m * m * A + (wmm.cumsum(1) - wmm) - 2 * m * (wm.cumsum(1) - wm))).sum(1)
            if not want:
                out["depth"] = (w * depth).sum(1)
                out["normal"] = torch.einsum("blp,blc->bpc", w, nrm)
                out["alpha"] = 1 - Tend
                half = on & (before > 0.5)
                last = torch.where(half, k[None, :, None], -1).amax(1, keepdim=True)
                med = depth.gather(1, last.clamp(min=0))[:, 0]
                out["median"] = torch.where(last[:, 0] >= 0, med, 0.0)
        return out, q, gid, px.long(), py.long()

    def composite(self, distortion=False):
        full = not self.d3 and (distortion or self.case["kind"] == "maps")
        res = {}
        with torch.no_grad():
            for tiles, longest, lane in self._chunks():
                o, _, _, px, py = self._pixels(tiles, longest, lane, self.attr.detach(), False, full)
                inside = (px < self.W) & (py < self.H)
                for k, t in o.items():
                    if k != "w":
                        if k not in res:
                            res[k] = torch.zeros((self.H, self.W) + t.shape[2:], device=DEV, dtype=torch.float64)
                        res[k][py[inside], px[inside]] = t[inside]
        return res

    def backward(self, dimg, ddist):
        """Parameter gradients and the densification statistics."""
        attr = self.attr.detach()
        G = torch.zeros_like(attr)
        for tiles, longest, lane in self._chunks():
            if longest <= 1 and not bool(self.len[tiles].any()):
                continue
            o, q, gid, px, py = self._pixels(tiles, longest, lane, attr, True, ddist != 0)
            inside = (px < self.W) & (py < self.H)
            x, y = px.clamp(max=self.W - 1), py.clamp(max=self.H - 1)
            s = (o["image"] * dimg[y, x] * inside[..., None]).sum()
            if ddist:
                s = s + ddist * (o["distortion"] * inside).sum()
            s.backward()
            G.index_add_(0, gid.reshape(-1), q.grad.reshape(-1, G.shape[1]))
        self.attr.backward(G)
        grads = {k: t.grad for k, t in self.leaf.items()}
        w, h = self.W, self.H
        if self.d3:
            norm = (0.5 * w * G[:, 0]).abs() + (0.5 * h * G[:, 1]).abs()
        else:
            norm = (G[:, 6:8].abs() * self.depth[:, None] * torch.tensor([0.5 * w, 0.5 * h], device=DEV)).sum(1)
        zero = torch.zeros_like(norm)
        stats = dict(grad_norm=torch.where(self.ok, norm, zero), vis=self.ok.double(),
                     max2d=torch.where(self.ok, self.radius / max(w, h), zero))
        return grads, stats


def _loss64(img, gt, weight=0.2):
    """(1 - w) L1 + w (1 - SSIM), and its gradient by the image."""
    x = torch.arange(11, device=DEV).double() - 5
    g = (-x * x / (2 * 1.5 ** 2)).exp()
    g = (g / g.sum()).repeat(3, 1)

    def blur(t):
        t = sum(torch.nn.functional.pad(t, (5, 5))[..., k:k + t.shape[-1]] * g[0, k] for k in range(11))
        return sum(torch.nn.functional.pad(t, (0, 0, 5, 5))[..., k:k + t.shape[-2], :] * g[0, k] for k in range(11))

    a = img.detach().permute(2, 0, 1).contiguous().requires_grad_()
    b = gt.permute(2, 0, 1)
    m1, m2 = blur(a), blur(b)
    s1, s2, s12 = blur(a * a) - m1 * m1, blur(b * b) - m2 * m2, blur(a * b) - m1 * m2
    ssim = ((2 * m1 * m2 + 1e-4) * (2 * s12 + 9e-4)) / ((m1 * m1 + m2 * m2 + 1e-4) * (s1 + s2 + 9e-4))
    loss = (1 - weight) * (a - b).abs().mean() + weight * (1 - ssim.mean())
    loss.backward()
    return float(loss.detach()), a.grad.permute(1, 2, 0)


def _exact_densify(case, seed):
    params, m, v, grad, vis, max2d, noise = [
        [torch.tensor(np.asarray(x, np.float32), device=DEV).double() for x in a] if isinstance(a, list) else
        torch.tensor(np.asarray(a, np.float32), device=DEV).double() for a in _densify_inputs(case, seed)]
    params[4] = params[4].reshape(case["n"], -1)
    m[4], v[4] = m[4].reshape(case["n"], -1), v[4].reshape(case["n"], -1)
    mean, scale, quat, fdc, frest, opac = params
    high = (vis > 0) & (grad / vis.clamp(min=1) * 648.5 > 0.0002)
    large = scale.exp().amax(1) > 0.01
    split = high & (large | (max2d > 0.05))
    dup = high & ~large
    s = torch.nonzero(split)[:, 0]
    q = quat[s] / quat[s].norm(dim=1, keepdim=True)
    z = noise[: 2 * len(s)].reshape(len(s), 2, 3)
    off = torch.einsum("nij,nkj->nki", _rotation(q)[:, :, :2], z[:, :, :2] * scale[s].exp()[:, None])
    child = [(mean[s][:, None] + off).reshape(-1, 3)] + [p[s].repeat_interleave(2, 0) for p in params[1:]]
    child[1] = child[1] - math.log(1.6)
    # a splat that is both split and duplicated passes on its reduced scales
    params[1] = torch.where(split[:, None], scale - math.log(1.6), scale)
    keep = ~(opac.sigmoid()[:, 0] < 0.1)

    def grown(p, c):
        parts = [p[keep & ~split], c[c_keep]] + [p[dup & keep]]
        return torch.cat(parts)

    c_keep = keep[s].repeat_interleave(2)
    out = {}
    for i, name in enumerate(D.GROUPS):
        out[name] = grown(params[i], child[i])
        for tag, mom in (("m_", m), ("v_", v)):
            rest = torch.zeros(len(out[name]) - int((keep & ~split).sum()), mom[i].shape[1], device=DEV).double()
            out[tag + name] = torch.cat([mom[i][keep & ~split], rest])
    out["count"] = len(out["means"])
    return out


def _exact_mesh(case, seed):
    dim = case["dim"]
    vs, origin = _mesh_grid(case)
    c = [origin[k] + (torch.arange(dim, device=DEV).double() + 0.5) * vs for k in range(3)]
    p = torch.stack(torch.meshgrid(c[2], c[1], c[0], indexing="ij")[::-1], -1).reshape(-1, 3)
    sdf, wt = torch.zeros(len(p), device=DEV).double(), torch.zeros(len(p), device=DEV).double()
    h, w, trunc = case["h"], case["w"], 4 * vs
    for (vm, fx, fy, cx, cy), (depth, alpha) in zip(_mesh_cameras(case, seed), _mesh_maps(case, seed)):
        m = torch.tensor(vm, device=DEV).double()
        pv = p @ m[:3, :3].T + m[:3, 3]
        ix = (pv[:, 0] / pv[:, 2] * float(fx) + float(cx)).trunc().long()
        iy = (pv[:, 1] / pv[:, 2] * float(fy) + float(cy)).trunc().long()
        ok = (pv[:, 2] > 0.01) & (ix >= 0) & (ix < w) & (iy >= 0) & (iy < h)
        at = (iy.clamp(0, h - 1) * w + ix.clamp(0, w - 1))
        d, a = depth.double().reshape(-1)[at], alpha.double().reshape(-1)[at]
        s = d - pv[:, 2]
        ok = ok & (a >= 0.5) & (d > 0) & (s >= -trunc)
        nw = wt + a
        sdf = torch.where(ok, (sdf * wt + s.clamp(-trunc, trunc) * a) / nw, sdf)
        wt = torch.where(ok, nw, wt)
    return dict(grid=torch.stack([sdf, wt], -1).reshape(dim, dim, dim, 2), triangles=None, count=None)
