"""The work that a user of helio_amd has it do, as measurable cases.

A case names one call pattern of the public entry points and its sizes:

  frame    light cull (tiles or clusters) + deferred shading of one view
  shadow   the same with shadow maps and radiance-cascade GI
  reflect  both draws of the deferred pass: the lit frame, then the reflection composite added to it
  pack     the G-buffer producer's target writes
  forward  forward-lit fragments under the clustered light grid
  train    cluster cull + fused forward / L2 loss / adjoint
  grad     cluster cull + adjoint of a given dL/dradiance
  views    many views (probe faces, eyes with the adjoint) in one captured plan

Scenes are made on the GPU from the seed: a ground plane with boxes seen by a
perspective camera, one material per object with a little texture noise, the
surfaces' own normals with a little normal-map noise, and lights spread
uniformly over the scene's volume.  Sizes, light counts, ranges, cluster grids
and formats are those of helio_amd.synth's workloads and of bench.py.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from helio_amd import abi
from helio_amd import batch as hb
from helio_amd import device as hd

DEV = "cuda"
F32, F64 = torch.float32, torch.float64
# format set -> (albedo / orm format, texel bytes, normal / emissive format, texel bytes)
FORMATS = {
    "ref": (abi.HL_FMT_RGBA8_UNORM, 4, abi.HL_FMT_RGBA16_FLOAT, 8),
    "f16": (abi.HL_FMT_RGBA16_FLOAT, 8, abi.HL_FMT_RGBA16_FLOAT, 8),
    "f32": (abi.HL_FMT_RGBA32_FLOAT, 16, abi.HL_FMT_RGBA32_FLOAT, 16),
}
AMBIENT = (0.5, 0.5, 0.6)
NEAR, FAR = 0.1, 1000.0
# the smoothest material of a scene (textures seldom go below), and of a scene that is fitted, where
# roughness is kept away from mirrors, whose gradients are spikes
SMOOTHEST, SMOOTHEST_FITTED = 0.15, 0.2
CSM = (16.0, 80.0, 300.0, 1400.0)


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one face of a reflection probe: the smallest call, latency and launches
        dict(name="face_128", kind="frame", w=128, h=128, fmt="ref", lights=256, spots=0.0, half=20.0,
             grid="clusters", gx=4, gy=4, gz=24, out="f32", pose="face"),
        # an ordinary small frame the reference's way: 16-px tiles, RGBA16F target
        dict(name="frame_720p_tiles", kind="frame", w=1280, h=720, fmt="ref", lights=64, spots=0.0, half=20.0,
             grid="tiles", gx=0, gy=0, gz=0, out="f16", pose="front"),
        # an ordinary frame on clustered lists, a quarter of the lights spots
        dict(name="frame_1080p", kind="frame", w=1920, h=1080, fmt="ref", lights=1024, spots=0.25, half=40.0,
             grid="clusters", gx=16, gy=9, gz=24, out="f32", pose="front"),
        # the largest frame: 4K, fp16 G-buffer, 16384 lights, clustered
        dict(name="frame_4k", kind="frame", w=3840, h=2160, fmt="f16", lights=16384, spots=0.0, half=100.0,
             grid="clusters", gx=32, gy=18, gz=48, out="f32", pose="front"),
        # the same lights on the reference's tile lists (cap 64)
        dict(name="frame_4k_tiles", kind="frame", w=3840, h=2160, fmt="ref", lights=16384, spots=0.0, half=100.0,
             grid="tiles", gx=0, gy=0, gz=0, out="f32", pose="front"),
        # a frame with everything fs_main samples: sun, point and spot shadows (PCSS) and RC GI
        dict(name="shadow_1080p", kind="shadow", w=1920, h=1080, fmt="ref", lights=1024, half=40.0, gx=16, gy=9,
             gz=24, points=4, spotcasters=4, atlas=1024, quality="high", rc=True),
        # both draws of a 1440p frame: reflection captures, SSR, planar and RC specular over the lights
        dict(name="reflect_1440p", kind="reflect", w=2560, h=1440, fmt="ref", lights=256, half=40.0, gx=16, gy=9,
             gz=24, boxes=8, spheres=8, face=128, mips=8, rc=True),
        # the G-buffer producer's writes of a 4K frame in the reference formats
        dict(name="pack_4k", kind="pack", w=3840, h=2160, fmt="ref", f0=False),
        # transparent / forward-shaded surfaces of a frame of odd size, lights read through transforms
        dict(name="forward_1917x1079", kind="forward", w=1917, h=1079, lights=4096, spots=0.25, half=40.0, gx=16,
             gy=9, gz=24),
        # one step of inverse rendering at 512^2 (fp32 G-buffer)
        dict(name="train_512", kind="train", w=512, h=512, fmt="f32", lights=256, spots=0.0, half=20.0, gx=16, gy=9,
             gz=24),
        # the adjoint alone under a caller's own loss, a ragged size
        dict(name="grad_773x431", kind="grad", w=773, h=431, fmt="f32", lights=512, spots=0.25, half=20.0, gx=16,
             gy=9, gz=24),
        # probe faces and two eyes with the adjoint in one captured plan
        dict(name="views_26", kind="views", faces=24, size=128, eye_w=1032, eye_h=1104, lights=4096, subset=512,
             half=50.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, most=3840 * 2160):
    """A width and height, 128^2 to `most` pixels, odd ones among them."""
    px = math.exp(rng.uniform(math.log(128 * 128), math.log(most)))
    aspect = rng.choice((1.0, 4.0 / 3.0, 16.0 / 9.0))
    w, h = int(math.sqrt(px * aspect)), int(math.sqrt(px / aspect))
    if rng.random() < 0.5:
        w, h = w // 8 * 8, h // 8 * 8
    return max(w, 64), max(h, 64)


def _half(lights):
    return 20.0 if lights <= 512 else 40.0 if lights <= 4096 else 100.0


def _cluster_grid(w, h):
    return (32, 18, 48) if w * h > 3e6 else (16, 9, 24) if w * h > 1e5 else (4, 4, 24)


def draw(rng):
    kind = rng.choice(("frame",) * 5 + ("shadow", "reflect", "pack", "forward", "train", "grad", "views"))
    if kind == "views":
        return dict(kind=kind, faces=rng.randint(6, 24), size=rng.choice((64, 96, 128)),
                    eye_w=rng.randint(500, 1032), eye_h=rng.randint(500, 1104), lights=_log(rng, 512, 4096),
                    subset=rng.randint(32, 512), half=50.0)
    most = {"frame": 3840 * 2160, "shadow": 1920 * 1080, "reflect": 2560 * 1440, "pack": 3840 * 2160,
            "forward": 1920 * 1080, "train": 768 * 768, "grad": 768 * 768}[kind]
    w, h = _size(rng, most)
    c = dict(kind=kind, w=w, h=h)
    if kind == "pack":
        return dict(c, fmt=rng.choice(("ref", "ref", "f16", "f32")), f0=rng.random() < 0.3)
    gx, gy, gz = _cluster_grid(w, h)
    if kind == "reflect":
        n = _log(rng, 32, 1024)
        return dict(c, fmt=rng.choice(("ref", "f16", "f32")), lights=n, half=_half(n), gx=gx, gy=gy, gz=gz,
                    boxes=rng.randint(1, 8), spheres=rng.randint(1, 8), face=rng.choice((64, 128)), mips=7,
                    rc=rng.random() < 0.5)
    if kind == "shadow":
        n = _log(rng, 64, 1024)
        return dict(c, fmt=rng.choice(("ref", "f16")), lights=n, half=_half(n), gx=gx, gy=gy, gz=gz,
                    points=rng.randint(1, 4), spotcasters=rng.randint(1, 4), atlas=rng.choice((512, 1024)),
                    quality=rng.choice(("medium", "high")), rc=rng.random() < 0.5)
    if kind in ("train", "grad"):
        n = _log(rng, 32, 512)
        return dict(c, fmt="f32", lights=n, spots=rng.choice((0.0, 0.25)), half=20.0, gx=16, gy=9, gz=24)
    n = _log(rng, 64, 16384 if kind == "frame" else 4096)
    if kind == "forward":
        return dict(c, lights=n, spots=rng.choice((0.0, 0.25)), half=_half(n), gx=gx, gy=gy, gz=gz)
    tiles = rng.random() < 0.4
    return dict(c, fmt=rng.choice(("ref", "ref", "f16", "f32")), lights=n, spots=rng.choice((0.0, 0.25)),
                half=_half(n), grid="tiles" if tiles else "clusters", gx=0 if tiles else gx, gy=0 if tiles else gy,
                gz=0 if tiles else gz, out=rng.choice(("f32", "f16")), pose=rng.choice(("front", "front", "face")))


# ------------------------------------------------------------------- scenes
def _gen(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFFFFFFFFFF)
    return g


def _rand(g, *shape, lo=0.0, hi=1.0):
    return torch.rand(*shape, generator=g, device=DEV, dtype=F32) * (hi - lo) + lo


def _unit(v):
    return v / np.linalg.norm(v)


def _look(eye, fwd):
    """Right-handed view matrix from eye along fwd, and its axes (float64)."""
    f = _unit(np.asarray(fwd, float))
    up = np.array((0.0, 1.0, 0.0)) if abs(f[1]) <= 0.999 else np.array((0.0, 0.0, -1.0))
    r = _unit(np.cross(f, up))
    u = np.cross(r, f)
    m = np.eye(4)
    m[0, :3], m[1, :3], m[2, :3] = r, u, -f
    m[:3, 3] = -m[:3, :3] @ np.asarray(eye, float)
    return m, f, r, u


def _persp(sx, sy, near, far):
    r = far / (near - far)
    p = np.zeros((4, 4))
    p[0, 0], p[1, 1], p[2, 2], p[2, 3], p[3, 2] = sx, sy, r, r * near, -1.0
    return p


def _camera(w, h, eye, fwd, fov):
    view, f, r, u = _look(eye, fwd)
    t = math.tan(math.radians(fov) / 2)
    proj = _persp(1 / (t * w / h), 1 / t, NEAR, FAR)
    vp = proj @ view
    cam = abi.GpuCameraUniforms()
    for name, m in (("view", view), ("proj", proj), ("view_proj", vp), ("inv_view_proj", np.linalg.inv(vp)),
                    ("prev_view_proj", vp)):
        getattr(cam, name)[:] = m.T.ravel().tolist()  # column-major
    cam.position_near[:] = (*eye, NEAR)
    cam.forward_far[:] = (*f, FAR)
    return dict(cam=cam, eye=np.asarray(eye, float), f=f, r=r, u=u, t=t, aspect=w / h)


def _pose(pose, half, rng):
    if pose == "face":  # a probe inside the scene
        eye = (rng.uniform(-0.4, 0.4) * half, rng.uniform(2.0, 8.0), rng.uniform(-0.4, 0.4) * half)
        fwd = ((0, 0, -1), (0, 0, 1), (1, 0, 0), (-1, 0, 0))[rng.integers(4)]
        return eye, fwd, 90.0
    eye = (rng.uniform(-0.05, 0.05) * half, 7.0 + 0.05 * half, 1.15 * half + 9.0)
    return eye, (-eye[0], -eye[1], -eye[2]), 60.0


def _field(half, g, rng, smoothest=SMOOTHEST):
    """Boxes on the ground (lo, hi as host arrays) and a material per object (last: the ground)."""
    n = 40 if half <= 20 else 60 if half <= 50 else 96
    big = half / 20.0
    c = rng.uniform(-half, half, (n, 2))
    s = rng.uniform(1.0, 4.0, (n, 2)) * max(1.0, 0.5 * big)
    y = rng.uniform(0.5, 6.0, n) * max(1.0, 0.5 * big)
    lo = np.stack([c[:, 0] - s[:, 0] / 2, np.zeros(n), c[:, 1] - s[:, 1] / 2], 1)
    hi = np.stack([c[:, 0] + s[:, 0] / 2, y, c[:, 1] + s[:, 1] / 2], 1)
    mat = dict(smoothest=smoothest, albedo=_rand(g, n + 1, 3), rough=_rand(g, n + 1, lo=smoothest), metal=(_rand(g, n + 1) < 0.3).to(F32),
               glow=(_rand(g, n + 1, 1) < 0.05).to(F32) * _rand(g, n + 1, 3, hi=0.5))
    return lo, hi, mat


def _hits(o, d, lo, hi, step=1, first=0, ground=True):
    """First hit along rays o + t d (host origin or tensors): t (inf: none), object, face axis."""
    n = len(lo)
    ox, oy, oz = o
    dx, dy, dz = (torch.where(v.abs() < 1e-9, torch.full_like(v, 1e-9), v) for v in d)
    inv = (1 / dx, 1 / dy, 1 / dz)
    t = torch.full_like(dx, math.inf)
    obj = torch.full(dx.shape, n, device=DEV, dtype=torch.int32)
    axis = torch.ones(dx.shape, device=DEV, dtype=torch.int32)
    if ground:
        tg = -oy * inv[1]
        t = torch.where(tg > 0, tg, t)
    for b in range(first, n, step):
        near = far = near_axis = None
        for a, (oa, ia) in enumerate(zip((ox, oy, oz), inv)):
            t0, t1 = (float(lo[b, a]) - oa) * ia, (float(hi[b, a]) - oa) * ia
            n0, n1 = torch.minimum(t0, t1), torch.maximum(t0, t1)
            if near is None:
                near, far, near_axis = n0, n1, torch.zeros_like(axis)
            else:
                near_axis = torch.where(n0 > near, a, near_axis)
                near, far = torch.maximum(near, n0), torch.minimum(far, n1)
        hit = (near <= far) & (near > 0) & (near < t)
        t = torch.where(hit, near, t)
        obj = torch.where(hit, b, obj)
        axis = torch.where(hit, near_axis, axis)
    return t, obj, axis


def _unorm8(v):
    return (v.clamp(0, 1) * 255).round().to(torch.uint8)


def _gbuffer(w, h, cam, field, fmt, g):
    lo, hi, mat = field
    px = ((torch.arange(w, device=DEV, dtype=F32) + 0.5) / w * 2 - 1)[None, :].expand(h, w)
    py = (1 - (torch.arange(h, device=DEV, dtype=F32) + 0.5) / h * 2)[:, None].expand(h, w)
    d = [float(cam["f"][a]) + px * float(cam["t"] * cam["aspect"] * cam["r"][a]) + py * float(cam["t"] * cam["u"][a])
         for a in range(3)]  # advances one unit of view distance per t
    t, obj, axis = _hits([float(v) for v in cam["eye"]], d, lo, hi)
    sky = ~(t < 0.999 * FAR)
    vd = t.to(F64).clamp(min=1.01 * NEAR)
    pr = cam["cam"].proj
    depth = ((pr[10] * -vd + pr[14]) / vd).to(F32)
    depth = torch.where(sky, torch.ones_like(depth), depth.clamp(max=1 - 2.0 ** -24))
    obj = obj.long()
    n = torch.randn(h, w, 3, generator=g, device=DEV, dtype=F32) * 0.08
    n.scatter_add_(2, axis.long()[..., None], -torch.sign(torch.stack(d, -1).gather(2, axis.long()[..., None])))
    n = n / n.norm(dim=-1, keepdim=True)
    tex = _rand(g, h, w, 1, lo=0.7)
    alb = mat["albedo"][obj] * tex
    rough = (mat["rough"][obj] + _rand(g, h, w, lo=-0.05, hi=0.05)).clamp(mat["smoothest"], 1)
    ao = _rand(g, h, w, lo=0.8)
    metal = mat["metal"][obj]
    glow = mat["glow"][obj]
    one = torch.ones(h, w, 1, device=DEV, dtype=F32)
    if fmt == "ref":
        alb, ao, rough = (_unorm8(v).to(F32) / 255 for v in (alb, ao, rough))
    elif fmt == "f16":
        alb, ao, rough = (v.half().to(F32) for v in (alb, ao, rough))
    f0 = (0.04 * (1 - metal[..., None]) + alb * metal[..., None]).clamp(0, 0.999)
    planes = dict(albedo=torch.cat([alb, one], -1), normal=torch.cat([n, f0[..., :1]], -1),
                  orm=torch.stack([ao, rough, metal, f0[..., 1]], -1), emissive=torch.cat([glow, f0[..., 2:]], -1))
    if fmt == "ref":
        planes = {k: _unorm8(v) if k in ("albedo", "orm") else v.half() for k, v in planes.items()}
    elif fmt == "f16":
        planes = {k: v.half() for k, v in planes.items()}
    return dict({k: v.contiguous() for k, v in planes.items()}, depth=depth.contiguous())


def _lights(n, half, spots, g):
    """GpuLight records (host) and their fields (device)."""
    height = max(10.0, 0.3 * half)
    p = _rand(g, n, 3)
    pos = torch.stack([(p[:, 0] - 0.5) * 2 * half, p[:, 1] * height, (p[:, 2] - 0.5) * 2 * half], 1)
    rng = _rand(g, n, lo=2.0, hi=10.0) if half <= 40 else _rand(g, n, lo=1.0, hi=8.0)
    color, inten = _rand(g, n, 3, lo=0.5), _rand(g, n, lo=0.5, hi=5.0)
    kind = torch.where(_rand(g, n) < spots, abi.HL_LIGHT_SPOT, abi.HL_LIGHT_POINT).to(torch.int32)
    dirs = torch.randn(n, 3, generator=g, device=DEV, dtype=F32)
    dirs[:, 1] = -dirs[:, 1].abs() - 0.2
    dirs = dirs / dirs.norm(dim=1, keepdim=True)
    angle = torch.deg2rad(_rand(g, n, lo=10.0, hi=45.0))
    return _light_records(dict(pos=pos, range=rng, color=color, intensity=inten, kind=kind, dir=dirs,
                               outer=torch.cos(angle), inner=torch.cos(0.8 * angle)))


def _light_records(f):
    rec = np.zeros(len(f["range"]), dtype=abi.GPU_LIGHT_DTYPE)
    host = {k: v.cpu().numpy() for k, v in f.items()}
    rec["position_range"] = np.concatenate([host["pos"], host["range"][:, None]], 1)
    rec["color_intensity"] = np.concatenate([host["color"], host["intensity"][:, None]], 1)
    rec["direction_outer"] = np.concatenate([host["dir"], host["outer"][:, None]], 1)
    rec["inner_angle"], rec["light_type"] = host["inner"], host["kind"]
    rec["shadow_index"], rec["ies_profile_index"], rec["light_function_index"] = abi.HL_NO_SHADOW, -1, -1
    return dict(f, records=rec)


def _scene(case, seed):
    """Camera, G-buffer and lights of a single-view case."""
    g, rng = _gen(seed), np.random.default_rng(int(seed))
    field = _field(case["half"], g, rng, SMOOTHEST_FITTED if case["kind"] in ("train", "grad") else SMOOTHEST)
    eye, fwd, fov = _pose(case.get("pose", "front"), case["half"], rng)
    cam = _camera(case["w"], case["h"], eye, fwd, fov)
    fmt = case.get("fmt", "f32")
    s = dict(w=case["w"], h=case["h"], fmt=fmt, cam=cam, field=field, rng=rng, g=g,
             planes=_gbuffer(case["w"], case["h"], cam, field, fmt, g))
    if "lights" in case:
        s["lights"] = _lights(case["lights"], case["half"], case.get("spots", 0.0), g)
    return s


def _globals(w, n):
    g = abi.DeferredGlobals()
    g.light_count, g.ambient_intensity, g.num_tiles_x, g.enable_reflections = n, 1.0, (w + 15) // 16, 1
    g.ambient_color[:] = (*AMBIENT, 1.0)
    g.csm_splits[:] = CSM
    return g


# ------------------------------------------------ the framework's handles
_CTX = None


def _ctx():
    """The program's one context, on torch's stream."""
    global _CTX
    if _CTX is None:
        torch.cuda.init()
        _CTX = hd.Context(0)
        _CTX.lib.call("hl_set_stream", _CTX.h, torch.cuda.current_stream().cuda_stream or None)
    return _CTX


class _Buf:
    """A torch tensor where the passes take a device buffer."""

    def __init__(self, t):
        self.tensor, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()


class _View:
    """The device memory of a pass's own buffer, which it keeps alive, as torch sees it."""

    def __init__(self, arr, shape, typestr):
        self.arr = arr
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=typestr, data=(arr.ptr, False), version=2)


def _tensor(arr, shape, typestr="<f4", zero=True):
    t = torch.as_tensor(_View(arr, shape, typestr), device=DEV)
    return t.zero_() if zero else t


class _Host:
    def __init__(self, w, h, camera, globals_, lights):
        self.width, self.height, self.camera, self.globals, self.lights = w, h, camera, globals_, lights


def _upload(a):
    return torch.from_numpy(np.frombuffer(bytes(a), dtype=np.uint8).copy()).to(DEV)


def _device_scene(s, records=None, light_buf=None):
    records = s["lights"]["records"] if records is None else records
    cam = s["cam"]["cam"]
    fa, ta, fn, tn = FORMATS[s["fmt"]]
    gb = abi.hl_gbuffer()
    gb.width, gb.height = s["w"], s["h"]
    bufs = {k: _Buf(v) for k, v in s["planes"].items()}
    for name, fmt, tb in (("albedo", fa, ta), ("orm", fa, ta), ("normal", fn, tn), ("emissive", fn, tn),
                          ("depth", abi.HL_FMT_R32_FLOAT, 4)):
        t = getattr(gb, name)
        t.data_d, t.pitch_bytes, t.format = bufs[name].ptr, s["w"] * tb, fmt
    host = _Host(s["w"], s["h"], cam, _globals(s["w"], len(records)), records)
    lights = light_buf or _Buf(_upload(records.tobytes()) if len(records) else torch.zeros(128, device=DEV))
    return hd.DeviceScene(host, _Buf(_upload(cam)), lights, bufs, gb)


def _params(ctx, cam, w, h, grid):
    p = abi.hl_cluster_params()
    ctx.lib.call("hl_cluster_params_init", C.byref(cam), w, h, *grid, 0, C.byref(p))
    return p


def _cluster_cull(ctx, s, case, ds):
    grid = (case["gx"], case["gy"], case["gz"])
    params = _params(ctx, s["cam"]["cam"], s["w"], s["h"], grid)
    cull = hd.LightCullPass(ctx, s["w"], s["h"], clusters=params, pool_cap=1 << 21)
    cull.prepare(ds)
    c = cull.cgrid
    n = c.ncell
    lists = [_tensor(c.counts, (n,), "<i4"), _tensor(c.offsets, (n,), "<i4"), _tensor(c.pool, (c.pool_cap,), "<i4")]
    return cull, lists


# --------------------------------------------------------------- frame, shadow
def _prepare_frame(case, seed):
    ctx, s = _ctx(), _scene(case, seed)
    ds = _device_scene(s)
    if case["grid"] == "tiles":
        cull = hd.LightCullPass(ctx, s["w"], s["h"])
        cull.prepare(ds)
        n = cull.tiles.ntx * cull.tiles.nty
        lists = [_tensor(cull.tiles.counts, (n,), "<i4"), _tensor(cull.tiles.lists, (n, 64), "<i4")]
    else:
        cull, lists = _cluster_cull(ctx, s, case, ds)
    f16 = case["out"] == "f16"
    shade = hd.DeferredLightPass(ctx, s["w"], s["h"], abi.HL_FMT_RGBA16_FLOAT if f16 else abi.HL_FMT_RGBA32_FLOAT)
    shade.prepare(ds)
    out = _tensor(shade.out, (s["h"], s["w"], 4), "<f2" if f16 else "<f4")
    return dict(kind="frame", ds=ds, cull=cull, grid=cull.publish(), shade=shade, outputs=[out, lists])


def _run_frame(st):
    st["cull"].execute(st["ds"])
    st["shade"].execute(st["ds"], st["grid"], flags=abi.HL_SHADE_LIGHTS_FROM_CULL)
    return st["outputs"]


def _exact_frame(case, seed):
    s = _scene(case, seed)
    px = _pixels(s)
    li = _lights64(s["lights"])
    cand = _tile_lists(s, li) if case["grid"] == "tiles" else None
    lo = _lit(px, li, cand)
    rgba = torch.cat([lo + _ambient(px), px["alpha"][..., None]], -1)
    return [_untile(torch.where(px["live"][..., None], rgba, torch.zeros_like(rgba)), s), None]


def _casters(case, s):
    """The first lights as shadow casters (a sun, points, spots) and their maps."""
    rec, rng = s["lights"]["records"], s["rng"]
    npt, nsp, size = case["points"], case["spotcasters"], case["atlas"]
    faces = ((1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1))
    sun = _unit(np.array((0.35, -1.0, 0.25)))
    rec[0]["light_type"], rec[0]["shadow_index"] = abi.HL_LIGHT_DIRECTIONAL, 0
    rec[0]["direction_outer"], rec[0]["color_intensity"] = (*sun, 0.0), (1.0, 0.95, 0.85, 1.5)
    mats = []
    for k in range(4):
        v = _look(s["cam"]["eye"] - 500.0 * sun, sun)[0]
        p = np.diag([1 / CSM[k], 1 / CSM[k], -1e-3, 1.0])
        mats.append(p @ v)
    for i in range(1, 1 + npt + nsp):
        pos, r = rec[i]["position_range"][:3].astype(float), float(rec[i]["position_range"][3])
        rec[i]["shadow_index"] = len(mats)
        if i <= npt:
            rec[i]["light_type"] = abi.HL_LIGHT_POINT
            mats += [_persp(1.0, 1.0, 0.05, r) @ _look(pos, f)[0] for f in faces]
        else:
            d = rng.normal(size=3)
            d[1] = -abs(d[1]) - 0.5
            outer = math.radians(rng.uniform(25.0, 45.0))
            rec[i]["light_type"], rec[i]["inner_angle"] = abi.HL_LIGHT_SPOT, math.cos(0.8 * outer)
            rec[i]["direction_outer"] = (*_unit(d), math.cos(outer))
            t = 1 / math.tan(outer + math.radians(5.0))
            mats.append(_persp(t, t, 0.05, r) @ _look(pos, d)[0])
    c = (torch.arange(size, device=DEV, dtype=F32) + 0.5) / size * 2 - 1
    nx, ny = c[None, :].expand(size, size), -c[:, None].expand(size, size)
    atlas = torch.empty(2, len(mats), size, size, device=DEV, dtype=F32)
    lo, hi, _ = s["field"]
    for k, m in enumerate(mats):
        inv = np.linalg.inv(m)

        def at(z):
            p = [float(inv[r, 0]) * nx + float(inv[r, 1]) * ny + float(inv[r, 2] * z + inv[r, 3]) for r in range(4)]
            return [v / p[3] for v in p[:3]]
        a, b = at(0.0), at(1.0)
        d = [y - x for x, y in zip(a, b)]
        for j in range(2):  # dynamic: every other box; static: the rest and the ground
            t, _, _ = _hits(a, d, lo, hi, step=2, first=1 - j, ground=j == 1)
            p = [x + torch.where(t < 1, t, torch.ones_like(t)) * y for x, y in zip(a, d)]
            z, w = (float(m[r, 0]) * p[0] + float(m[r, 1]) * p[1] + float(m[r, 2]) * p[2] + float(m[r, 3])
                    for r in (2, 3))
            atlas[j, k] = torch.where(t < 1, (z / w).clamp(0, 1), torch.ones_like(t))
    mats = torch.tensor(np.stack([m.T.ravel() for m in mats]), device=DEV, dtype=F32)
    return atlas[0].contiguous(), atlas[1].contiguous(), mats


# ShadowConfig presets: (filter radius, PCSS light size) per cascade, PCSS, blocker / filter / PCF samples
_QUALITY = {"medium": (((1.5, 0.0), (2.0, 0.0), (2.5, 0.0), (3.5, 0.0)), 0, 8, 8, 12),
            "high": (((2.0, 2.0), (2.5, 4.0), (3.0, 8.0), (4.0, 16.0)), 1, 8, 16, 12)}


def _rc_atlas(g):
    """A smooth radiance-cascade probe atlas: 16^3 probes of 4 x 4 directions."""
    base = _rand(g, 3, 4, 4, hi=0.6)
    i = torch.arange(16, device=DEV, dtype=F32)
    wave = 0.4 * i[:, None, None] + 0.3 * i[None, :, None] + 0.5 * i[None, None, :]  # [px, py, pz]
    t = torch.ones(16, 16, 4, 16, 4, 4, device=DEV, dtype=F32)  # [py, pz, dy, px, dx, rgba]
    for c in range(3):
        v = 0.5 + 0.5 * torch.sin(wave + c)
        t[..., c] = base[c].T[None, None, :, None, :] * v.permute(1, 2, 0)[:, :, None, :, None]
    return t.reshape(1024, 64, 4).half().contiguous()


def _rc_box(g, half):
    g.rc_world_min[:], g.rc_world_max[:], g.has_rc_gi = (-half, -1.0, -half, 0.0), (half, 0.3 * half, half, 0.0), 1


def _texture(t, fmt, texel):
    d = abi.hl_texture()
    d.data_d, d.pitch_bytes, d.format = t.data_ptr(), t.shape[1] * texel, fmt
    return d


class _Desc:
    def __init__(self, desc, *keep):
        self.desc, self.keep = desc, keep


def _prepare_shadow(case, seed):
    ctx, s = _ctx(), _scene(case, seed)
    maps = _casters(case, s)
    ds = _device_scene(s)
    casc, pcss, nb, nf, npcf = _QUALITY[case["quality"]]
    d = abi.hl_shadow_maps()
    d.atlas_d, d.static_atlas_d, d.matrices_d = (m.data_ptr() for m in maps)
    d.num_layers, d.atlas_size = maps[0].shape[0], case["atlas"]
    for k, (radius, size) in enumerate(casc):
        d.config.cascades[k].filter_radius, d.config.cascades[k].pcss_light_size = radius, size
        d.config.cascades[k].split_distance = CSM[k]
    d.config.enable_pcss, d.config.pcss_blocker_samples = pcss, nb
    d.config.pcss_filter_samples, d.config.pcf_sample_count = nf, npcf
    rc = None
    if case["rc"]:
        atlas = _rc_atlas(s["g"])
        _rc_box(ds.host.globals, case["half"])
        rc = _Desc(_texture(atlas, abi.HL_FMT_RGBA16_FLOAT, 8), atlas)
    cull, lists = _cluster_cull(ctx, s, case, ds)
    shade = hd.DeferredLightPass(ctx, s["w"], s["h"])
    shade.prepare(ds)
    out = _tensor(shade.out, (s["h"], s["w"], 4))
    return dict(kind="shadow", ds=ds, cull=cull, grid=cull.publish(), shade=shade, maps=_Desc(d, maps), rc=rc,
                outputs=[out, lists])


def _run_shadow(st):
    st["cull"].execute(st["ds"])
    st["shade"].execute(st["ds"], st["grid"], flags=abi.HL_SHADE_LIGHTS_FROM_CULL, shadows=st["maps"], rc=st["rc"])
    return st["outputs"]


# ------------------------------------------------------------------- reflect
def _cubes(n, face, mips, g):
    """n smooth pre-filtered cubes, RGBA16F: cubes, then mips, then faces +X -X +Y -Y +Z -Z."""
    tint, k, ph = _rand(g, n, 3, lo=0.3, hi=1.5), _rand(g, n, 3, lo=1.0, hi=3.0), _rand(g, n, 3, hi=6.28)
    parts = []
    for m in range(mips):
        r = max(1, face >> m)
        c = (torch.arange(r, device=DEV, dtype=F32) + 0.5) / r * 2 - 1
        tc, sc = torch.meshgrid(c, c, indexing="ij")
        o = torch.ones_like(sc)
        d = torch.stack([torch.stack(v, -1) for v in ((o, -tc, -sc), (-o, -tc, sc), (sc, o, tc), (sc, -o, -tc),
                                                      (sc, -tc, o), (-sc, -tc, -o))])
        d = d / d.norm(dim=-1, keepdim=True)
        v = tint[:, None, None, None] * (0.55 + 0.45 * torch.sin(
            k[:, None, None, None] * d + d.roll(-1, -1) + ph[:, None, None, None])) * (1 - 0.06 * m)
        parts.append(torch.cat([v, torch.ones_like(v[..., :1])], -1).reshape(n, -1))
    return torch.cat(parts, 1).half().contiguous()


def _reflect_inputs(case, seed):
    s = _scene(case, seed)
    g, rng, w, h = s["g"], s["rng"], s["w"], s["h"]
    nb, n = case["boxes"], case["boxes"] + case["spheres"]
    caps = np.zeros(n, abi.CAPTURE_DTYPE)
    half = case["half"]
    for i in range(n):
        p = np.array((rng.uniform(-0.7, 0.7) * half, rng.uniform(0.5, 4.0), rng.uniform(-0.7, 0.9) * half))
        c = caps[i]
        c["cubemap_index"], c["brightness"] = i + 1, rng.uniform(0.6, 1.4)
        if i < nb:
            yaw, ext = rng.uniform(0, 2 * math.pi), rng.uniform((3.0, 2.0, 3.0), (10.0, 6.0, 10.0))
            rot = np.array([[math.cos(yaw), 0, math.sin(yaw)], [0, 1, 0], [-math.sin(yaw), 0, math.cos(yaw)]])
            m = np.eye(4)
            m[:3, :3], m[:3, 3] = rot.T, -rot.T @ p
            c["position_radius"], c["world_to_local"] = (*p, np.linalg.norm(ext)), m.T.ravel()
            c["extents_transition"], c["shape"] = (*ext, rng.uniform(0.5, 2.5)), abi.HL_CAPTURE_SHAPE_BOX
        else:
            c["position_radius"], c["world_to_local"] = (*p, rng.uniform(4.0, 14.0)), np.eye(4).ravel()
            c["shape"] = abi.HL_CAPTURE_SHAPE_SPHERE
    caps = caps[np.argsort(caps["position_radius"][:, 3], kind="stable")]  # smallest first
    cubes = _cubes(n + 1, case["face"], case["mips"], g)
    yy, xx = torch.meshgrid(torch.arange(h, device=DEV, dtype=F32), torch.arange(w, device=DEV, dtype=F32),
                            indexing="ij")
    a = (torch.sin(xx * 0.013) * torch.cos(yy * 0.017) * 1.5).clamp(0, 1)
    ssr = torch.cat([_rand(g, h, w, 3, hi=2.0), a[..., None]], -1).half().contiguous()
    up = (s["planes"]["normal"][..., 1:2].to(F32) > 0.9).to(F32)
    planar = torch.cat([_rand(g, h, w, 3, hi=1.5) * up, 0.6 * up], -1).half().contiguous()
    return s, caps, cubes, ssr, planar, _rc_atlas(g) if case["rc"] else None


def _prepare_reflect(case, seed):
    ctx = _ctx()
    s, caps, cubes, ssr, planar, rc = _reflect_inputs(case, seed)
    ds = _device_scene(s)
    gl = ds.host.globals
    gl.reflection_capture_count, gl.enable_env_reflections = len(caps), 1
    dcaps = _upload(caps.tobytes())
    r = abi.hl_reflection_inputs()
    r.env.data_d, r.env.face_size, r.env.mip_levels = cubes.data_ptr(), case["face"], case["mips"]
    r.env.num_cubes, r.env.format = len(cubes), abi.HL_FMT_RGBA16_FLOAT
    r.captures_d = dcaps.data_ptr()
    r.ssr, r.planar = (_texture(t, abi.HL_FMT_RGBA16_FLOAT, 8) for t in (ssr, planar))
    if rc is not None:
        r.rc_cascade0 = _texture(rc, abi.HL_FMT_RGBA16_FLOAT, 8)
        _rc_box(gl, case["half"])
    refl = _Desc(None, cubes, dcaps, ssr, planar, rc)
    refl.inputs = r
    cull, lists = _cluster_cull(ctx, s, case, ds)
    shade = hd.DeferredLightPass(ctx, s["w"], s["h"])
    shade.prepare(ds)
    out = _tensor(shade.out, (s["h"], s["w"], 4))
    return dict(kind="reflect", ds=ds, cull=cull, grid=cull.publish(), shade=shade, refl=refl,
                rp=hd.ReflectionPass(ctx), outputs=[out, lists])


def _run_reflect(st):
    _run_frame(st)
    st["rp"].execute(st["ds"], st["refl"], st["shade"].out)
    return st["outputs"]


# ---------------------------------------------------------------------- pack
def _pack_inputs(case, seed):
    g, w, h = _gen(seed), case["w"], case["h"]
    alb, orm = _rand(g, h, w, 4), _rand(g, h, w, 4)
    orm[..., 2] = (orm[..., 2] < 0.3).to(F32)
    n = torch.randn(h, w, 4, generator=g, device=DEV, dtype=F32)
    n = n / n[..., :3].norm(dim=-1, keepdim=True)
    emi = _rand(g, h, w, 4, hi=2.0) * (_rand(g, h, w, 1) < 0.1)
    f0 = _rand(g, h, w, 4, lo=0.02, hi=0.3) if case["f0"] else None
    return alb, n, orm, emi.contiguous(), f0


def _prepare_pack(case, seed):
    ctx, w, h = _ctx(), case["w"], case["h"]
    planes = [None if p is None else _Buf(p) for p in _pack_inputs(case, seed)]
    sf = abi.hl_surface()
    sf.width, sf.height, sf.pitch_bytes = w, h, 16 * w
    sf.albedo_d, sf.normal_d, sf.orm_d, sf.emissive_d = (p.ptr for p in planes[:4])
    sf.specular_f0_d = planes[4].ptr if planes[4] else None
    fa, ta, fn, tn = FORMATS[case["fmt"]]
    types = {4: torch.uint8, 8: torch.float16, 16: F32}
    gb = abi.hl_gbuffer()
    gb.width, gb.height = w, h
    outs = []
    for name, fmt, tb in (("albedo", fa, ta), ("normal", fn, tn), ("orm", fa, ta), ("emissive", fn, tn)):
        outs.append(torch.zeros(h, w, 4, device=DEV, dtype=types[tb]))
        t = getattr(gb, name)
        t.data_d, t.pitch_bytes, t.format = outs[-1].data_ptr(), w * tb, fmt
    return dict(kind="pack", ctx=ctx, surface=sf, gbuffer=gb, planes=planes, outputs=outs)


def _run_pack(st):
    hd.pack_gbuffer(st["ctx"], st["surface"], st["gbuffer"])
    return st["outputs"]


def _exact_pack(case, seed):
    alb, n, orm, emi, f0 = (None if p is None else p.to(F64) for p in _pack_inputs(case, seed))
    m = orm[..., 2:3]
    f = f0[..., :3] if f0 is not None else (0.04 * (1 - m) + alb[..., :3] * m).clamp(0, 0.999)
    whole = case["fmt"] == "ref"
    return [None if whole else alb, torch.cat([n[..., :3], f[..., :1]], -1),
            None if whole else torch.cat([orm[..., :3], f[..., 1:2]], -1), torch.cat([emi[..., :3], f[..., 2:]], -1)]


# ------------------------------------------------------------------- forward
def _forward_inputs(case, seed):
    """Every surface of the frame as one fragment, in 8x8-pixel blocks, and the lights' transforms."""
    s = _scene(case, seed)
    w, h = s["w"], s["h"]
    p, cam = s["planes"], s["cam"]
    yy, xx = torch.meshgrid(torch.arange(h, device=DEV), torch.arange(w, device=DEV), indexing="ij")
    world = _world(s)
    frag = torch.zeros(h, w, 20, device=DEV, dtype=F32)
    frag[..., 0:3] = world.to(F32)
    frag[..., 3] = (xx | (yy << 16)).to(torch.int32).view(F32)
    frag[..., 4:7] = p["normal"][..., :3]
    frag[..., 7] = 0.5
    frag[..., 8:11], frag[..., 11] = p["albedo"][..., :3], p["orm"][..., 0]
    frag[..., 12], frag[..., 13], frag[..., 14] = p["normal"][..., 3], p["orm"][..., 3], p["emissive"][..., 3]
    frag[..., 15], frag[..., 16:19], frag[..., 19] = p["orm"][..., 1], p["emissive"][..., :3], p["orm"][..., 2]
    key = ((yy // 8) * ((w + 7) // 8) + xx // 8) * 64 + (yy % 8) * 8 + xx % 8
    live = p["depth"] < 1
    frag = frag[live][key[live].argsort()].contiguous()
    li, g = s["lights"], s["g"]
    n = len(li["range"])
    rot = _rand(g, n, 3, lo=-180.0, hi=180.0)
    entity = torch.randperm(2 * n + 3, generator=g, device=DEV)[:n]
    tr = torch.zeros(2 * n + 3, 9, device=DEV, dtype=F32)
    tr[:, 6:] = 1.0
    tr[entity, 0:3], tr[entity, 3:6] = li["pos"], rot
    r = torch.deg2rad(rot.to(F64))
    cx, sx, cy, sy = torch.cos(r[:, 0]), torch.sin(r[:, 0]), torch.cos(r[:, 1]), torch.sin(r[:, 1])
    dir64 = -torch.stack([sy * cx, -sx, cy * cx], -1)  # -Z under yaw, pitch, roll
    fields = {k: v for k, v in li.items() if k != "records"}
    s["lights"] = _light_records(dict(fields, dir=dir64.to(F32)))
    return s, frag, entity.to(torch.int32), tr, dir64, cam


def _prepare_forward(case, seed):
    ctx = _ctx()
    s, frag, entity, tr, _, _ = _forward_inputs(case, seed)
    ds = _device_scene(s)
    cull, lists = _cluster_cull(ctx, s, case, ds)
    fwd = hd.ForwardLitPass(ctx, s["w"], s["h"])
    g = abi.ForwardLitGlobals()
    g.light_count, g.ambient_intensity = len(s["lights"]["records"]), 1.0
    g.ambient_color[:] = (*AMBIENT, 1.0)
    g.num_tiles_x, g.num_tiles_y = (s["w"] + 15) // 16, (s["h"] + 15) // 16
    g.screen_width, g.screen_height = float(s["w"]), float(s["h"])
    fwd.globals = g
    n = len(frag)
    fwd.out = ctx.alloc(16 * max(n, 1))
    return dict(kind="forward", ds=ds, cull=cull, grid=cull.publish(), fwd=fwd, n=n, frag=_Buf(frag),
                entity=_Buf(entity), tr=_Buf(tr), nt=len(tr), outputs=[_tensor(fwd.out, (n, 4)), lists])


def _run_forward(st):
    st["cull"].execute(st["ds"])
    st["fwd"].execute(st["ds"], st["frag"], st["n"], st["grid"], entity=st["entity"], transforms=st["tr"],
                      num_transforms=st["nt"])
    return st["outputs"]


def _exact_forward(case, seed):
    s, frag, _, _, dir64, cam = _forward_inputs(case, seed)
    li = dict(_lights64(s["lights"]), dir=dir64)
    n = len(frag)
    pad = (-n) % 256
    f = torch.cat([frag, torch.zeros(pad, 20, device=DEV)]).to(F64).reshape(-1, 256, 20)
    live = (torch.arange(n + pad, device=DEV) < n).reshape(-1, 256)
    v = torch.tensor([cam["cam"].position_near[k] for k in range(3)], device=DEV, dtype=F64) - f[..., 0:3]
    px = dict(pos=f[..., 0:3], n=f[..., 4:7], v=v / v.norm(dim=-1, keepdim=True), albedo=f[..., 8:11],
              ao=f[..., 11], f0=f[..., 12:15], rough=f[..., 15], glow=f[..., 16:19], metal=f[..., 19], live=live)
    amb = torch.tensor(AMBIENT, device=DEV, dtype=F32).to(F64)
    out = _lit(px, li, None, cut=False) + amb * px["albedo"] * px["ao"][..., None] + px["glow"]
    out = torch.cat([out, f[..., 7:8]], -1)
    return [out.reshape(-1, 4)[:n], None]


# --------------------------------------------------------------- train, grad
def _perturbed(li, g):
    """The current guess of the lights: moved and rescaled."""
    f = {k: v for k, v in li.items() if k != "records"}
    f["pos"] = f["pos"] + 0.5 * torch.randn(f["pos"].shape, generator=g, device=DEV, dtype=F32)
    f["intensity"] = f["intensity"] * _rand(g, len(f["intensity"]), lo=0.7, hi=1.3)
    return _light_records(f)


def _train_inputs(case, seed):
    s = _scene(case, seed)
    s["lights"] = _perturbed(s["lights"], s["g"])
    h, w = s["h"], s["w"]
    # the target of the L2 loss, or the caller's dL/dradiance
    t = _rand(s["g"], h, w, 4) if case["kind"] == "train" else \
        torch.randn(h, w, 4, generator=s["g"], device=DEV, dtype=F32)
    return s, t.contiguous()


def _prepare_train(case, seed):
    ctx = _ctx()
    s, t = _train_inputs(case, seed)
    ds = _device_scene(s)
    cull, lists = _cluster_cull(ctx, s, case, ds)
    w, h, n = s["w"], s["h"], len(s["lights"]["records"])
    shade = hd.DeferredLightPass(ctx, w, h)
    shade.prepare(ds)
    grads = hd.AdjointBuffers(ctx, w, h, n)
    outs = [_tensor(grads.d_pixel, (5, h, w)), _tensor(grads.d_pos, (n, 3)), _tensor(grads.d_int, (n,))]
    if case["kind"] == "train":
        outs += [_tensor(shade.out, (h, w, 4)), _tensor(grads.loss, (1,), "<f8")]
    return dict(kind=case["kind"], ds=ds, cull=cull, grid=cull.publish(), shade=shade, grads=grads, t=_Buf(t),
                outputs=outs + [lists])


def _run_train(st):
    st["cull"].execute(st["ds"])
    if st["kind"] == "train":
        st["shade"].forward_backward_l2(st["ds"], st["grid"], st["t"], st["grads"])
    else:
        st["shade"].backward(st["ds"], st["grid"], st["t"], st["grads"])
    return st["outputs"]


def _exact_train(case, seed):
    s, t = _train_inputs(case, seed)
    px, li = _pixels(s), _lights64(s["lights"])
    return [*_adjoint64(s, px, li, t, case["kind"] == "train"), None]


def _adjoint64(s, px, li, t, fused):
    """d_pixel, d_pos, d_int (and with fused the frame and the loss), by torch's autograd in float64."""
    t = _tile(t.to(F64)[..., :3], s)
    live = px["live"][..., None]
    leaf = {k: px[k].clone().requires_grad_() for k in ("albedo", "rough", "metal")}
    lf = {k: li[k].clone().requires_grad_() for k in ("pos", "intensity")}

    def f0_of(p):
        m = p["metal"][..., None]
        return (0.04 * (1 - m) + p["albedo"] * m).clamp(0, 0.999)
    gl = t
    if fused:
        plain = dict(px, f0=f0_of(px))
        out = _lit(plain, li, None) + _ambient(plain)
        gl = torch.where(live, 2 * (out - t), torch.zeros_like(t))
    p = dict(px, **leaf)
    _lit(p, dict(li, **lf), None, grad=torch.where(live, gl, torch.zeros_like(gl)), f0_of=f0_of)
    (torch.where(live, _ambient(p), torch.zeros_like(gl)) * gl).sum().backward()
    g = torch.cat([leaf["albedo"].grad, leaf["rough"].grad[..., None], leaf["metal"].grad[..., None]], -1)
    res = [_untile(g, s).permute(2, 0, 1).contiguous(), lf["pos"].grad, lf["intensity"].grad]
    if fused:
        rgba = torch.cat([out, px["alpha"][..., None]], -1)
        res += [_untile(torch.where(live, rgba, torch.zeros_like(rgba)), s),
                torch.where(live, (out - t) ** 2, torch.zeros_like(t)).sum().reshape(1)]
    return res


# --------------------------------------------------------------------- views
def _views_inputs(case, seed):
    """Scenes of the faces (three sizes) and the two eyes over one light pool, and each view's subset."""
    g, rng = _gen(seed), np.random.default_rng(int(seed))
    half = case["half"]
    field = _field(half, g, rng, SMOOTHEST_FITTED)
    pool = _lights(case["lights"], half, 0.0, g)
    dirs = ((0, 0, -1), (0, 0, 1), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0))
    views = []
    for i in range(case["faces"] + 2):
        eye_view = i >= case["faces"]
        if eye_view:
            w, h = case["eye_w"], case["eye_h"]
            cam = _camera(w, h, (-0.032 if i == case["faces"] else 0.032, 1.7, 0.6 * half), (0.0, -0.05, -1.0), 100.0)
        else:
            if i % 6 == 0:
                probe = (rng.uniform(-0.8, 0.8) * half, rng.uniform(2.0, 15.0), rng.uniform(-0.8, 0.8) * half)
            w = h = case["size"] << (i % 3)
            cam = _camera(w, h, probe, dirs[i % 6], 90.0)
        n = min(case["lights"], case["subset"] * 4 if eye_view else max(32, case["subset"] >> (i % 4)))
        sub = torch.randperm(case["lights"], generator=g, device=DEV)[:n].sort().values
        s = dict(w=w, h=h, fmt="ref", cam=cam, planes=_gbuffer(w, h, cam, field, "ref", g), sub=sub, adjoint=eye_view)
        if eye_view:
            s["target"] = _rand(g, h, w, 4)
        views.append(s)
    return pool, views


class _Plan:
    """A captured plan and the buffers of its views."""

    def __init__(self, ctx, pool, npool, views):
        self.pool, self.views = pool, views
        self.plan = hb.BatchPlan(ctx, pool, npool, views)
        self.plan.capture()

    def __del__(self):
        self.plan.destroy()


def _prepare_views(case, seed):
    ctx = _ctx()
    pool, scenes = _views_inputs(case, seed)
    records = pool["records"]
    npool = len(records)
    buf = _Buf(_upload(records.tobytes()))
    views, outs = [], []
    for s in scenes:
        sub = s["sub"]
        ds = _device_scene(s, records, buf)
        w, h = s["w"], s["h"]
        out = torch.zeros(h, w, 4, device=DEV, dtype=F32)
        v = hb.BatchView(scene=ds, subset=_Buf(sub.to(torch.int32)), num_lights=len(sub), out=_Buf(out),
                         adjoint=s["adjoint"])
        outs.append(out)
        if s["adjoint"]:
            g = [torch.zeros(5, h, w, device=DEV), torch.zeros(npool, 3, device=DEV), torch.zeros(npool, device=DEV),
                 torch.zeros(1, device=DEV, dtype=F64)]
            v.target, v.d_pixel, v.d_pos, v.d_int, v.loss = (_Buf(t) for t in (s["target"], *g))
            outs.append(g)
        views.append(v)
    return dict(kind="views", plan=_Plan(ctx, buf, npool, views), outputs=outs)


def _run_views(st):
    st["plan"].plan.launch()
    return st["outputs"]


def _exact_views(case, seed):
    pool, scenes = _views_inputs(case, seed)
    li = _lights64(pool)
    res = []
    for s in scenes:
        px, sub = _pixels(s), {k: v[s["sub"]] for k, v in li.items()}
        if not s["adjoint"]:
            rgba = torch.cat([_lit(px, sub, None) + _ambient(px), px["alpha"][..., None]], -1)
            res.append(_untile(torch.where(px["live"][..., None], rgba, torch.zeros_like(rgba)), s))
            continue
        dpx, dpos, dint, out, loss = _adjoint64(s, px, sub, s["target"], True)
        full = [torch.zeros(case["lights"], 3, device=DEV, dtype=F64),
                torch.zeros(case["lights"], device=DEV, dtype=F64)]
        full[0][s["sub"]], full[1][s["sub"]] = dpos, dint
        res += [out, [dpx, *full, loss]]
    return res


# --------------------------------------------------- float64 reference: set-up
def _tile(t, s):
    """[h, w, ...] as 16x16-pixel tiles [tiles, 256, ...], zero-padded."""
    h, w = t.shape[:2]
    th, tw = (h + 15) // 16, (w + 15) // 16
    p = torch.zeros(th * 16, tw * 16, *t.shape[2:], device=DEV, dtype=t.dtype)
    p[:h, :w] = t
    return p.reshape(th, 16, tw, 16, *t.shape[2:]).transpose(1, 2).reshape(th * tw, 256, *t.shape[2:])


def _untile(t, s):
    th, tw = (s["h"] + 15) // 16, (s["w"] + 15) // 16
    rest = t.shape[2:]
    t = t.reshape(th, tw, 16, 16, *rest).transpose(1, 2).reshape(th * 16, tw * 16, *rest)
    return t[: s["h"], : s["w"]].contiguous()


def _matrix64(m):
    return torch.tensor(list(m), device=DEV, dtype=F64).reshape(4, 4).T


def _world(s):
    """World position of every pixel's centre from its depth."""
    w, h = s["w"], s["h"]
    m = _matrix64(s["cam"]["cam"].inv_view_proj)
    x = ((torch.arange(w, device=DEV, dtype=F64) + 0.5) / w * 2 - 1)[None, :, None]
    y = (1 - (torch.arange(h, device=DEV, dtype=F64) + 0.5) / h * 2)[:, None, None]
    q = m[:, 0] * x + m[:, 1] * y + m[:, 2] * s["planes"]["depth"].to(F64)[..., None] + m[:, 3]
    return q[..., :3] / q[..., 3:]


def _pixels(s):
    p = {k: (v.to(F64) / 255 if v.dtype == torch.uint8 else v.to(F64)) for k, v in s["planes"].items()}
    pos = _world(s)
    v = torch.tensor([s["cam"]["cam"].position_near[k] for k in range(3)], device=DEV, dtype=F64) - pos
    n = p["normal"][..., :3]
    one = dict(pos=pos, v=v / v.norm(dim=-1, keepdim=True), n=n / n.norm(dim=-1, keepdim=True),
               albedo=p["albedo"][..., :3], alpha=p["albedo"][..., 3], ao=p["orm"][..., 0], rough=p["orm"][..., 1],
               metal=p["orm"][..., 2], glow=p["emissive"][..., :3], live=s["planes"]["depth"] < 1,
               f0=torch.stack([p["normal"][..., 3], p["orm"][..., 3], p["emissive"][..., 3]], -1).clamp(0, 0.999))
    return {k: _tile(t, s) for k, t in one.items()}


def _lights64(li):
    return {k: v.to(F64) for k, v in li.items() if k != "records"}


def _ambient(px):
    sky = torch.tensor(AMBIENT, device=DEV, dtype=F32).to(F64)
    ht = px["n"][..., 1:2] * 0.5 + 0.5
    return (sky * 0.15 * (1 - ht) + sky * ht) * px["albedo"] * px["ao"][..., None] + px["glow"]


# -------------------------------------------------- float64 reference: lights
def _dot(a, b):
    return (a * b).sum(-1)


def _term(p, l, cut):
    """The light's contribution to the pixel, both given pair by pair."""
    to = l["pos"] - p["pos"]
    d2 = _dot(to, to)
    d = d2.sqrt()
    L = to / d[..., None]
    att = (1 - (d / l["range"]) ** 4).clamp(min=0) / (d2 + 0.0001)
    cos = -_dot(L, l["dir"])
    spot = ((cos - l["outer"]) / (l["inner"] - l["outer"])).clamp(0, 1)
    att = torch.where(l["kind"] == abi.HL_LIGHT_SPOT, att * spot * spot * (3 - 2 * spot), att)
    rad = l["color"] * (l["intensity"] * att)[..., None]
    ndl = _dot(p["n"], L).clamp(min=0)
    keep = (d <= l["range"]) & (ndl > 0)
    if cut:
        keep = keep & (rad >= 0.002).any(-1)
    H = p["v"] + L
    H = H / H.norm(dim=-1, keepdim=True)
    ndv = _dot(p["n"], p["v"]).clamp(min=0)
    ndh, hdv = _dot(p["n"], H).clamp(min=0), _dot(H, p["v"]).clamp(min=0)
    a2 = p["rough"] ** 4
    den = ndh * ndh * (a2 - 1) + 1
    D = a2 / (math.pi * den * den + 0.0001)
    k = (p["rough"] + 1) ** 2 / 8
    G = ndv / (ndv * (1 - k) + k + 0.0001) * ndl / (ndl * (1 - k) + k + 0.0001)
    F = p["f0"] + (1 - p["f0"]) * ((1 - hdv).clamp(0, 1) ** 5)[..., None]
    spec = (D * G / (4 * ndv * ndl + 0.0001))[..., None] * F
    kd = (1 - F) * (1 - p["metal"][..., None])
    o = (kd * p["albedo"] / math.pi + spec) * rad * ndl[..., None]
    return torch.where(keep[..., None], o, torch.zeros_like(o))


_PIXEL = ("pos", "n", "v", "albedo", "rough", "metal", "f0")


def _lit(px, li, cand, cut=True, grad=None, f0_of=None):
    """Sum of the lights over tiled pixels.  cand: each tile's light indices (-1: none) where the lists are
    capped, else every light in reach counts.  grad: backpropagate this dL/dout instead of returning the sum."""
    T = px["live"].shape[0]
    out = torch.zeros(T * 256, 3, device=DEV, dtype=F64)
    flat = {k: px[k].reshape(T * 256, *px[k].shape[2:]) for k in _PIXEL if k in px}
    live = px["live"].reshape(-1)
    if cand is None:
        inf = torch.full((), math.inf, device=DEV, dtype=F64)
        lo = torch.where(px["live"][..., None], px["pos"], inf).amin(1)
        hi = torch.where(px["live"][..., None], px["pos"], -inf).amax(1)
        lo, hi = (torch.where(px["live"].any(1)[:, None], b, inf) for b in (lo, hi))  # no pixel: far away
    with torch.no_grad():
        pos, rng = li["pos"].detach(), li["range"]
        tiles, lights = [], []
        step = max(1, (1 << 25) // max(1, len(rng)))
        for t0 in range(0, T, step):
            if cand is None:
                d2 = sum((torch.maximum(lo[t0:t0 + step, a, None] - pos[:, a], pos[:, a] - hi[t0:t0 + step, a, None])
                          .clamp(min=0)) ** 2 for a in range(3))
                t, i = (d2 <= (rng * 1.001) ** 2).nonzero(as_tuple=True)
            else:
                t, j = (cand[t0:t0 + step] >= 0).nonzero(as_tuple=True)
                i = cand[t0:t0 + step][t, j]
            tiles.append(t + t0)
            lights.append(i)
        tiles, lights = torch.cat(tiles), torch.cat(lights)
    lane = torch.arange(256, device=DEV)
    for c0 in range(0, len(tiles), 1 << 15):
        with torch.no_grad():
            p = (tiles[c0:c0 + (1 << 15), None] * 256 + lane).reshape(-1)
            i = lights[c0:c0 + (1 << 15), None].expand(-1, 256).reshape(-1)
            to = pos[i] - flat["pos"][p].detach()
            on = (_dot(to, to) <= (rng[i] * 1.001) ** 2) & live[p]
            p, i = p[on], i[on]
        if not len(p):
            continue
        a = {k: v[p] for k, v in flat.items()}
        if f0_of is not None:
            a["f0"] = f0_of(a)
        o = _term(a, {k: v[i] for k, v in li.items()}, cut)
        if grad is None:
            out.index_add_(0, p, o)
        else:
            (o * grad.reshape(-1, 3)[p]).sum().backward(retain_graph=True)
    return out.reshape(T, 256, 3)


def _tile_lists(s, li):
    """The reference's tile lists: the first 64 lights whose sphere touches the tile's four lateral planes."""
    w, h = s["w"], s["h"]
    tw, th = (w + 15) // 16, (h + 15) // 16
    cam = s["cam"]["cam"]
    view = _matrix64(cam.view)
    c = li["pos"] @ view[:3, :3].T + view[:3, 3]
    p00, p11 = float(cam.proj[0]), float(cam.proj[5])

    def inside(e, axis, scale, sign):
        """sphere against the plane through the eye and the NDC edge e (one row per edge)"""
        s_ = torch.sqrt(1 + (e / scale) ** 2)
        return sign * (c[:, axis] + (e / scale)[:, None] * c[:, 2]) / s_[:, None] >= -li["range"]
    x = torch.arange(tw + 1, device=DEV, dtype=F64) * 16 / w * 2 - 1
    y = 1 - torch.arange(th + 1, device=DEV, dtype=F64) * 16 / h * 2
    x, y = x.clamp(max=1.0), y.clamp(min=-1.0)
    col = inside(x[:-1], 0, p00, 1.0) & inside(x[1:], 0, p00, -1.0)
    row = inside(y[:-1], 1, p11, -1.0) & inside(y[1:], 1, p11, 1.0)
    n = len(li["range"])
    cand = torch.full((th, tw, 65), -1, device=DEV, dtype=torch.int64)
    for r in range(th):
        both = col & row[r]
        at = both.cumsum(1, dtype=torch.int32) - 1
        t, i = (both & (at < 64)).nonzero(as_tuple=True)
        cand[r, t, at[t, i].long()] = i
    return cand.reshape(th * tw, 65)[:, :min(64, n)]


# ----------------------------------------------- float64 reference: reflections
def _smooth(e0, e1, x):
    t = ((x - e0) / (e1 - e0)).clamp(0, 1)
    return t * t * (3 - 2 * t)


def _rc64(atlas, half, p, n):
    """Cosine-weighted probe radiance around n at p, trilinear between the probes of the box."""
    lo = torch.tensor((-half, -1.0, -half), device=DEV, dtype=F32).to(F64)
    size = torch.tensor((half, 0.3 * half, half), device=DEV, dtype=F32).to(F64) - lo
    t = (p - lo) / size
    fade = (_smooth(0.0, 0.05, t) * _smooth(1.0, 0.95, t)).prod(-1)
    i = (torch.arange(4, device=DEV, dtype=F64) + 0.5) / 4 * 2 - 1
    fx, fy = i[:, None].expand(4, 4), i[None, :].expand(4, 4)  # [dx, dy]
    y = 1 - fx.abs() - fy.abs()
    ox = torch.where(y < 0, (1 - fy.abs()) * fx.sign(), fx)
    oz = torch.where(y < 0, (1 - fx.abs()) * fy.sign(), fy)
    d = torch.stack([ox, y, oz], -1)
    d = d / d.norm(dim=-1, keepdim=True)
    wgt = torch.einsum("pc,xyc->pxy", n, d).clamp(min=0)
    wgt = torch.where(wgt > 0.001, wgt, torch.zeros_like(wgt))
    wgt = (wgt / wgt.sum((1, 2), keepdim=True).clamp(min=0.001)).reshape(-1, 16)
    probes = atlas.to(F64)[..., :3].reshape(16, 16, 4, 16, 4, 3).permute(3, 0, 1, 4, 2, 5).reshape(-1, 16, 3)
    f = (t * 16 - 0.5).clamp(0, 15)
    b, q = f.floor().long(), f - f.floor()
    out = torch.zeros_like(p)
    for k in range(8):
        o = torch.tensor(((k >> 2) & 1, (k >> 1) & 1, k & 1), device=DEV)
        c = (b + o).clamp(max=15)
        m = torch.where(o.bool(), q, 1 - q).prod(-1)
        probe = probes[(c[:, 0] * 16 + c[:, 1]) * 16 + c[:, 2]]
        out = out + m[:, None] * torch.einsum("pk,pkc->pc", wgt, probe)
    return out * fade[:, None]


def _cube64(cubes, face, mips, cube, d, lod):
    """Trilinear sample of RGBA16F cube array, clamped to the face that the major axis selects."""
    a = d.abs()
    isx = (a[:, 0] >= a[:, 1]) & (a[:, 0] >= a[:, 2])
    isy = ~isx & (a[:, 1] >= a[:, 2])
    x, y, z = d.unbind(-1)
    side = torch.where(isx, torch.where(x >= 0, 0, 1), torch.where(isy, torch.where(y >= 0, 2, 3),
                                                                  torch.where(z >= 0, 4, 5)))
    ma = torch.where(isx, a[:, 0], torch.where(isy, a[:, 1], a[:, 2]))
    sc = torch.where(isx, torch.where(x >= 0, -z, z), torch.where(isy, x, torch.where(z >= 0, x, -x)))
    tc = torch.where(isy, torch.where(y >= 0, z, -z), -y)
    u, v = (sc / ma + 1) / 2, (tc / ma + 1) / 2
    res = [max(1, face >> m) for m in range(mips)]
    off = torch.tensor([0] + list(np.cumsum([6 * r * r for r in res])), device=DEV)
    rt = torch.tensor(res, device=DEV)
    lod = lod.clamp(0, mips - 1)
    m0 = lod.floor().long()
    m1 = (m0 + 1).clamp(max=mips - 1)
    tex = cubes.reshape(len(cubes), -1, 4)

    def at(m):
        r = rt[m]
        gx, gy = u * r - 0.5, v * r - 0.5
        x0, y0 = gx.floor(), gy.floor()
        wx, wy = (gx - x0)[:, None], (gy - y0)[:, None]

        def texel(xi, yi):
            xi, yi = (torch.minimum(k.long().clamp(min=0), r - 1) for k in (xi, yi))
            return tex[cube, off[m] + (side * r + yi) * r + xi][:, :3].to(F64)
        return (texel(x0, y0) * (1 - wx) + texel(x0 + 1, y0) * wx) * (1 - wy) + \
               (texel(x0, y0 + 1) * (1 - wx) + texel(x0 + 1, y0 + 1) * wx) * wy
    t = (lod - m0)[:, None]
    return at(m0) * (1 - t) + at(m1) * t


def _exact_reflect(case, seed):
    s, caps, cubes, ssr, planar, rc = _reflect_inputs(case, seed)
    px = _pixels(s)
    lit = torch.cat([_lit(px, _lights64(s["lights"]), None) + _ambient(px), px["alpha"][..., None]], -1)
    lit = torch.where(px["live"][..., None], lit, torch.zeros_like(lit))
    live = px["live"].reshape(-1)
    p, n, v = (px[k].reshape(-1, 3)[live] for k in ("pos", "n", "v"))
    rough, ao, f0 = px["rough"].reshape(-1)[live], px["ao"].reshape(-1)[live], px["f0"].reshape(-1, 3)[live]
    ssr, planar = (_tile(t.to(F64), s).reshape(-1, 4)[live] for t in (ssr, planar))
    ndv = _dot(n, v).clamp(min=0)
    fi = f0 + (torch.maximum(1 - rough[:, None], f0) - f0) * ((1 - ndv).clamp(0, 1) ** 5)[:, None]
    R = 2 * _dot(n, v)[:, None] * n - v
    acc, cover = torch.zeros_like(p), torch.zeros_like(rough)

    def sample(cube, d, lod):
        return _cube64(cubes, case["face"], case["mips"], cube, d, lod)
    for c in caps:
        centre, r = (torch.tensor(c["position_radius"][k], device=DEV).to(F64) for k in (slice(0, 3), 3))
        if c["shape"] == abi.HL_CAPTURE_SHAPE_BOX:
            m = torch.tensor(c["world_to_local"], device=DEV).to(F64).reshape(4, 4).T
            e = torch.tensor(c["extents_transition"], device=DEV).to(F64)
            pl, rl = p @ m[:3, :3].T + m[:3, 3], R @ m[:3, :3].T
            gap = e[:3] - pl.abs()
            wgt = torch.where((gap < 0).any(-1), torch.zeros_like(rough),
                              (gap.amin(-1) / e[3].clamp(min=1e-4)).clamp(0, 1))
            t = torch.maximum((-e[:3] - pl) / rl, (e[:3] - pl) / rl).amin(-1)
        else:
            o = p - centre
            dist = o.norm(dim=-1)
            wgt = torch.where(dist > r, torch.zeros_like(rough), ((r - dist) / (r * 0.1).clamp(min=1e-4)).clamp(0, 1))
            b = _dot(o, R)
            disc = b * b - (_dot(o, o) - r * r)
            t = torch.where(disc < 0, torch.full_like(b, -1.0), -b + disc.clamp(min=0).sqrt())
        ok = (wgt > 0) & (cover < 0.999)
        d = torch.where((t > 0)[:, None], p + R * t[:, None] - centre, R)[ok]
        col = sample(int(c["cubemap_index"]), d, rough[ok] * 8) * float(c["brightness"])
        add = wgt[ok] * (1 - cover[ok])
        acc[ok] += col * add[:, None]
        cover[ok] += add
    open_ = cover < 0.999
    acc[open_] += sample(0, R[open_], rough[open_] * 8) * (1 - cover[open_])[:, None]
    r4 = [rough * a + b for a, b in ((-1.0, 1.0), (-0.0275, 0.0425), (-0.572, 1.04), (0.022, -0.04))]
    a004 = torch.minimum(r4[0] * r4[0], torch.exp2(-9.28 * ndv)) * r4[0] + r4[1]
    spec = acc * (f0 * (-1.04 * a004 + r4[2])[:, None] + (1.04 * a004 + r4[3])[:, None])
    for img in (ssr, planar):
        spec = spec * (1 - img[:, 3:]) + img[:, :3] * fi * img[:, 3:]
    if rc is not None:
        t = rough[:, None] * 0.5
        L = R * (1 - t) + n * t
        mix = torch.where(rough > 0.6, _smooth(0.6, 0.9, rough) * 0.4, torch.zeros_like(rough))[:, None]
        glossy = torch.cat([_rc64(rc, case["half"], p[k], (L / L.norm(dim=-1, keepdim=True))[k])
                            for k in torch.arange(len(p), device=DEV).split(1 << 19)])
        spec = spec * (1 - mix) + glossy * mix
    add = torch.zeros(live.numel(), 4, device=DEV, dtype=F64)
    add[live, :3] = spec * ao[:, None]
    return [_untile(lit + add.reshape(-1, 256, 4), s), None]


# ------------------------------------------------------------------ interface
_PREPARE = dict(frame=_prepare_frame, shadow=_prepare_shadow, reflect=_prepare_reflect, pack=_prepare_pack,
                forward=_prepare_forward, train=_prepare_train, grad=_prepare_train, views=_prepare_views)
_RUN = dict(frame=_run_frame, shadow=_run_shadow, reflect=_run_reflect, pack=_run_pack, forward=_run_forward,
            train=_run_train, grad=_run_train, views=_run_views)
# shadow: the taps' rotation is a hash of the pixel's coordinates and every tap
# a comparison, so the frame has no value in 64 bits to be near to
_EXACT = dict(frame=_exact_frame, reflect=_exact_reflect, pack=_exact_pack, forward=_exact_forward,
              train=_exact_train, grad=_exact_train, views=_exact_views)


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, int(seed))


def run(state):
    return _RUN[state["kind"]](state)


def exact(case, seed):
    f = _EXACT.get(case["kind"])
    return f(case, int(seed)) if f else None


def _reach(case, lights):
    """Lights in reach of a surface point on the ground, on average."""
    half = case["half"]
    lo, hi = (2.0, 10.0) if half <= 40 else (1.0, 8.0)
    cube = (hi ** 4 - lo ** 4) / (4 * (hi - lo))
    return lights * (2.0 / 3.0) * math.pi * cube / (4 * half * half * max(10.0, 0.3 * half))


def work(case):
    """Inputs read once and outputs written once; 60 flops per pixel and 130 per pixel and light in reach
    (three times that with the adjoint)."""
    kind = case["kind"]
    if kind == "views":
        px = sum((case["size"] << (i % 3)) ** 2 for i in range(case["faces"]))
        eyes = 2 * case["eye_w"] * case["eye_h"]
        near = _reach(case, case["subset"] / 2)
        return {"bytes": px * 44.0 + eyes * (44.0 + 16 + 20) + case["lights"] * (56.0 + 32),
                "flops": px * (60 + 130 * near) + eyes * (60 + 390 * 8 * near)}
    px = float(case["w"] * case["h"])
    if kind == "pack":
        _, ta, _, tn = FORMATS[case["fmt"]]
        return {"bytes": px * (64 + (16 if case["f0"] else 0) + 2 * ta + 2 * tn), "flops": px * 24}
    _, ta, _, tn = FORMATS[case.get("fmt", "f32")]
    texels = 2 * ta + 2 * tn + 4
    n = case["lights"]
    near = _reach(case, n)
    if kind == "reflect":
        return {"bytes": px * (texels + 16 + 16) + n * 56,
                "flops": px * (60 + 130 * near + 400 + (500 if case["rc"] else 0))}
    if kind == "forward":
        return {"bytes": px * 96 + n * 100, "flops": px * (60 + 130 * near)}
    if kind in ("train", "grad"):
        return {"bytes": px * (texels + 16 + 20 + (16 if kind == "train" else 0)) + n * 72,
                "flops": px * (60 + 390 * near)}
    if kind == "shadow":
        layers = 4 + 6 * case["points"] + case["spotcasters"]
        return {"bytes": px * (texels + 16) + n * 56 + 8.0 * layers * case["atlas"] ** 2 * 0.1,
                "flops": px * (60 + 130 * near + 24 * 60 + (900 if case["rc"] else 0))}
    return {"bytes": px * (texels + (8 if case["out"] == "f16" else 16)) + n * 56,
            "flops": px * (60 + 130 * min(near, 64 if case["grid"] == "tiles" else near))}
