"""Timed cases of the voxel GI path: what a program has it do, through final184_amd.vgi.

A case is a dict of plain values; `kind` says which calls one pass makes:

  frame     voxelize + build_mips + trace of one scene (geometry that moves every frame)
  view      trace alone: a resident scene, a camera that moves
  batch     the three batched calls over scenes of uneven size
  views     one batched trace: several requests' frames over resident scenes
  screen    decode + temporal blend + blur along y + blur along x on given images
  indirect  decode + trace + temporal blend + both blurs: a frame of the reference's
            indirect chain over a resident scene

Scenes are the package's seeded generators: `soup` (small random triangles, a G-buffer of
points on them, one directional light) and `room` (walls, columns, tiles, debris, a pinhole
camera's G-buffer, four point lights). `exact` restates every stage in 64 bits on plain
torch tensors: integer voxel sums, radiance and mips without storage rounding, the cone
march and the screen passes.
"""
from __future__ import annotations

import math

import numpy as np
import torch  # before the package: both then share one HIP runtime

from final184_amd import scenegen as sg
from final184_amd import vgi

TILES = {"8x8": (8, 8, vgi.ORDER_TILES), "16x16": (16, 16, vgi.ORDER_TILES), "32x8": (32, 8, vgi.ORDER_TILES),
         "morton": (16, 16, vgi.ORDER_MORTON)}


def _frame(scene, tris, n, width, height, cones, prec, tile, **more):
    c = dict(kind="frame", scene=scene, tris=tris, n=n, width=width, height=height, cones=cones, prec=prec,
             tile=tile, textured=False, shadow=False, meshes=1, index="none")
    c.update(more)
    return c


def listed():
    return [
        # the smallest whole frame (an importer's preview, a unit test): launches and host
        # work count, not throughput
        dict(_frame("soup", 2_000, 32, 64, 64, 6, "fp32", "16x16"), name="soup_32_frame"),
        # 10,000 triangles at 64^3, the package's first workload, with the default tuning
        dict(_frame("soup", 10_000, 64, 256, 256, 6, "fp32", "16x16"), name="soup_64_frame"),
        # the headline frame: 262,144 triangles, 256^3, 1080p, 9 + 1 cones, FP16 x-pair mips
        dict(_frame("room", 262_144, 256, 1920, 1080, 9, "fp16x2", "8x8"), name="room_256_1080p_frame"),
        # a lit, textured, imported room in a window of odd size: sampled albedo, shadow walks
        dict(_frame("room", 100_000, 128, 957, 541, 9, "fp16", "8x8", textured=True, shadow=True, index="u32"),
             name="room_128_textured_shadow"),
        # geometry of many primitives re-voxelized for a low-resolution light-probe pass:
        # the front end and the mips set the time
        dict(_frame("room", 262_144, 256, 96, 54, 9, "fp16x2", "8x8", meshes=48, index="u16"),
             name="room_256_probe_frame"),
        # the largest: 1,048,576 triangles, 512^3, 4K, 16 + 1 cones, FP32 mips
        dict(_frame("room", 1_048_576, 512, 3840, 2160, 16, "fp32", "8x8"), name="room_512_4k_frame"),
        # a static scene seen by a moving camera, odd window
        dict(kind="view", scene="room", tris=200_000, n=256, width=1279, height=719, cones=9, prec="fp16",
             tile="8x8", name="room_256_view"),
        # offline batches: 16 scenes of uneven size, scattered G-buffer points, Morton order
        dict(kind="batch", scenes=16, median=20_000, side=512, prec="fp16", tile="morton", name="soup_batch_16"),
        # a server's batch: frames of several requests over resident scenes
        dict(kind="views", scenes=3, frames=8, tris=60_000, n=128, width=512, height=512, prec="fp16", tile="16x16",
             name="served_views_8"),
        # the screen passes of a 1080p frame on the reference's render targets
        dict(kind="screen", width=1920, height=1080, image="rgba16f", name="screen_1080p"),
        # the same in a small window of odd size on FP32 images
        dict(kind="screen", width=643, height=361, image="rgba32f", name="screen_odd_fp32"),
        # the reference's indirect frame at 720p over a resident volume, BF16 mips
        dict(kind="indirect", tris=100_000, n=128, width=1280, height=720, cones=6, prec="bf16", tile="8x8",
             image="rgba16f", name="indirect_720p"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "view", "batch", "views", "screen", "indirect"])
    width = _log(rng, 60, 1920)
    height = max(40, int(width * rng.uniform(0.5, 1.0)))
    prec = rng.choice(["fp32", "fp16", "bf16", "fp16x2"])
    if kind == "frame":
        if rng.random() < 0.4:
            return _frame("soup", _log(rng, 500, 100_000), rng.choice([32, 64, 128, 256]), width, height,
                          rng.choice([4, 6, 9]), prec, rng.choice(["16x16", "8x8", "morton"]))
        return _frame("room", _log(rng, 90_000, 600_000), rng.choice([64, 128, 256]), width, height,
                      rng.choice([6, 9, 16]), prec, rng.choice(["8x8", "16x16", "32x8"]),
                      textured=rng.random() < 0.3, shadow=rng.random() < 0.3, meshes=rng.choice([1, 3, 17, 48]),
                      index=rng.choice(["none", "u32", "u16"]))
    if kind == "view":
        return dict(kind=kind, scene="room", tris=_log(rng, 90_000, 400_000), n=rng.choice([64, 128, 256]),
                    width=width, height=height, cones=rng.choice([6, 9, 16]), prec=prec,
                    tile=rng.choice(["8x8", "16x16", "32x8"]))
    if kind == "batch":
        return dict(kind=kind, scenes=rng.randint(2, 24), median=_log(rng, 2_000, 40_000),
                    side=rng.choice([128, 256, 512]), prec=prec, tile=rng.choice(["morton", "16x16"]))
    if kind == "views":
        return dict(kind=kind, scenes=rng.randint(1, 4), frames=rng.randint(2, 12), tris=_log(rng, 20_000, 120_000),
                    n=rng.choice([64, 128]), width=_log(rng, 128, 1024), height=_log(rng, 128, 768), prec=prec,
                    tile=rng.choice(["16x16", "8x8"]))
    if kind == "screen":
        return dict(kind=kind, width=width, height=height, image=rng.choice(["rgba16f", "rgba32f"]))
    return dict(kind=kind, tris=_log(rng, 90_000, 300_000), n=rng.choice([64, 128, 256]), width=width, height=height,
                cones=rng.choice([6, 9]), prec=prec, tile="8x8", image=rng.choice(["rgba16f", "rgba32f"]))


# ---------------------------------------------------------------------------
# inputs, from the seed alone (host arrays)
# ---------------------------------------------------------------------------

def _soup(seed, tris, n, width, height, cones):
    w = sg.random_soup(seed=seed, ntri=tris, n=n, levels=int(math.log2(n)), width=width, height=height)
    d = np.random.default_rng(seed).normal(size=3)
    d[1] = -abs(d[1]) - 0.5
    w.lights = [dict(type="directional", vec=tuple(float(v) for v in d / np.linalg.norm(d)), color=(1.0, 1.0, 1.0))]
    w.cones["num_diffuse"] = cones
    return w


def _camera(seed):
    """A camera pose in the room whose eye is clear of the columns."""
    for k in range(64):
        cam = sg.camera_pose(seed + 7919 * k, (0.25, 0.15, 0.15), (0.75, 0.30, 0.45))
        x = (cam[0] / sg.ROOM_DIMS[0] - 0.1) / 0.8 * 7.0
        z = (cam[2] / sg.ROOM_DIMS[2] - 0.1) / 0.8 * 7.0
        dx = (x - round(x)) / 7.0 * 0.8 * sg.ROOM_DIMS[0]
        dz = (z - round(z)) / 7.0 * 0.8 * sg.ROOM_DIMS[2]
        if dx * dx + dz * dz > 0.03 ** 2:
            break
    return cam


def _room(seed, tris, n, width, height, cones, camera_seed=None):
    pos, alb, rough = sg.room_triangles(seed, tris, sg.ROOM_DIMS)
    cam = _camera(seed if camera_seed is None else camera_seed)
    gp, gn, gr = sg.gbuffer_camera(pos, rough, cam, width, height, 60.0)
    L = sg.point_lights(seed, 4, (0.05, 0.10, 0.05), (0.95, 0.40, 0.55), 1.0, 5.0)
    return sg.Workload(
        name="room", positions=pos, albedo=alb,
        grid=dict(origin=(-0.02, -0.02, -0.02), extent=1.04, n=n, levels=int(math.log2(n))),
        lights=[dict(type="point", vec=tuple(float(v) for v in p[:3]), color=(float(p[3]),) * 3, min_distance=0.05)
                for p in L],
        gb_pos=gp, gb_nrm=gn, gb_rough=gr, width=width, height=height,
        cones=dict(num_diffuse=cones, specular=True, diffuse_aperture_deg=60.0, diffuse_ring_deg=60.0,
                   specular_aperture_deg=10.0, step_factor=0.5, max_distance=1.0, alpha_cutoff=0.99,
                   normal_offset=1.0, start_offset=1.0, eye=tuple(float(v) for v in cam[:3])),
        meta=dict(camera=cam))


def _workload(case, seed):
    make = _soup if case["scene"] == "soup" else _room
    w = make(seed, case["tris"], case["n"], case["width"], case["height"], case["cones"])
    if case.get("shadow"):
        w.lights = [dict(light, shadow=True) for light in w.lights]
    return w


def _batch_workloads(case, seed):
    """Scenes of uneven size. Their sizes (lognormal triangle counts, grids, G-buffer sides)
    are the case's, the same for every seed; their contents are the seed's."""
    rng = np.random.default_rng(case["scenes"])
    counts = sg.lognormal_ints(case["scenes"], case["scenes"], case["median"], 1.0, 1_000, 200_000)
    sides = [case["side"] // 2, case["side"]]
    return [_soup(seed + 104729 * (i + 1), int(counts[i]), int(rng.choice([32, 64, 128, 256])),
                  *(int(rng.choice(sides)),) * 2, 6) for i in range(case["scenes"])]


def _views_workloads(case, seed):
    """Per frame: the scene it reads and its workload (G-buffer and cones)."""
    return [(k % case["scenes"], _room(seed + 31 * (k % case["scenes"]), case["tris"], case["n"], case["width"],
                                       case["height"], 9, camera_seed=seed + 1009 * (k + 1)))
            for k in range(case["frames"])]


def _texture(seed):
    rng = np.random.default_rng(seed)
    tex = rng.integers(0, 256, (1024, 1024, 4), dtype=np.uint8)
    tex[..., 3] = np.where(rng.random((1024, 1024)) < 0.1, 0, 255)
    return tex


def _parts(case, w):
    """The workload's triangles split into the case's meshes: (slice, texcoords or None).
    Indexed meshes name every vertex of their own range in reverse vertex order."""
    step = -(-w.num_triangles // case["meshes"])
    if case["index"] == "u16":
        step = min(step, 21_845)  # vertices of a 16-bit mesh
    for a in range(0, w.num_triangles, step):
        part = slice(a, min(a + step, w.num_triangles))
        uv = None
        if case["textured"]:
            p = w.positions[part].reshape(-1, 3)
            uv = np.ascontiguousarray(p[:, :2] * 4.0 + p[:, 2:3], np.float32)
        yield part, uv


def _reference_targets(w, seed):
    """The reference's render targets for a room's G-buffer, and last frame's camera."""
    depth, normals, inv_proj, inv_mv, view, proj = sg.reference_gbuffer(w.gb_pos, w.gb_nrm, w.meta["camera"],
                                                                        w.width, w.height)
    prev = np.array(w.meta["camera"], np.float64)
    prev[:3] += np.random.default_rng(seed + 5).uniform(-0.01, 0.01, 3)
    return dict(depth=depth, normals=normals, inv_proj=inv_proj, inv_mv=inv_mv,
                prev_proj=sg.glsl_mat4(proj), prev_mv=sg.glsl_mat4(sg.camera_view_matrix(prev)))


def _image(rng, pixels, depth, image):
    """A colour image in [0, 3] whose alpha is a view depth near `depth`."""
    a = np.empty((pixels, 4), np.float32)
    a[:, :3] = rng.uniform(0.0, 3.0, (pixels, 3))
    a[:, 3] = depth + rng.choice([0.0, 0.01, 0.3, 1.5], pixels) * rng.standard_normal(pixels)
    return a.astype(np.float16 if image == "rgba16f" else np.float32)


def _screen_inputs(case, seed):
    """Targets, traced irradiance and history of the screen passes."""
    w = _room(seed, 30_000, 64, case["width"], case["height"], 6)
    t = _reference_targets(w, seed)
    rng = np.random.default_rng(seed)
    t["indirect"] = rng.uniform(0.0, 3.0, (w.num_pixels, 4)).astype(np.float32)
    cam = np.asarray(w.meta["camera"], np.float64)
    t["history"] = _image(rng, w.num_pixels, (w.gb_pos - cam[:3]) @ cam[3:6], case["image"])
    return w, t


# ---------------------------------------------------------------------------
# what a program holds between calls
# ---------------------------------------------------------------------------

_contexts = {}


def _context(tile):
    """The program's context for one tuning (its own stream and workspaces)."""
    if tile not in _contexts:
        ctx = vgi.Context(torch.cuda.current_device())
        w, h, order = TILES[tile]
        ctx.set_tuning(bin_size=8, chunk_tris=64, tile_w=w, tile_h=h, pixel_order=order)
        _contexts[tile] = ctx
    return _contexts[tile]


class _Out:
    """A torch tensor as an output buffer of the package's calls."""

    def __init__(self, shape, dtype=torch.float32, tensor=None):
        self.tensor = torch.empty(shape, dtype=dtype, device="cuda") if tensor is None else tensor
        self.ptr = self.tensor.data_ptr()


def _image_out(pixels, image):
    return _Out((pixels, 4), torch.float16 if image == "rgba16f" else torch.float32)


FORMATS = {"rgba16f": vgi.IMAGE_RGBA16F, "rgba32f": vgi.IMAGE_RGBA32F}


def _meshes(ctx, case, w, seed):
    out = []
    tex = _texture(seed) if case["textured"] else None
    for part, uv in _parts(case, w):
        pos = w.positions[part].reshape(-1, 3)
        idx = None
        if case["index"] != "none":  # the vertices stored last to first
            pos = np.ascontiguousarray(pos[::-1])
            uv = None if uv is None else np.ascontiguousarray(uv[::-1])
            idx = np.arange(pos.shape[0] - 1, -1, -1).astype(np.uint16 if case["index"] == "u16" else np.uint32)
        out.append(vgi.MeshData(ctx, pos, indices=idx, albedo=w.albedo[part], texcoords=uv, texture=tex))
    return out


class _Scene:
    """One workload on the device: scene handle, meshes, G-buffer and parameters."""

    def __init__(self, ctx, w, meshes):
        self.scene = ctx.scene()
        self.meshes = meshes
        self.grid = vgi.make_grid(**w.grid)
        self.lights = vgi.make_lights(w.lights)
        self.gb = vgi.GBufferData(ctx, w.gb_pos, w.gb_nrm, w.width, w.height, w.gb_rough)
        self.cones = vgi.make_cones(**w.cones)

    def build(self, prec):
        self.scene.voxelize(self.meshes, self.grid)
        self.scene.build_mips(self.lights, prec)


class _Chain:
    """Images and parameters of the screen passes."""

    def __init__(self, ctx, case, w, t):
        px = w.num_pixels
        self.ctx, self.width, self.height, self.t = ctx, w.width, w.height, t
        self.fmt = FORMATS[case["image"]]
        self.depth = vgi.DeviceArray.from_numpy(ctx, t["depth"])
        self.normals = vgi.DeviceArray.from_numpy(ctx, t["normals"])
        self.history = vgi.DeviceArray.from_numpy(ctx, t["history"])
        self.position, self.normal, self.view_depth = _Out((px, 3)), _Out((px, 3)), _Out((px,))
        self.blend, self.blur_y, self.blur_x = (_image_out(px, case["image"]) for _ in range(3))

    def decode(self):
        t = self.t
        self.ctx.gbuffer_decode(self.depth, self.normals, t["inv_proj"], t["inv_mv"], self.width, self.height,
                                self.position, self.normal, self.view_depth)

    def resolve(self, indirect):
        t = self.t
        self.ctx.temporal_resolve(indirect, self.position, self.view_depth, self.history, self.blend, t["prev_proj"],
                                  t["prev_mv"], self.width, self.height, self.fmt, self.fmt)
        self.ctx.bilateral_blur(self.blend, self.depth, self.blur_y, self.width, self.height, 1, self.fmt, self.fmt)
        self.ctx.bilateral_blur(self.blur_y, self.depth, self.blur_x, self.width, self.height, 0, self.fmt, self.fmt)

    def outputs(self):
        return dict(position=self.position.tensor, normal=self.normal.tensor, view_depth=self.view_depth.tensor,
                    blend=self.blend.tensor, blur_y=self.blur_y.tensor, blur_x=self.blur_x.tensor)


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case = case
    s.ctx = ctx = _context(case.get("tile", "16x16"))
    kind = case["kind"]
    if kind == "screen":
        w, t = _screen_inputs(case, seed)
        s.chain = _Chain(ctx, case, w, t)
        s.indirect = vgi.DeviceArray.from_numpy(ctx, t["indirect"])
        return s
    s.prec = vgi.PREC_NAMES[case["prec"]]
    if kind in ("frame", "view"):
        w = _workload(case, seed)
        plain = dict(textured=False, meshes=1, index="none")
        s.one = _Scene(ctx, w, _meshes(ctx, {**plain, **case}, w, seed))
        s.diffuse, s.specular = _Out((w.num_pixels, 4)), _Out((w.num_pixels, 4))
        if kind == "view":
            s.one.build(s.prec)
    elif kind == "indirect":
        w = _room(seed, case["tris"], case["n"], case["width"], case["height"], case["cones"])
        s.one = _Scene(ctx, w, [vgi.MeshData(ctx, w.positions.reshape(-1, 3), albedo=w.albedo)])
        s.one.build(s.prec)
        t = _reference_targets(w, seed)
        cam = np.asarray(w.meta["camera"], np.float64)
        t["history"] = _image(np.random.default_rng(seed), w.num_pixels, (w.gb_pos - cam[:3]) @ cam[3:6],
                              case["image"])
        s.chain = _Chain(ctx, case, w, t)
        s.diffuse, s.specular = _Out((w.num_pixels, 4)), _Out((w.num_pixels, 4))
        s.gbuffer = s.one.gb
        s.gbuffer.desc.position, s.gbuffer.desc.normal = s.chain.position.ptr, s.chain.normal.ptr
    else:
        if kind == "batch":
            ws = _batch_workloads(case, seed)
            s.scenes = [_Scene(ctx, w, [vgi.MeshData(ctx, w.positions.reshape(-1, 3), albedo=w.albedo)]) for w in ws]
            reads = s.scenes
        else:
            pairs = _views_workloads(case, seed)
            ws = [w for _, w in pairs]
            s.scenes, reads = {}, []
            for i, w in pairs:
                one = _Scene(ctx, w, [])
                if i not in s.scenes:
                    one.meshes = [vgi.MeshData(ctx, w.positions.reshape(-1, 3), albedo=w.albedo)]
                    one.build(s.prec)
                    s.scenes[i] = one
                one.scene = s.scenes[i].scene
                reads.append(one)
        pixels = [w.num_pixels for w in ws]
        s.diffuse, s.specular = (torch.empty((sum(pixels), 4), dtype=torch.float32, device="cuda") for _ in range(2))
        outs = [(_Out(None, tensor=d), _Out(None, tensor=r))
                for d, r in zip(s.diffuse.split(pixels), s.specular.split(pixels))]
        s.jobs = [(o.scene, o.gb, o.cones, d, r) for o, (d, r) in zip(reads, outs)]
        s.reads = reads
        if kind == "batch":
            s.voxelize = [(o.scene, o.meshes, o.grid) for o in s.scenes]
            s.mips = [(o.scene, o.lights) for o in s.scenes]
    ctx.sync()
    return s


def run(s):
    kind = s.case["kind"]
    if kind == "frame":
        s.one.build(s.prec)
        s.one.scene.trace(s.one.gb, s.one.cones, s.diffuse, s.specular)
        return dict(diffuse=s.diffuse.tensor, specular=s.specular.tensor)
    if kind == "view":
        s.one.scene.trace(s.one.gb, s.one.cones, s.diffuse, s.specular)
        return dict(diffuse=s.diffuse.tensor, specular=s.specular.tensor)
    if kind == "screen":
        s.chain.decode()
        s.chain.resolve(s.indirect)
        return s.chain.outputs()
    if kind == "indirect":
        s.chain.decode()
        s.one.scene.trace(s.gbuffer, s.one.cones, s.diffuse, s.specular)
        s.chain.resolve(s.diffuse)
        return dict(s.chain.outputs(), diffuse=s.diffuse.tensor, specular=s.specular.tensor)
    if kind == "batch":
        s.ctx.voxelize_batch(s.voxelize)
        s.ctx.build_mips_batch(s.mips, s.prec)
    s.ctx.trace_batch(s.jobs)
    return dict(diffuse=s.diffuse, specular=s.specular)


# ---------------------------------------------------------------------------
# the work of one pass
# ---------------------------------------------------------------------------

def _samples(n, aperture_tan, extent=1.0):
    h, t, m = extent / n, extent / n, 0
    while t <= 1.0:
        m += 1
        t += 0.5 * max(h, 2.0 * t * aperture_tan)
    return m


def _trace_work(pixels, n, cones, rough):
    """G-buffer in, irradiance out; 64 operations for each of the two gathers of a sample.
    Opacity or the boundary ends a cone after about two thirds of its schedule."""
    tan_s = 0.25 if rough else math.tan(math.radians(5.0))
    samples = cones * _samples(n, math.tan(math.radians(30.0))) + _samples(n, tan_s)
    return pixels * ((28 if rough else 24) + 32), pixels * samples * 2 * 64 * 0.65


def _build_work(tris, n, texel):
    """Triangles in (36 B of vertices, 3 of albedo); the occupied voxels' texels out, about
    six voxels a triangle up to a tenth of the volume, and an eighth of them a level up."""
    voxels = min(6 * tris, n ** 3 // 10)
    return tris * 39 + voxels * texel * 8 // 7, tris * 300 + voxels * 100


def work(case):
    kind = case["kind"]
    texel = {"fp32": 16, "fp16": 8, "bf16": 8, "fp16x2": 8}[case.get("prec", "fp32")]
    image = 8 if case.get("image") == "rgba16f" else 16
    px = case.get("width", 0) * case.get("height", 0)
    if kind in ("frame", "view"):
        b, f = _trace_work(px, case["n"], case["cones"], case["scene"] == "room")
        if kind == "frame":
            vb, vf = _build_work(case["tris"], case["n"], texel)
            b, f = b + vb, f + vf
        return dict(bytes=b, flops=f)
    if kind == "batch":
        tris, side = case["median"] * 1.6 * case["scenes"], case["side"]
        b, f = _trace_work(case["scenes"] * (side * side + side * side // 4) // 2, 120, 6, False)
        vb, vf = _build_work(tris / case["scenes"], 120, texel)
        return dict(bytes=b + case["scenes"] * vb, flops=f + case["scenes"] * vf)
    if kind == "views":
        b, f = _trace_work(px * case["frames"], case["n"], 9, True)
        return dict(bytes=b, flops=f)
    # decode 12 + 28, temporal 16 + history + out, each blur colour and depth in and colour out
    screen = px * (40 + (16 if kind == "screen" else 0) + 2 * image + 2 * (2 * image) + 4)
    if kind == "screen":
        return dict(bytes=screen, flops=px * 800)
    b, f = _trace_work(px, case["n"], case["cones"], True)
    return dict(bytes=b + screen, flops=f + px * 800)


# ---------------------------------------------------------------------------
# 64-bit restatement (plain torch)
# ---------------------------------------------------------------------------

F64, I64 = torch.float64, torch.int64


def _t(a, dtype=None):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda").to(dtype) if dtype else torch.as_tensor(
        np.ascontiguousarray(a), device="cuda")


def _sat(q, N, b, d):
    """Closed box [b, b + d]^3 against triangles whose bounding boxes overlap it (integers)."""
    zero = torch.zeros((), dtype=I64, device=b.device)
    t0 = (N * (b - q[:, 0])).sum(1)
    ok = (t0 + torch.minimum(N * d, zero).sum(1) <= 0) & (t0 + torch.maximum(N * d, zero).sum(1) >= 0)
    for u in range(3):
        A, B = (u + 1) % 3, (u + 2) % 3
        sign = torch.where(N[:, u] < 0, -1, 1)
        for i in range(3):
            j = (i + 1) % 3
            na, nb = -(q[:, j, B] - q[:, i, B]) * sign, (q[:, j, A] - q[:, i, A]) * sign
            e = na * (b[:, A] - q[:, i, A]) + nb * (b[:, B] - q[:, i, B])
            ok &= e + torch.maximum(na * d, zero) + torch.maximum(nb * d, zero) >= 0
    return ok


def _sample_texture(tex, uv, e):
    """Bilinear wrap-addressed texel of the clamped barycentric numerators e."""
    e = e.clamp(min=0).to(F64)
    p = (e[:, :, None] * uv).sum(1) / e.sum(1, keepdim=True)
    p = torch.where(torch.isfinite(p).all(1, keepdim=True), p, torch.zeros_like(p))
    H, W = tex.shape[:2]
    x, y = (p[:, 0] - p[:, 0].floor()) * W - 0.5, (p[:, 1] - p[:, 1].floor()) * H - 0.5
    x0, y0 = x.floor(), y.floor()
    gx, gy = (x - x0)[:, None], (y - y0)[:, None]
    ix, iy = x0.to(I64), y0.to(I64)
    at = lambda i, j: tex[j % H, i % W]  # noqa: E731
    top = at(ix, iy) + gx * (at(ix + 1, iy) - at(ix, iy))
    bot = at(ix, iy + 1) + gx * (at(ix + 1, iy + 1) - at(ix, iy + 1))
    return top + gy * (bot - top)


def _voxels64(case, w, seed):
    """Occupied voxels (flat index x + n (y + n z)) and their sums R, G, B, count, normal."""
    g, n = w.grid, w.grid["n"]
    pos, alb = _t(w.positions).reshape(-1, 3, 3), _t(w.albedo, I64)
    # the snap is defined in single precision: v = (p - origin) * (n * 256 / extent), rounded
    scale = torch.tensor(np.float32(n * 256) / np.float32(g["extent"]), device="cuda")
    origin = torch.tensor(g["origin"], dtype=torch.float32, device="cuda")
    v = (pos - origin) * scale
    keep = (v.abs() <= 262144).all(2).all(1)
    q = torch.round(v).to(I64)
    e0, e1 = q[:, 1] - q[:, 0], q[:, 2] - q[:, 0]
    N = torch.stack([e0[:, 1] * e1[:, 2] - e0[:, 2] * e1[:, 1], e0[:, 2] * e1[:, 0] - e0[:, 0] * e1[:, 2],
                     e0[:, 0] * e1[:, 1] - e0[:, 1] * e1[:, 0]], 1)
    lo, hi = ((q.amin(1) - 1) >> 8).clamp(min=0), (q.amax(1) >> 8).clamp(max=n - 1)
    keep &= (N != 0).any(1) & (lo <= hi).all(1)
    q, N, lo, hi, alb = q[keep], N[keep], lo[keep], hi[keep], alb[keep]
    Nd = N.to(F64)
    nq = torch.round(Nd * 1024.0 / Nd.square().sum(1, keepdim=True).sqrt()).to(I64)
    tex = uvs = None
    if case.get("textured"):
        tex = _t(_texture(seed), F64) / 255.0
        uvs = _t(np.concatenate([uv for _, uv in _parts(case, w)])).to(F64).reshape(-1, 3, 2)[keep]
        a = N.abs()
        axis = torch.where(a[:, 0] > a[:, 1], torch.where(a[:, 0] > a[:, 2], 0, 2),
                           torch.where(a[:, 1] > a[:, 2], 1, 2))
    size = hi - lo + 1
    ends = size.prod(1).cumsum(0)
    found_v, found_r = [], []
    total, done, step = int(ends[-1]) if len(ends) else 0, 0, 1 << 23
    while done < total:
        c = torch.arange(done, min(done + step, total), device="cuda")
        t = torch.searchsorted(ends, c, right=True)
        r = c - (ends[t] - size[t].prod(1))
        s = size[t]
        vox = lo[t] + torch.stack([r % s[:, 0], (r // s[:, 0]) % s[:, 1], r // (s[:, 0] * s[:, 1])], 1)
        hit = _sat(q[t], N[t], vox * 256, 256)
        t, vox = t[hit], vox[hit]
        rgb = alb[t]
        if tex is not None:
            centre = vox * 256 + 128
            u = axis[t]
            A, B = (u + 1) % 3, (u + 2) % 3
            pick = lambda x, k: x.gather(1, k[:, None])[:, 0]  # noqa: E731
            sign = torch.where(pick(N[t], u) < 0, -1, 1)
            qa = torch.stack([pick(q[t, k], A) for k in range(3)], 1)
            qb = torch.stack([pick(q[t, k], B) for k in range(3)], 1)
            ca, cb = pick(centre, A), pick(centre, B)
            e = []
            for k in range(3):
                i, j = (k + 1) % 3, (k + 2) % 3
                e.append(sign * ((qa[:, j] - qa[:, i]) * (cb - qb[:, i]) - (qb[:, j] - qb[:, i]) * (ca - qa[:, i])))
            col = _sample_texture(tex, uvs[t], torch.stack(e, 1))
            on = col[:, 3] >= 0.05
            t, vox = t[on], vox[on]
            rgb = (col[on, :3].clamp(0.0, 1.0) * 255.0 + 0.5).to(I64)
        found_v.append(vox[:, 0] + n * (vox[:, 1] + n * vox[:, 2]))
        found_r.append(torch.cat([rgb, torch.ones_like(rgb[:, :1]), nq[t]], 1).to(torch.int32))
        done += step
    flat = torch.cat(found_v)
    ids, inverse = torch.unique(flat, return_inverse=True)
    sums = torch.zeros((len(ids), 7), dtype=I64, device="cuda")
    rows = torch.cat(found_r)
    for a in range(0, len(rows), step):
        sums.index_add_(0, inverse[a:a + step], rows[a:a + step].to(I64))
    return ids, sums


def _visible(occupied, ids, sums, light, grid):
    """The visibility walk of a shadow-casting light from each occupied voxel (integer steps)."""
    n = grid["n"]
    vox = torch.stack([ids % n, (ids // n) % n, ids // (n * n)], 1)
    nrm = sums[:, 4:]
    a = nrm.abs()
    ax = torch.where((a[:, 0] >= a[:, 1]) & (a[:, 0] >= a[:, 2]), 0, torch.where(a[:, 1] >= a[:, 2], 1, 2))
    start = vox + torch.zeros_like(vox).scatter_(1, ax[:, None], nrm.gather(1, ax[:, None]).sign())
    f32 = torch.float32
    steps = torch.full((len(ids),), n + 2, dtype=I64, device="cuda")
    if light["type"] == "directional":
        d = -torch.tensor(light["vec"], dtype=f32, device="cuda").expand(len(ids), 3)
    else:
        h = torch.tensor(np.float32(grid["extent"]) / np.float32(n), device="cuda")
        pv = (torch.tensor(light["vec"], dtype=f32, device="cuda")
              - torch.tensor(grid["origin"], dtype=f32, device="cuda")) / h
        d = pv - (start.to(f32) + 0.5)
    la = d.abs().amax(1, keepdim=True)
    if light["type"] != "directional":
        steps = torch.minimum(steps, la[:, 0].ceil().to(I64))
    s = torch.round((d / la) * 65536.0).nan_to_num().to(I64)
    p = start * 65536 + 32768
    lit = torch.ones(len(ids), dtype=torch.bool, device="cuda")
    walking = la[:, 0] > 0
    for m in range(n + 2):
        c = p >> 16
        walking &= (m < steps) & ((c >= 0) & (c < n)).all(1)
        if not bool(walking.any()):
            break
        c = c.clamp(0, n - 1)
        blocked = walking & occupied[c[:, 0] + n * (c[:, 1] + n * c[:, 2])] & (c != vox).any(1)
        lit &= ~blocked
        walking &= ~blocked
        p = p + s
    return lit


def _levels64(case, w, seed):
    """The mip chain without storage rounding: per level (n_k + 2)^3 padded texels, flat."""
    grid, n = w.grid, w.grid["n"]
    ids, sums = _voxels64(case, w, seed)
    count = sums[:, 3]
    mean = (sums[:, :3] + count[:, None] // 2) // count[:, None]
    albedo = (mean.to(F64) / 255.0) ** 2.2
    nrm = sums[:, 4:].to(F64) / (1024.0 * count.to(F64))[:, None]
    vox = torch.stack([ids % n, (ids // n) % n, ids // (n * n)], 1).to(F64)
    h = grid["extent"] / n
    p = torch.tensor(grid["origin"], dtype=F64, device="cuda") + (vox + 0.5) * h
    occupied = None
    if any(light.get("shadow") for light in w.lights):
        occupied = torch.zeros(n ** 3, dtype=torch.bool, device="cuda")
        occupied[ids] = True
    e = torch.zeros_like(p)
    for light in w.lights:
        vec = torch.tensor(light["vec"], dtype=F64, device="cuda")
        if light["type"] == "directional":
            f = -(nrm * vec).sum(1)
        else:
            d = vec - p
            d2 = d.square().sum(1)
            f = (nrm * d).sum(1) / d2.sqrt() / d2.clamp(min=light.get("min_distance", 0.0) ** 2)
        f = torch.where(f > 0, f, torch.zeros_like(f))
        if light.get("shadow"):
            f = f * _visible(occupied, ids, sums, light, grid)
        e += f[:, None] * torch.tensor(light["color"], dtype=F64, device="cuda")
    level = torch.zeros((n ** 3, 4), dtype=F64, device="cuda")
    level[ids] = torch.cat([albedo * e, torch.ones_like(e[:, :1])], 1)
    level = level.reshape(n, n, n, 4)
    out = []
    for k in range(grid["levels"]):
        nk = n >> k
        if k:
            level = level.reshape(nk, 2, nk, 2, nk, 2, 4).mean((1, 3, 5))
        pad = torch.zeros((nk + 2,) * 3 + (4,), dtype=F64, device="cuda")
        pad[1:-1, 1:-1, 1:-1] = level
        out.append(pad.reshape(-1, 4))
    return out


def _gather64(levels, k, n, u):
    p1 = (n >> k) + 2
    g = u * 2.0 ** -k - 0.5
    i = g.floor()
    f = g - i
    i = i.to(I64) + 1
    base = i[:, 0] + p1 * (i[:, 1] + p1 * i[:, 2])
    out = 0.0
    for dz in range(2):
        for dy in range(2):
            for dx in range(2):
                wt = (f[:, 0] if dx else 1 - f[:, 0]) * (f[:, 1] if dy else 1 - f[:, 1]) * (
                    f[:, 2] if dz else 1 - f[:, 2])
                out = out + wt[:, None] * levels[k][base + dx + p1 * (dy + p1 * dz)]
    return out


def _cone64(levels, grid, cones, o, d, tan):
    """Front-to-back march of one cone per row; tan: a number, or one per row."""
    n, h = grid["n"], grid["extent"] / grid["n"]
    top = grid["levels"] - 1
    origin = torch.tensor(grid["origin"], dtype=F64, device="cuda")
    out = torch.zeros((len(o), 4), dtype=F64, device="cuda")
    rows = torch.arange(len(o), device="cuda")
    uo, ud, acc = (o - origin) / h, d / h, out.clone()
    t = torch.full((len(o),), cones["start_offset"] * h, dtype=F64, device="cuda")
    tan = torch.as_tensor(tan, dtype=F64, device="cuda").expand(len(o))
    for _ in range(4096):
        u = uo + ud * t[:, None]
        go = (t <= cones["max_distance"]) & (u >= 0).all(1) & (u <= n).all(1) & (acc[:, 3] < cones["alpha_cutoff"])
        if not bool(go.all()):
            out[rows[~go]] = acc[~go]
            rows, uo, ud, t, tan, acc, u = (x[go] for x in (rows, uo, ud, t, tan, acc, u))
        if not len(rows):
            break
        diam = (2.0 * t * tan).clamp(min=h)
        lvl = torch.log2(diam / h).clamp(min=0.0, max=float(top))
        l0 = lvl.floor().clamp(max=max(top - 1, 0))
        s = torch.zeros_like(acc)
        for k in torch.unique(l0).tolist():
            k = int(k)
            at = (l0 == k).nonzero()[:, 0]
            fr = (lvl[at] - k)[:, None]
            v = _gather64(levels, k, n, u[at]) * (1 - fr)
            if top > 0:
                v = v + _gather64(levels, k + 1, n, u[at]) * fr
            s[at] = v
        acc = acc + (1.0 - acc[:, 3:]) * s
        t = t + cones["step_factor"] * diam
    else:
        out[rows] = acc
    return out


def _trace64(levels, w, pos, nrm, rough):
    """Diffuse and specular irradiance of every pixel, a million rows at a time."""
    c, grid = w.cones, w.grid
    h = grid["extent"] / grid["n"]
    K, ring = c["num_diffuse"], math.radians(c["diffuse_ring_deg"])
    wsum = 1.0 + (K - 1) * math.cos(ring)
    eye = torch.tensor(c["eye"], dtype=F64, device="cuda")
    diffuse = torch.zeros((len(pos), 4), dtype=F64, device="cuda")
    specular = torch.zeros_like(diffuse)
    for a in range(0, len(pos), 1 << 20):
        rows = a + (nrm[a:a + (1 << 20)] != 0).any(1).nonzero()[:, 0]
        P, nn = pos[rows], nrm[rows]
        nn = nn / nn.square().sum(1, keepdim=True).sqrt()
        o = P + nn * (c["normal_offset"] * h)
        x, y, z = nn.unbind(1)
        s = torch.where(torch.signbit(z), -1.0, 1.0).to(F64)
        ab = -1.0 / (s + z)
        b = x * y * ab
        T = torch.stack([1.0 + s * x * x * ab, s * b, -s * x], 1)
        B = torch.stack([b, s + y * y * ab, -y], 1)
        acc = torch.zeros((len(rows), 4), dtype=F64, device="cuda")
        for k in range(K):
            if k == 0:
                d, wt = nn, 1.0 / wsum
            else:
                phi = 2.0 * math.pi * (k - 1) / (K - 1)
                d = T * (math.sin(ring) * math.cos(phi)) + B * (math.sin(ring) * math.sin(phi)) + nn * math.cos(ring)
                wt = math.cos(ring) / wsum
            acc += wt * _cone64(levels, grid, c, o, d, math.tan(math.radians(c["diffuse_aperture_deg"]) / 2))
        acc[:, 3] = 1.0 - acc[:, 3]
        diffuse[rows] = acc
        i = P - eye
        i = i / i.square().sum(1, keepdim=True).sqrt()
        r = i - 2.0 * (nn * i).sum(1, keepdim=True) * nn
        tan = math.tan(math.radians(c["specular_aperture_deg"]) / 2) if rough is None else rough[rows].clamp(0.0087, 1)
        specular[rows] = _cone64(levels, grid, c, o, r, tan)
    return diffuse, specular


def _mat(m, v):
    return v @ _t(m, F64).reshape(4, 4)  # column-major storage: rows of the reshape are columns


def _chain64(case, w, t, indirect=None):
    """Decode, and a function taking the irradiance through temporal blend and both blurs."""
    W, H = w.width, w.height
    y, x = torch.meshgrid(torch.arange(H, device="cuda"), torch.arange(W, device="cuda"), indexing="ij")
    depth = _t(t["depth"], F64)
    uv = torch.stack([(x.reshape(-1) + 0.5) / W, (y.reshape(-1) + 0.5) / H], 1).to(F64)
    one = torch.ones_like(depth)[:, None]
    c = _mat(t["inv_proj"], torch.cat([uv * 2 - 1, depth[:, None], one], 1))
    cs = c[:, :3] / c[:, 3:]
    position = _mat(t["inv_mv"], torch.cat([cs, one], 1))[:, :3]
    raw = _t(t["normals"].astype(np.int32), F64)[:, :3] / 65535.0 * 2.0 - 1.0
    raw = raw / raw.square().sum(1, keepdim=True).sqrt()
    normal = _mat(t["inv_mv"], torch.cat([raw, torch.zeros_like(one)], 1))[:, :3]
    view_depth = -cs[:, 2]
    history = _t(t["history"], F64).reshape(H, W, 4)

    def blend(colour):
        q = _mat(t["prev_proj"], _mat(t["prev_mv"], torch.cat([position, one], 1)))
        r = q[:, :2] / q[:, 3:] * 0.5 + 0.5
        on = ((r >= 0) & (r <= 1)).all(1)
        r = torch.where(on[:, None], r, torch.zeros_like(r))
        px, py = r[:, 0] * W - 0.5, r[:, 1] * H - 0.5
        x0, y0 = px.floor(), py.floor()
        fx, fy = (px - x0)[:, None], (py - y0)[:, None]
        x0, y0 = x0.to(I64), y0.to(I64)
        at = lambda i, j: history[j % H, i % W]  # noqa: E731
        hist = ((at(x0, y0) * (1 - fx) + at(x0 + 1, y0) * fx) * (1 - fy)
                + (at(x0, y0 + 1) * (1 - fx) + at(x0 + 1, y0 + 1) * fx) * fy)
        s = (1.0 - (hist[:, 3] - view_depth).abs()).clamp(0.0, 1.0)
        f = (0.95 * s * s * (3.0 - 2.0 * s))[:, None]
        mixed = (colour[:, :3] * (1 - f) + hist[:, :3] * f).clamp(0.0, 16.0)
        return torch.cat([torch.where(on[:, None], mixed, colour[:, :3]), view_depth[:, None]], 1)

    def blur(img, axis):
        img, d = img.reshape(H, W, 4), depth.reshape(H, W)
        size = W if axis == 0 else H
        total, wsum = img[..., :3].clone(), torch.ones_like(d)
        for r, off in ((1, 2), (2, 4), (3, 6), (4, 8), (5, 11), (7, 15)):
            for o in (off, -off):
                at = (torch.arange(size, device="cuda") + o).clamp(0, size - 1)
                dim = 1 if axis == 0 else 0
                wt = torch.exp2(-r * r / 32.0 - ((d - d.index_select(dim, at)) * 512.0) ** 2)
                total += wt[..., None] * img.index_select(dim, at)[..., :3]
                wsum += wt
        return torch.cat([total / wsum[..., None], torch.zeros_like(wsum)[..., None]], 2).reshape(-1, 4)

    def resolve(colour):
        b = blend(colour)
        by = blur(b, 1)
        return dict(position=position, normal=normal, view_depth=view_depth, blend=b, blur_y=by, blur_x=blur(by, 0))

    return position, normal, resolve


def exact(case, seed):
    kind = case["kind"]
    if kind == "screen":
        w, t = _screen_inputs(case, seed)
        _, _, resolve = _chain64(case, w, t)
        return resolve(_t(t["indirect"], F64))
    if kind in ("frame", "view"):
        w = _workload(case, seed)
        rough = None if w.gb_rough is None else _t(w.gb_rough, F64)
        d, r = _trace64(_levels64(case, w, seed), w, _t(w.gb_pos, F64), _t(w.gb_nrm, F64), rough)
        return dict(diffuse=d, specular=r)
    if kind == "indirect":
        w = _room(seed, case["tris"], case["n"], case["width"], case["height"], case["cones"])
        t = _reference_targets(w, seed)
        cam = np.asarray(w.meta["camera"], np.float64)
        t["history"] = _image(np.random.default_rng(seed), w.num_pixels, (w.gb_pos - cam[:3]) @ cam[3:6],
                              case["image"])
        position, normal, resolve = _chain64(case, w, t)
        d, r = _trace64(_levels64(case, w, seed), w, position, normal, _t(w.gb_rough, F64))
        return dict(resolve(d), diffuse=d, specular=r)
    if kind == "batch":
        pairs = list(enumerate(_batch_workloads(case, seed)))
    else:
        pairs = _views_workloads(case, seed)
    levels, ds, rs = {}, [], []
    for i, w in pairs:
        if i not in levels:
            if kind == "batch":
                levels.clear()  # each scene is read once
            levels[i] = _levels64(case, w, seed)
        rough = None if w.gb_rough is None else _t(w.gb_rough, F64)
        d, r = _trace64(levels[i], w, _t(w.gb_pos, F64), _t(w.gb_nrm, F64), rough)
        ds.append(d)
        rs.append(r)
    return dict(diffuse=torch.cat(ds), specular=torch.cat(rs))
