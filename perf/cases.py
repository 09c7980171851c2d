"""The work that programs built on helios_amd have it do, as cases that can be timed.

Each case is one call (or the few calls of one displayed frame) through the
public entry points: progressive path tracing one frame per call and many
frames per call, batches of views, scene edits, output-buffer views, ray
queries on device buffers, and the learned denoiser's inference and training.

Geometry is generated once per process and shape; the seed moves the spheres,
the lights and the camera (path tracing) or draws the images (denoiser).
"""
import functools
import math
from pathlib import Path

import numpy as np
import torch

from helios_amd import abi, runtime, scenegen
from helios_amd.denoise import Denoiser, forward_bytes, forward_flops

WEIGHTS = Path(__file__).resolve().parents[1] / "helios_amd" / "data" / "denoiser_unet.bin"

# What one path-traced sample takes on the icosphere field, measured by the
# counting traversal: segments and shadow rays per sample, nodes and triangles
# visited per ray. A node test is 4 boxes of 24 operations, a triangle test
# 50, one shaded hit about 400.
SEGMENTS, SHADOW_RAYS = 1.37, 0.48
RAY_FLOPS = 12.6 * 96 + 5.1 * 50
NODE_BYTES_PER_TRI, TRI_BYTES = 22, 48 + 64     # BVH4 nodes; leaf triangle + shading record


def listed():
    return [
        # a viewer on a small scene, one progressive frame per call: launches and host work count
        {"name": "frame_cornell_256", "kind": "frames", "scene": "cornell", "width": 256, "height": 256, "frames": 1,
         "in_flight": 4, "block": 256, "blocks_per_cu": 8, "continuation": 0, "mega": False, "bounces": 5},
        # a viewer window of odd size on a scene with every texture kind: one frame, then its RGBA8 image on the host
        {"name": "viewer_showcase_639x359", "kind": "viewer", "scene": "showcase", "width": 639, "height": 359,
         "in_flight": 4, "block": 256, "blocks_per_cu": 8, "bounces": 4},
        # a viewer on 1.3 M triangles at 1080p, the single-frame form of the integrator
        {"name": "frame_field_1080p", "kind": "frames", "scene": "field", "spheres": 64, "level": 5, "leaves": 2000,
         "width": 1920, "height": 1080, "frames": 1, "in_flight": 256, "block": 64, "blocks_per_cu": 32,
         "continuation": 4, "mega": True, "bounces": 8},
        # offline progressive rendering: 20 samples of every pixel in one call
        {"name": "frames_field_1080p_x20", "kind": "frames", "scene": "field", "spheres": 64, "level": 5, "leaves": 2000,
         "width": 1920, "height": 1080, "frames": 20, "in_flight": 256, "block": 64, "blocks_per_cu": 32,
         "continuation": 4, "mega": False, "bounces": 8},
        # views of one instanced scene with power-sampled emitters, an equirectangular sky and feature planes
        {"name": "batch_combined_2x1280x720", "kind": "combined", "views": 2, "width": 1280, "height": 720, "spp": 2,
         "instances": 1000, "meshes": 12, "bounces": 16, "in_flight": 4, "block": 64, "blocks_per_cu": 32},
        # many independent scenes and views of uneven size in shared passes
        {"name": "batch_scenes_8", "kind": "batch", "views": 8, "min_side": 128, "max_side": 1024, "max_tris": 200000,
         "spp": 4, "bounces": 8, "in_flight": 16, "block": 64, "blocks_per_cu": 32},
        # an editor moves a node: new transform, commit, one frame
        {"name": "edit_field_960x540", "kind": "edit", "spheres": 48, "level": 4, "leaves": 1500, "width": 960,
         "height": 540, "bounces": 5, "in_flight": 4, "block": 64, "blocks_per_cu": 32},
        # an editor's normals view
        {"name": "normals_field_1080p", "kind": "view", "spheres": 48, "level": 4, "leaves": 1500, "width": 1920,
         "height": 1080, "which": abi.OUTPUT_BUFFER_NORMALS},
        # visibility and picking queries of a serving loop on device buffers, at its largest batch
        {"name": "rays_field_32768", "kind": "rays", "spheres": 48, "level": 4, "leaves": 1500, "rays": 32768,
         "flags": 0},
        # the denoiser on a rendered 1080p frame
        {"name": "denoise_1080p", "kind": "denoise", "width": 1920, "height": 1080, "frames": 2},
        # the denoiser on a small odd window (padded to multiples of 8)
        {"name": "denoise_417x233", "kind": "denoise", "width": 417, "height": 233, "frames": 4},
        # one training step of the denoiser as denoise_train runs it: 8 crops of 128 x 128
        {"name": "train_8x128x128", "kind": "train", "images": 8, "height": 128, "width": 128, "loss": "relmse"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frames", "frames", "viewer", "combined", "batch", "edit", "view", "rays", "denoise", "train"])
    field = {"spheres": rng.randint(8, 64), "level": rng.randint(2, 4), "leaves": rng.randint(0, 2000)}
    big = {"block": 64, "blocks_per_cu": 32}
    if kind == "frames":
        w, h = _log(rng, 64, 1920), _log(rng, 64, 1080)
        scene = rng.choice(["cornell", "showcase", "field"])
        c = {"kind": kind, "scene": scene, "width": w, "height": h, "frames": rng.choice([1, 1, 2, 5, 8, 16]),
             "in_flight": rng.choice([1, 4, 8, 16]), "continuation": rng.choice([0, 4]), "mega": rng.random() < 0.3,
             "bounces": rng.randint(2, 8)}
        c.update(big if rng.random() < 0.6 else {"block": 256, "blocks_per_cu": 8})
        return {**c, **field} if scene == "field" else c
    if kind == "viewer":
        return {"kind": kind, "scene": rng.choice(["cornell", "showcase"]), "width": _log(rng, 64, 1920),
                "height": _log(rng, 64, 1080), "in_flight": 4, "block": 256, "blocks_per_cu": 8,
                "bounces": rng.randint(2, 7)}
    if kind == "combined":
        return {"kind": kind, "views": rng.randint(1, 4), "width": _log(rng, 160, 1280), "height": _log(rng, 90, 720),
                "spp": rng.randint(1, 4), "instances": _log(rng, 50, 1000), "meshes": rng.randint(2, 12),
                "bounces": rng.randint(4, 16), "in_flight": 4, **big}
    if kind == "batch":
        return {"kind": kind, "views": rng.randint(2, 8), "min_side": 64, "max_side": _log(rng, 128, 1024),
                "max_tris": _log(rng, 20000, 200000), "spp": rng.randint(1, 8), "bounces": rng.randint(3, 8),
                "in_flight": rng.choice([1, 4, 16]), **big}
    if kind == "edit":
        return {"kind": kind, **field, "width": _log(rng, 128, 1280), "height": _log(rng, 96, 720),
                "bounces": rng.randint(2, 8), "in_flight": 4, **big}
    if kind == "view":
        return {"kind": kind, **field, "width": _log(rng, 128, 1920), "height": _log(rng, 96, 1080),
                "which": rng.randint(0, 4)}
    if kind == "rays":
        return {"kind": kind, **field, "rays": _log(rng, 1, 32768),
                "flags": rng.choice([0, abi.HH_TRACE_OPAQUE, abi.HH_TRACE_OPAQUE | abi.HH_TRACE_TERMINATE_ON_FIRST])}
    if kind == "denoise":
        return {"kind": kind, "width": _log(rng, 64, 1920), "height": _log(rng, 48, 1080), "frames": rng.randint(1, 8)}
    return {"kind": "train", "images": rng.randint(1, 8), "height": rng.randint(4, 16) * 8, "width": rng.randint(33, 128),
            "loss": rng.choice(["relmse", "log_mse"])}


# ---------------------------------------------------------------------------
# Scenes
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=12)
def _field_geometry(spheres, level, leaves):
    return scenegen.icosphere_field(seed=0, n_spheres=spheres, level=level, n_leaves=leaves)


@functools.lru_cache(maxsize=4)
def _combined_geometry(meshes, instances, views):
    d, cams = scenegen.combined_workload(seed=0, n_meshes=meshes, n_instances=instances, equirect_width=2048)
    return d, cams


@functools.lru_cache(maxsize=12)
def _triangles_geometry(triangles):
    return scenegen.field_for_triangles(0, triangles, 64, 64)


def _copy(d):
    return scenegen.SceneDesc(textures=d.textures, materials=d.materials, meshes=d.meshes, instances=list(d.instances),
                              lights=[dict(x) for x in d.lights], ibl=d.ibl, sky=d.sky, camera=dict(d.camera),
                              width=d.width, height=d.height, max_ray_bounces=d.max_ray_bounces, spp=d.spp)


def _orbit(rng):
    """A camera around the field, as denoise_train and the batched workload place theirs."""
    a, r = rng.uniform(0, 2 * np.pi), rng.uniform(100.0, 150.0)
    return scenegen.look_at_camera((r * math.cos(a), rng.uniform(20.0, 50.0), r * math.sin(a)),
                                   (rng.uniform(-10, 10), 0.0, rng.uniform(-10, 10)), fov_y=60.0, aperture=0.0)


def _turned(inst, rng):
    """The instance turned about its own vertical axis."""
    model, normal, mesh, override = inst
    a = rng.uniform(0, 2 * np.pi)
    r = np.eye(4)
    r[0, 0], r[0, 2], r[2, 0], r[2, 2] = math.cos(a), math.sin(a), -math.sin(a), math.cos(a)
    m, n = (np.asarray(x, np.float64).reshape(4, 4).T @ r for x in (model, normal))
    return m.T.astype(np.float32).ravel(), n.T.astype(np.float32).ravel(), mesh, override


def _field(base, rng):
    d = _copy(base)
    last = len(d.instances) - (1 if len(d.meshes[-1].materials) and d.materials[d.meshes[-1].materials[0]]["alpha_test"] else 0)
    for i in range(1, last):
        d.instances[i] = _turned(d.instances[i], rng)
    for light in d.lights:
        if light["type"] == abi.LIGHT_POINT:
            light["position"] = (float(rng.uniform(-60, 60)), float(rng.uniform(15, 30)), float(rng.uniform(-60, 60)))
    d.camera = _orbit(rng)
    return d


def _desc(case, rng):
    if case["scene"] == "cornell":
        d = scenegen.cornell_box(width=case["width"], height=case["height"], max_ray_bounces=case["bounces"])
        eye = (rng.uniform(-0.05, 0.05), rng.uniform(-0.05, 0.05), rng.uniform(-0.05, 0.05))
        d.camera["position"] = tuple(float(p + e) for p, e in zip(d.camera["position"], eye))
        return d
    if case["scene"] == "showcase":
        d = scenegen.textured_showcase(width=case["width"], height=case["height"], max_ray_bounces=case["bounces"])
        a = rng.uniform(-0.6, 0.6)
        d.camera = scenegen.look_at_camera((6.0 * math.sin(a), rng.uniform(2.5, 4.0), 6.0 * math.cos(a)), (0.0, 0.4, 0.0),
                                           fov_y=45.0)
        return d
    return _field(_field_geometry(case["spheres"], case["level"], case["leaves"]), rng)


# ---------------------------------------------------------------------------
# States
# ---------------------------------------------------------------------------
class Program:
    """A program's context and its objects, closed in reverse order when nothing refers to them any more."""

    def __init__(self):
        self.owned = []
        self.ctx = runtime.Context(0)

    def __del__(self):
        if hasattr(self, "ctx"):
            self.ctx.sync()
            while self.owned:
                self.owned.pop().close()
            self.ctx.close()


class _Memory:
    """Device memory of the library, seen by torch without a copy. The tensor keeps this object, and
    this object keeps the program whose memory it is."""

    def __init__(self, program, address, shape):
        self.program = program
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (address, False), "version": 3}


class State:
    def __init__(self, case):
        self.case = case
        self.program = Program()
        self.ctx = self.program.ctx

    def own(self, x):
        self.program.owned.append(x)
        return x

    def tune(self):
        c = self.case
        self.ctx.set_tuning(extend_block=c["block"], persistent_blocks_per_cu=c["blocks_per_cu"],
                            frames_in_flight=c["in_flight"], continuation_depth=c.get("continuation", 0))

    def surface(self, w, h, features=False):
        s = self.own(runtime.Surface(self.ctx, w, h))
        if features:
            s.enable_features()
        s.clear()
        return s, torch.as_tensor(_Memory(self.program, s.device_ptr(), (h, w, 4)), device="cuda")

    def integrator(self, bounces, flags=0):
        it = self.own(runtime.PathIntegrator(self.ctx))
        it.set_max_ray_bounces(bounces)
        it.set_max_samples(1 << 20)
        it.set_flags(flags)
        return it


def _rng(case, seed):
    return np.random.Generator(np.random.PCG64(seed))


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, _rng(case, seed), State(case))


def run(state):
    return globals()["_run_" + state.case["kind"]](state)


def _prepare_frames(case, rng, s):
    s.tune()
    d = _desc(case, rng)
    s.scene = s.own(runtime.Scene(s.ctx, d))
    s.camera = runtime.camera_struct(d.camera)
    s.out, s.image = s.surface(case["width"], case["height"])
    s.it = s.integrator(case["bounces"], abi.HH_FLAG_MEGAKERNEL if case["mega"] else 0)
    return s


def _run_frames(s):
    # from a cleared image, as after every camera move
    s.it.restart_bake()
    s.it.render(s.scene, s.camera, s.out, frames=s.case["frames"])
    return s.image


def _prepare_viewer(case, rng, s):
    return _prepare_frames({**case, "mega": False}, rng, s)


def _run_viewer(s):
    s.it.restart_bake()
    s.it.render(s.scene, s.camera, s.out)
    return {"radiance": s.image, "display": s.out.tone_map()}


def _prepare_combined(case, rng, s):
    s.tune()
    base, cams = _combined_geometry(case["meshes"], case["instances"], case["views"])
    d = _copy(base)
    d.instances = [_turned(x, rng) if i and x[2] <= case["meshes"] else x for i, x in enumerate(d.instances)]
    s.scene = s.own(runtime.Scene(s.ctx, d))
    s.views, s.images = [], []
    for cam in cams[:case["views"]]:
        p = [float(x + rng.uniform(-5, 5)) for x in cam["position"]]
        surf, image = s.surface(case["width"], case["height"], features=True)
        s.images.append(image)
        s.views.append({"scene": s.scene, "surface": surf, "camera": runtime.camera_struct({**cam, "position": p}),
                        "spp": case["spp"], "max_ray_bounces": case["bounces"], "flags": abi.HH_FLAG_LIGHT_POWER})
    return s


def _run_combined(s):
    runtime.render_batch(s.ctx, s.views)
    return s.images


def _batch_params(case):
    """(side, triangles) of the batch's views: log-uniform, the same for every seed."""
    rng = np.random.Generator(np.random.PCG64(7919))
    out = []
    for _ in range(case["views"]):
        side = math.exp(rng.uniform(math.log(case["min_side"]), math.log(case["max_side"])))
        out.append((int(round(side)), int(round(math.exp(rng.uniform(math.log(10000), math.log(case["max_tris"])))))))
    return out


def _prepare_batch(case, rng, s):
    s.tune()
    s.views, s.images = [], []
    for side, triangles in _batch_params(case):
        d = _field(_triangles_geometry(triangles), rng)
        surf, image = s.surface(side, side)
        s.images.append(image)
        s.views.append({"scene": s.own(runtime.Scene(s.ctx, d)), "surface": surf, "camera": runtime.camera_struct(d.camera),
                        "spp": case["spp"], "max_ray_bounces": case["bounces"]})
    return s


def _run_batch(s):
    runtime.render_batch(s.ctx, s.views)
    return s.images


def _prepare_edit(case, rng, s):
    s = _prepare_frames({**case, "scene": "field", "mega": False}, rng, s)
    place = s.scene.desc.instances[1]
    s.places = []
    for _ in range(2):      # the node goes back and forth between two places
        model, normal, _, _ = _turned(place, rng)
        model[12:15] += rng.uniform(-3.0, 3.0, 3).astype(np.float32)
        normal[12:15] = model[12:15]
        s.places.append((model, normal))
    s.at = 0
    return s


def _run_edit(s):
    model, normal = s.places[s.at]
    s.at ^= 1
    runtime.check(runtime.lib().hh_scene_set_instance_transform(s.scene.h, 1, abi.ptr(model), abi.ptr(normal)))
    s.scene.commit()
    s.it.render(s.scene, s.camera, s.out)
    return s.image


def _prepare_view(case, rng, s):
    d = _field(_field_geometry(case["spheres"], case["level"], case["leaves"]), rng)
    s.scene = s.own(runtime.Scene(s.ctx, d))
    s.camera = runtime.camera_struct(d.camera)
    s.out, s.image = s.surface(case["width"], case["height"])
    return s


def _run_view(s):
    runtime.render_output_buffer(s.scene, s.camera, s.case["which"], s.out)
    return s.image


def _prepare_rays(case, rng, s):
    d = _field(_field_geometry(case["spheres"], case["level"], case["leaves"]), rng)
    s.scene = s.own(runtime.Scene(s.ctx, d))
    rays = scenegen.random_rays(case["rays"], (-100.0, 0.5, -100.0), (100.0, 40.0, 100.0), seed=int(rng.integers(1 << 31)))
    s.rays = torch.from_numpy(rays.view(np.float32).reshape(-1, 8)).cuda()
    s.hits = torch.zeros((case["rays"], 6), dtype=torch.int32, device="cuda")
    s.image = {"t_u_v": s.hits.view(torch.float32)[:, :3], "ids": s.hits[:, 3:]}
    torch.cuda.synchronize()
    return s


def _run_rays(s):
    s.scene.trace_rays_device(s.rays.data_ptr(), s.case["rays"], s.case["flags"], s.hits.data_ptr())
    return s.image


def _prepare_denoise(case, rng, s):
    # a noisy frame of the field with its feature planes, rendered by the tracer
    d = _field(_field_geometry(12, 3, 300), rng)
    s.scene = s.own(runtime.Scene(s.ctx, d))
    s.noisy, s.noisy_image = s.surface(case["width"], case["height"], features=True)
    s.out, s.image = s.surface(case["width"], case["height"])
    s.integrator(4).render(s.scene, d.camera, s.noisy, frames=case["frames"])
    s.dn = s.own(Denoiser(s.ctx, params=np.fromfile(WEIGHTS, np.float32)))
    return s


def _run_denoise(s):
    s.dn.denoise(s.noisy, s.case["frames"], s.out)
    return s.image


def _crops(case, rng):
    """Raw records (n, h, w, 12) and targets (n, h, w, 3) as crops of rendered views have them: smooth
    radiance and features with edges, radiance noise falling with the samples held."""
    n, h, w = case["images"], case["height"], case["width"]

    def smooth(c, cells):
        g = rng.random((n, cells + 2, cells + 2, c), np.float32)
        y, x = np.linspace(0, cells, h, endpoint=False), np.linspace(0, cells, w, endpoint=False)
        iy, ix = y.astype(int), x.astype(int)
        fy, fx = (y - iy).astype(np.float32)[None, :, None, None], (x - ix).astype(np.float32)[None, None, :, None]
        a, b = g[:, iy][:, :, ix], g[:, iy][:, :, ix + 1]
        c0, d0 = g[:, iy + 1][:, :, ix], g[:, iy + 1][:, :, ix + 1]
        return (a * (1 - fx) + b * fx) * (1 - fy) + (c0 * (1 - fx) + d0 * fx) * fy

    edge = smooth(1, 6) > 0.5
    albedo = np.where(edge, smooth(3, 4), smooth(3, 9))
    normal = np.where(edge, smooth(3, 5), smooth(3, 2)) * 2 - 1
    normal /= np.maximum(np.linalg.norm(normal, axis=-1, keepdims=True), 1e-6)
    target = albedo * (0.1 + 0.9 * smooth(3, 5))
    held = np.array([1, 2, 4, 8, 16, 32], np.float32)[rng.integers(0, 6, n)][:, None, None, None] * np.ones((n, h, w, 1), np.float32)
    noise = rng.gamma(0.5 * held, 2.0 / held).astype(np.float32)      # mean 1, variance 2 / held
    radiance = np.minimum(target * noise, 1.0)
    m2 = 2.0 * (target.mean(-1, keepdims=True) ** 2) * np.maximum(held - 1, 0)
    feats = np.concatenate([radiance, albedo, 0.2 + 0.6 * smooth(1, 4), normal, m2, held], -1)
    return np.ascontiguousarray(feats, np.float32), np.ascontiguousarray(target, np.float32)


def _prepare_train(case, rng, s):
    s.feats, s.target = _crops(case, rng)
    s.dn = s.own(Denoiser(s.ctx, seed=0))       # a fresh network, as training starts
    s.dn.set_loss(case["loss"])
    return s


def _run_train(s):
    loss = s.dn.train_step(s.feats, s.target, 1e-3)
    return {"loss": np.float32(loss), "grads": s.dn.grads()}


# ---------------------------------------------------------------------------
# Work
# ---------------------------------------------------------------------------
def _field_triangles(case):
    return 20 * 4 ** case["level"] * case["spheres"] + 2 * case["leaves"] + 2


def _paths(samples, triangles):
    return {"bytes": triangles * (NODE_BYTES_PER_TRI + TRI_BYTES), "flops": samples * (SEGMENTS * (RAY_FLOPS + 400) + SHADOW_RAYS * RAY_FLOPS)}


def work(case):
    """Bytes and operations of one pass: scene records read once, images written once; the tests and
    shading that the pass's paths take."""
    kind = case["kind"]
    px = case.get("width", 0) * case.get("height", 0)
    if kind in ("frames", "viewer"):
        tris = {"cornell": 36, "showcase": 1294}.get(case["scene"]) or _field_triangles(case)
        w = _paths(px * case.get("frames", 1), tris)
        w["bytes"] += px * (16 + (16 + 4 if kind == "viewer" else 0))
        return w
    if kind == "combined":
        w = _paths(px * case["views"] * case["spp"], 10000 * case["meshes"])
        w["bytes"] += px * case["views"] * 48 + case["instances"] * 208
        return w
    if kind == "batch":
        params = _batch_params(case)
        w = _paths(sum(s * s for s, _ in params) * case["spp"], sum(t for _, t in params))
        w["bytes"] += sum(s * s for s, _ in params) * 16
        return w
    if kind == "edit":
        w = _paths(px, _field_triangles(case))
        w["bytes"] += px * 16
        return w
    if kind == "view":
        return {"bytes": px * 16 + _field_triangles(case) * (NODE_BYTES_PER_TRI + 48 + 260), "flops": px * RAY_FLOPS}
    if kind == "rays":
        return {"bytes": case["rays"] * 56 + _field_triangles(case) * (NODE_BYTES_PER_TRI + 48), "flops": case["rays"] * RAY_FLOPS}
    if kind == "denoise":
        return {"bytes": px * 64, "flops": forward_flops(case["height"], case["width"])}
    n = case["images"]
    return {"bytes": n * px * 60 + 480675 * 4 * 7, "flops": 3 * n * forward_flops(case["height"], case["width"])}


# ---------------------------------------------------------------------------
# What the denoiser's passes give in 64 bits. A path-traced sample has no such value: it is a chain of
# decisions (which triangle, which lobe, whether the path goes on) taken on 32-bit numbers.
# ---------------------------------------------------------------------------
_LAYERS = [("enc0a", 10, 32), ("enc0b", 32, 32), ("enc1a", 32, 48), ("enc1b", 48, 48), ("enc2a", 48, 64), ("enc2b", 64, 64),
           ("mida", 64, 96), ("midb", 96, 96), ("dec2a", 160, 64), ("dec2b", 64, 64), ("dec1a", 112, 48), ("dec1b", 48, 48),
           ("dec0a", 80, 32), ("dec0b", 32, 32)]


def _unflatten(p):
    out, k = {}, 0
    for name, ci, co in _LAYERS:
        out[name] = (p[k:k + co * 9 * ci].view(co, 3, 3, ci), p[k + co * 9 * ci:k + co * 9 * ci + co])
        k += co * 9 * ci + co
    out["head"] = (p[k:k + 96].view(3, 32), p[k + 96:k + 99])
    return out


def _conv(x, w, b):
    """3x3 convolution with zero padding of NHWC x, as nine products."""
    n, h, wd, _ = x.shape
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    y = b.expand(n, h, wd, -1)
    for ky in range(3):
        for kx in range(3):
            y = y + xp[:, ky:ky + h, kx:kx + wd] @ w[:, ky, kx].t()
    return torch.relu(y)


def _pack(f):
    rad = torch.log1p(f[..., 0:3].clamp(min=0))
    n = f[..., 7:10]
    ln = n.norm(dim=-1, keepdim=True)
    n = torch.where(ln > 1e-12, n / ln.clamp(min=1e-30), torch.zeros_like(n))
    l1 = n.abs().sum(-1, keepdim=True)
    n = torch.where(l1 > 1e-12, n / l1.clamp(min=1e-30), torch.zeros_like(n))
    x, y, z = n[..., 0], n[..., 1], n[..., 2]
    sx, sy = torch.where(x >= 0, 1.0, -1.0), torch.where(y >= 0, 1.0, -1.0)
    octa = torch.stack([torch.where(z < 0, (1 - y.abs()) * sx, x), torch.where(z < 0, (1 - x.abs()) * sy, y)], -1)
    k = f[..., 11:12]
    std = torch.where(k >= 2, (f[..., 10:11].clamp(min=0) / (k * (k - 1)).clamp(min=1)).sqrt(), torch.zeros_like(k))
    return torch.cat([rad, f[..., 3:6], octa, f[..., 6:7], std], -1)


def _network(p, f):
    """Raw records (n, h, w, 12) -> network output (n, h, w, 3) in log(1 + radiance) space."""
    n, h, w, _ = f.shape
    x = torch.nn.functional.pad(_pack(f), (0, 0, 0, -w % 8, 0, -h % 8))
    q = _unflatten(p)

    def pool(a):
        return a.view(n, a.shape[1] // 2, 2, a.shape[2] // 2, 2, -1).mean((2, 4))

    def up(a):
        return a.repeat_interleave(2, 1).repeat_interleave(2, 2)

    e0 = _conv(_conv(x, *q["enc0a"]), *q["enc0b"])
    e1 = _conv(_conv(pool(e0), *q["enc1a"]), *q["enc1b"])
    e2 = _conv(_conv(pool(e1), *q["enc2a"]), *q["enc2b"])
    m = _conv(_conv(pool(e2), *q["mida"]), *q["midb"])
    d = _conv(_conv(torch.cat([up(m), e2], -1), *q["dec2a"]), *q["dec2b"])
    d = _conv(_conv(torch.cat([up(d), e1], -1), *q["dec1a"]), *q["dec1b"])
    d = _conv(_conv(torch.cat([up(d), e0], -1), *q["dec0a"]), *q["dec0b"])
    out = d @ q["head"][0].t() + q["head"][1] + x[..., :3]
    return out[:, :h, :w]


def exact(case, seed):
    if case["kind"] not in ("denoise", "train"):
        return None
    # the weights, and the rendered frame that the denoiser takes, are inputs: read back as numbers
    s = prepare(case, seed)
    p = torch.from_numpy(s.dn.params()).double().cuda()
    if case["kind"] == "denoise":
        a0, a1 = s.noisy.read_features()
        held = np.full(a0.shape[:2] + (1,), max(case["frames"] - 1, 1), np.float32)
        f = torch.from_numpy(np.concatenate([s.noisy.read()[..., :3], a0, a1[..., :4], held], -1)).double().cuda()
        with torch.no_grad():
            y = torch.expm1(_network(p, f[None])[0]).clamp(min=0)
        return torch.cat([y, torch.ones_like(y[..., :1])], -1)
    feats, target = (torch.from_numpy(a).double().cuda() for a in _crops(case, _rng(case, seed)))
    p.requires_grad_(True)
    out = _network(p, feats)
    if case["loss"] == "relmse":
        t = target.clamp(min=0)
        loss = ((torch.expm1(out) - t) ** 2 / (t * t + 0.01)).mean()
    else:
        loss = ((out - torch.log1p(target.clamp(min=0))) ** 2).mean()
    loss.backward()
    return {"loss": loss.detach(), "grads": p.grad}
