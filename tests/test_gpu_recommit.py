"""GPU: a scene committed again after an edit equals the edited scene committed once.

A commit rebuilds what its edits touch (geometry, environment, tables and
TLAS); images, lights, environment and hits must be those of a scene built
from the edited description, under every BVH tuning, and the images of the
captured launch sequences that outlive a commit must follow it.
"""
import numpy as np
import pytest

from helios_amd import abi, scenegen

pytestmark = pytest.mark.gpu


def describe(**edit):
    d = scenegen.icosphere_field(seed=5, n_spheres=6, level=2, n_leaves=40, width=96, height=64, max_ray_bounces=4)
    d.sky = (3.0, 0.1, 1.15, 32)
    if "move" in edit:
        model, normal = scenegen.trs((4.0, 9.0, -3.0), None, 5.0)
        d.instances[2] = (model, normal, d.instances[2][2], -1)
    if "light" in edit:
        d.lights.append(dict(d.lights[-1], position=(0.0, 20.0, 0.0), intensity=900.0))
    if "sky" in edit:
        d.sky = (6.0, 0.3, 1.15, 48)
    if "mesh" in edit:
        d.materials.append(scenegen.material((0.2, 0.4, 0.9, 1.0), emissive=(2.0, 1.0, 0.5, 1.0)))
        m = scenegen.displaced_sphere_mesh(2, 77, 0.1)
        m.materials = [len(d.materials) - 1]
        d.instances.append((*scenegen.trs((0.0, 25.0, 20.0), None, 6.0), len(d.meshes), -1))
        d.meshes.append(m)
    return d


def apply(scene, kind, d):
    from helios_amd import runtime
    L, out = runtime.lib(), runtime.C.c_uint32()
    if kind == "move":
        model, normal = (np.ascontiguousarray(x, np.float32) for x in d.instances[2][:2])
        runtime.check(L.hh_scene_set_instance_transform(scene.h, 2, abi.ptr(model), abi.ptr(normal)))
    elif kind == "light":
        runtime.check(L.hh_scene_add_light(scene.h, runtime.C.byref(runtime._struct(abi.LightDesc, d.lights[-1])),
                                           runtime.C.byref(out)))
    elif kind == "sky":
        runtime.check(L.hh_scene_set_sky(scene.h, runtime.C.byref(abi.SkyParams(*d.sky))))
    elif kind == "mesh":
        tail = scenegen.SceneDesc(materials=d.materials[-1:], meshes=d.meshes[-1:], instances=d.instances[-1:], sky=d.sky)
        scene.load(tail)
    scene.commit()


def shown(ctx, scene, d, surf, it):
    it.restart_bake()
    it.render(scene, d.camera, surf, frames=2)
    env = scene.env()
    return surf.read().tobytes(), scene.lights().tobytes(), env.tobytes(), \
        scene.primary_hits(d.camera, 48, 32).tobytes(), scene.bvh_stats()


@pytest.mark.parametrize("tuning", [dict(), dict(bvh_width=8), dict(bvh_compressed=True), dict(bvh_builder=1)])
@pytest.mark.parametrize("kinds", [("move",), ("light",), ("sky",), ("mesh",), ("move", "mesh", "light", "move")])
def test_recommit_equals_fresh(gpu_ctx, tuning, kinds):
    from helios_amd import runtime
    before = gpu_ctx.tuning()
    gpu_ctx.set_tuning(**tuning)
    try:
        scene = runtime.Scene(gpu_ctx, describe())
        surf = runtime.Surface(gpu_ctx, 96, 64)
        it = runtime.PathIntegrator(gpu_ctx)
        it.set_max_ray_bounces(4)
        first = shown(gpu_ctx, scene, scene.desc, surf, it)
        for n in range(len(kinds)):
            d = describe(**{k: True for k in kinds[:n + 1]})
            apply(scene, kinds[n], d)
            fresh = runtime.Scene(gpu_ctx, d)
            got, want = shown(gpu_ctx, scene, d, surf, it), shown(gpu_ctx, fresh, d, surf, it)
            assert got == want, kinds[n]
            fresh.close()
        assert got[0] != first[0]
        # another tuning at the next commit
        gpu_ctx.set_tuning(bvh_width=12 - (tuning.get("bvh_width", 4)))
        scene.commit()
        assert shown(gpu_ctx, scene, d, surf, it)[0] == got[0]
        for x in (it, surf, scene):
            x.close()
    finally:
        gpu_ctx.set_tuning(**before)


@pytest.mark.parametrize("n", [1, 2, 3, 64, 512, 513, 1025])
def test_tlas_sizes(gpu_ctx, n):
    """TLAS ranges around one workgroup's 512 primitives: hits of n instances
    from the GPU builder equal those from the host builder."""
    from helios_amd import runtime
    n = min(n, 1024)
    d = scenegen.SceneDesc(sky=(3.0, 0.1, 1.15, 16))
    d.materials.append(scenegen.material())
    m = scenegen.displaced_sphere_mesh(1, 3, 0.05)
    m.materials = [0]
    d.meshes.append(m)
    rng = np.random.default_rng(n)
    for _ in range(n):
        d.instances.append((*scenegen.trs(rng.uniform(-20, 20, 3), None, rng.uniform(0.5, 2.0)), 0, -1))
    rays = scenegen.random_rays(4096, (-25, -25, -25), (25, 25, 25), seed=n)
    before = gpu_ctx.tuning()
    hits = []
    for builder in (3, 1):
        gpu_ctx.set_tuning(bvh_builder=builder)
        s = runtime.Scene(gpu_ctx, d)
        hits.append(s.trace_rays(rays))
        s.close()
    gpu_ctx.set_tuning(**before)
    assert hits[0].tobytes() == hits[1].tobytes()
    assert np.any(hits[0]["t"] >= 0)
