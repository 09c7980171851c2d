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


def same_as_the_host_builder(gpu_ctx, d, rays):
    from helios_amd import runtime
    before = gpu_ctx.tuning()
    hits = []
    for builder in (3, 1):
        gpu_ctx.set_tuning(bvh_builder=builder)
        s = runtime.Scene(gpu_ctx, d)
        hits.append((s.trace_rays(rays), s.bvh_stats()))
        s.close()
    gpu_ctx.set_tuning(**before)
    assert hits[0][0].tobytes() == hits[1][0].tobytes()
    assert hits[0][1] == hits[1][1]
    assert np.any(hits[0][0]["t"] >= 0)


@pytest.mark.parametrize("n", [1, 2, 3, 64, 512, 513, 1023, 1024])
def test_tlas_sizes(gpu_ctx, n):
    """TLAS ranges around one and two workgroups' 512 primitives, up to the limit
    of 1,024 instances: hits and node counts of the GPU builder equal the host
    builder's."""
    d = scenegen.SceneDesc(sky=(3.0, 0.1, 1.15, 16))
    d.materials.append(scenegen.material())
    m = scenegen.displaced_sphere_mesh(1, 3, 0.05)
    m.materials = [0]
    d.meshes.append(m)
    rng = np.random.default_rng(n)
    for _ in range(n):
        d.instances.append((*scenegen.trs(rng.uniform(-20, 20, 3), None, rng.uniform(0.5, 2.0)), 0, -1))
    same_as_the_host_builder(gpu_ctx, d, scenegen.random_rays(4096, (-25, -25, -25), (25, 25, 25), seed=n))


@pytest.mark.parametrize("n", [1, 2, 511, 512, 513, 1024, 1025, 4097])
def test_blas_sizes(gpu_ctx, n):
    """The same for the triangles of one mesh (beside a mesh of one triangle)."""
    d = scenegen.SceneDesc(sky=(3.0, 0.1, 1.15, 16))
    d.materials.append(scenegen.material())
    rng = np.random.default_rng(n)
    for k in (n, 1):
        pos = (rng.uniform(-10, 10, (k, 1, 3)) + rng.normal(0, 1, (k, 3, 3))).reshape(-1, 3)
        up = np.tile([0.0, 1.0, 0.0], (3 * k, 1))
        d.meshes.append(scenegen._mesh_from_parts([(pos, up, np.zeros((3 * k, 2)), np.arange(3 * k, dtype=np.uint32), 0)], [0]))
        d.instances.append((*scenegen.trs((0.0, 0.0, 0.0)), len(d.meshes) - 1, -1))
    same_as_the_host_builder(gpu_ctx, d, scenegen.random_rays(4096, (-12, -12, -12), (12, 12, 12), seed=n))


def test_more_shapes_than_sequences_are_kept(gpu_ctx):
    """A context keeps 64 captured launch sequences; frames of 70 shapes drop
    them on the way, and the first shape's image is the same after that."""
    from helios_amd import runtime
    d = scenegen.icosphere_field(seed=5, n_spheres=3, level=1, n_leaves=10)
    scene = runtime.Scene(gpu_ctx, d)
    it = runtime.PathIntegrator(gpu_ctx)
    it.set_max_ray_bounces(3)

    surfs = {w: runtime.Surface(gpu_ctx, w, 5) for w in range(16, 16 + 71)}   # destroying one drops sequences too

    def image(w):
        it.restart_bake()
        it.render(scene, d.camera, surfs[w], frames=2)
        return surfs[w].read()

    first = image(16)
    for w in list(surfs)[1:]:
        image(w)
    assert image(16).tobytes() == first.tobytes()
    for x in (it, *surfs.values(), scene):
        x.close()
