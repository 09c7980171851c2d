"""GPU: traversal with four lanes per ray gives the per-lane traversal's results.

Ray queries of up to 131,072 rays and queue launches with at most 32 rays per
wave take four lanes per ray; larger ones, and the counting variant, one. The
hit is the smallest (t, instance, geometry, primitive) either way, so every
comparison is exact, also for walks deep enough to leave the part of a quad's
stack that LDS holds (96 entries), up to its capacity of 128.
"""
import numpy as np
import pytest

from helios_amd import abi, scenegen

pytestmark = pytest.mark.gpu

QUAD_MAX = 131072


@pytest.fixture(scope="module")
def scene(gpu_ctx):
    from helios_amd import runtime
    s = runtime.Scene(gpu_ctx, scenegen.icosphere_field(seed=3, n_spheres=12, level=3, n_leaves=300))
    yield s
    s.close()


@pytest.mark.parametrize("flags", [0, abi.HH_TRACE_OPAQUE])
def test_ray_queries(scene, flags):
    rays = scenegen.random_rays(QUAD_MAX + 1, (-100.0, 0.5, -100.0), (100.0, 30.0, 100.0), seed=4)
    rays["direction"][::7, 1] = 0.0          # axis-parallel components
    rays["direction"][::11, 0] = -0.0
    rays["tmax"][::5] = 20.0
    rays["tmin"][::13] = -5.0
    want = scene.trace_rays(rays, flags)
    assert 0.2 < np.mean(want["t"] >= 0) < 1.0
    for n in (1, 15, 16, 17, 4097, QUAD_MAX):
        got = scene.trace_rays(rays[:n], flags)
        assert got.tobytes() == want[:n].tobytes(), n


@pytest.mark.parametrize("w,h,frames", [(1, 1, 1), (17, 3, 2), (129, 67, 1), (256, 256, 4)])
def test_frames(gpu_ctx, scene, w, h, frames):
    from helios_amd import runtime
    surf = runtime.Surface(gpu_ctx, w, h)
    it = runtime.PathIntegrator(gpu_ctx)
    it.set_max_ray_bounces(6)
    images = []
    for counting in (False, True):           # the counting variant: one lane per ray
        gpu_ctx.set_profiling(counting=counting)
        it.restart_bake()
        it.render(scene, scene.desc.camera, surf, frames=frames)
        images.append((surf.read(), it.ray_stats()))
    gpu_ctx.set_profiling()
    assert images[0][0].tobytes() == images[1][0].tobytes()
    assert images[0][1] == images[1][1]
    it.close()
    surf.close()


def test_passes_on_both_sides_of_the_head_read(gpu_ctx, scene):
    """A pass of up to about 4 M paths reads a queue head before it claims, a
    longer one does not; the image and the ray counts are the same."""
    from helios_amd import runtime
    surf = runtime.Surface(gpu_ctx, 1920, 1080)
    it = runtime.PathIntegrator(gpu_ctx)
    it.set_max_ray_bounces(3)
    images = []
    for in_flight in (1, 3):                 # 2.07 and 6.2 M paths per pass
        gpu_ctx.set_tuning(frames_in_flight=in_flight)
        it.restart_bake()
        it.render(scene, scene.desc.camera, surf, frames=3)
        images.append((surf.read(), it.ray_stats()))
    gpu_ctx.set_tuning()
    assert images[0][0].tobytes() == images[1][0].tobytes()
    assert images[0][1] == images[1][1]
    it.close()
    surf.close()


@pytest.mark.parametrize("tuning", [dict(), dict(bvh_width=8), dict(bvh_compressed=True)])
@pytest.mark.parametrize("w,h", [(64, 3), (512, 512), (513, 512)])
def test_frames_around_the_merged_launches(gpu_ctx, tuning, w, h):
    """Passes of up to 262,144 paths and longer ones share launches between
    bounces differently, and so do node layouts without quads; the counting
    variant never shares one. The image and the ray counts are the same."""
    from helios_amd import runtime
    before = gpu_ctx.tuning()
    gpu_ctx.set_tuning(**tuning)
    try:
        s = runtime.Scene(gpu_ctx, scenegen.icosphere_field(seed=3, n_spheres=6, level=2, n_leaves=60))
        surf = runtime.Surface(gpu_ctx, w, h)
        it = runtime.PathIntegrator(gpu_ctx)
        it.set_max_ray_bounces(4)
        images = []
        for counting in (False, True):
            gpu_ctx.set_profiling(counting=counting)
            it.restart_bake()
            it.render(s, s.desc.camera, surf)
            images.append((surf.read(), it.ray_stats()))
        gpu_ctx.set_profiling()
        assert images[0][0].tobytes() == images[1][0].tobytes()
        assert images[0][1] == images[1][1]
        for x in (it, surf, s):
            x.close()
    finally:
        gpu_ctx.set_tuning(**before)


def nested(n):
    """n instances, each 1.2 times smaller than the last, of n triangles, each
    1.2 times smaller than the last, all around the origin: binned SAH splits off
    the largest few at a time, so a ray from the origin into +x, which enters
    every box and the smallest ones first, holds 3 siblings per node on the way
    down both trees: 99 entries for n = 140, 121 for 180 and 133 for 200 (a
    transcription of the split and collapse rules). A triangle covers the part of
    its box between a diagonal and a point near it, so the closest hits lie among
    many triangles of the smallest instance, whose boxes are entered first, and
    rays that miss it walk all the others."""
    d = scenegen.SceneDesc(sky=(3.0, 0.1, 1.15, 16))
    d.materials.append(scenegen.material())
    rng = np.random.default_rng(n)
    k = np.arange(n)
    scale = 1.2 ** (n / 2 - k)
    at, off = rng.uniform(0, 1, n), rng.choice([-1.0, 1.0], n) * rng.exponential(0.1, n)
    point = np.clip(np.stack([3 * at - 1 + off, 3 * at - 1 - off], 1), -1, 2)
    pos = np.ones((n, 3, 3))
    pos[:, 0, 1:], pos[:, 1, 1:], pos[:, 2, 1:] = -1.0, 2.0, point
    pos = (pos * scale[:, None, None]).reshape(-1, 3)
    flat = np.tile([-1.0, 0.0, 0.0], (3 * n, 1))
    d.meshes.append(scenegen._mesh_from_parts([(pos, flat, np.zeros((3 * n, 2)), np.arange(3 * n, dtype=np.uint32), 0)], [0]))
    for s in scale:
        d.instances.append((*scenegen.trs(scale=s), 0, -1))
    return d


def into_x(n):
    rng = np.random.default_rng(n)
    rays = np.zeros(n, abi.RAY_DTYPE)
    rays["direction"][:, 0] = 1.0
    y = rng.uniform(-1.1, 2.1, n)
    rays["direction"][:, 1] = y
    rays["direction"][:, 2] = y + rng.normal(0, 0.2, n)
    rays["tmax"] = 1e15
    return rays


@pytest.mark.parametrize("n", [140, 180])
def test_walks_that_leave_lds(gpu_ctx, n):
    from helios_amd import runtime
    scene = runtime.Scene(gpu_ctx, nested(n))
    rays = into_x(2048)
    want = scene.trace_rays(np.resize(rays, QUAD_MAX + 1))[:len(rays)]     # one lane per ray
    hit = want["t"] >= 0
    assert 0.3 < hit.mean() < 1.0 and len(np.unique(want["primitive"][hit])) > 16
    got = scene.trace_rays(rays)
    assert got.tobytes() == want.tobytes()
    assert scene.traversal_faults() == dict(lane_stack=0, packet_stack=0, trips=0)
    scene.close()


def test_a_full_stack_ends_the_ray(gpu_ctx):
    """A walk that needs more than 128 entries is ended and counted."""
    from helios_amd import runtime
    scene = runtime.Scene(gpu_ctx, nested(220))
    scene.trace_rays(into_x(256))
    assert scene.traversal_faults()["lane_stack"] > 0
    scene.close()
