// A commit that fails at any of its GPU calls, followed by one that succeeds,
// must leave a scene whose device memory is written in full: for every call k
// of a commit (first commits, and commits after each kind of edit), call k is
// made to fail and the commit repeated. Prints one line per fault found.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <string>
#include <vector>

#include "../../include/helios_hip.h"
#include "hip_stub.hpp"

static int faults = 0;
#define NEED(x)                                                                    \
    do {                                                                           \
        if (!(x)) {                                                                \
            std::printf("%s:%d: %s (%s)\n", __FILE__, __LINE__, #x, hh_last_error()); \
            std::fflush(stdout);                                                   \
            std::exit(2);                                                          \
        }                                                                          \
    } while (0)

static void identity(float m[16]) {
    std::memset(m, 0, 64);
    m[0] = m[5] = m[10] = m[15] = 1.0f;
}

static void add_mesh_and_instance(hh_scene s) {
    hh_material_desc md{};
    md.albedo_texture = md.normal_texture = md.roughness_texture = md.metallic_texture = md.emissive_texture = -1;
    uint32_t mat, mesh, inst;
    NEED(hh_scene_add_material(s, &md, &mat) == HH_OK);
    hh_vertex v[4];
    std::memset(v, 0, sizeof(v));
    for (int k = 0; k < 4; k++) {
        v[k].position[0] = (float)(k & 1);
        v[k].position[1] = (float)(k >> 1);
    }
    const uint32_t idx[6] = {0, 1, 2, 1, 3, 2};
    hh_submesh sm{};
    sm.index_count = 6;
    NEED(hh_scene_add_mesh(s, v, 4, idx, 6, &sm, 1, &mat, 1, &mesh) == HH_OK);
    hh_instance_desc in{};
    in.mesh = mesh;
    in.material_override = -1;
    identity(in.model);
    identity(in.normal);
    NEED(hh_scene_add_instance(s, &in, &inst) == HH_OK);
}
static void add_sun(hh_scene s) {
    hh_light_desc l{};
    l.type = HH_LIGHT_DIRECTIONAL;
    l.forward[1] = -1.0f;
    l.intensity = 1.0f;
    uint32_t id;
    NEED(hh_scene_add_light(s, &l, &id) == HH_OK);
}
static void move(hh_scene s) {
    float m[16], n[16];
    identity(m);
    identity(n);
    m[12] = 3.0f;
    NEED(hh_scene_set_instance_transform(s, 0, m, n) == HH_OK);
}

// Every array of the committed scene a kernel reads was written.
static void check(hh_context ctx, hh_scene s, const char* what, long k) {
    uint64_t st[4];
    NEED(hh_scene_bvh_stats(s, st) == HH_OK);
    hh_integrator it;
    hh_surface surf;
    NEED(hh_integrator_create(ctx, &it) == HH_OK);
    NEED(hh_surface_create(ctx, 8, 8, &surf) == HH_OK);
    const hh_camera cam{{0, 0, 5}, {0, 0, 0, 1}, 60.0f, 0.1f, 100.0f, 1.0f, 0.0f};
    std::memset(&stub_scene, 0, sizeof(stub_scene));
    NEED(hh_integrator_render(it, s, &cam, surf) == HH_OK);
    const hh::SceneGPU& g = stub_scene;
    const size_t nodes = st[0] + st[2], tris = st[1];
    const size_t nb = g.bvh_width == hh::kLayoutQ4 ? 64 : (g.bvh_width == hh::kLayoutB8 ? 256 : 128);
    const struct { const char* name; bool ok; } parts[] = {
        {"nodes", stub_range_written(g.nodes, nodes * nb)},
        {"triangles", stub_range_written(g.tris, tris * 48)},
        {"shading records", stub_range_written(g.shade, tris * 64)},
        {"vertices", stub_range_written(g.vtx, tris / 2 * 4 * 80)},
        {"indices", stub_range_written(g.idx, tris * 3 * 4)},
        {"instances", stub_range_written(g.inst_trav, st[3] * sizeof(hh::InstTrav))},
        {"environment", stub_range_written(g.env, size_t(6) * g.env_size * g.env_size * 16)},
    };
    for (const auto& p : parts)
        if (!p.ok) {
            faults++;
            std::printf("%s, call %ld failed: %s unwritten after the next commit\n", what, k, p.name);
        }
    hh_surface_destroy(surf);
    hh_integrator_destroy(it);
}

int main() {
    const struct { const char* name; uint32_t width, compressed; } tunings[] = {
        {"BVH4", 4, 0}, {"compressed BVH4", 4, 1}, {"BVH8", 8, 0}};
    const struct { const char* name; std::function<void(hh_scene)> edit; } edits[] = {
        {"first commit", nullptr}, {"moved instance", move}, {"added mesh", add_mesh_and_instance}, {"added sun", add_sun}};
    int tried = 0;
    for (const auto& t : tunings)
        for (const auto& e : edits) {
            const std::string what = std::string(t.name) + ", " + e.name;
            for (long k = 1;; k++) {
                hh_context ctx;
                hh_scene s;
                NEED(hh_context_create(0, &ctx) == HH_OK);
                hh_tuning tn;
                NEED(hh_context_get_tuning(ctx, &tn) == HH_OK);
                tn.bvh_width = t.width;
                tn.bvh_compressed = t.compressed;
                NEED(hh_context_set_tuning(ctx, &tn) == HH_OK);
                NEED(hh_scene_create(ctx, &s) == HH_OK);
                const hh_sky_params sky{3.0f, 0.1f, 1.15f, 16};
                NEED(hh_scene_set_sky(s, &sky) == HH_OK);
                add_mesh_and_instance(s);
                add_mesh_and_instance(s);
                if (e.edit) {
                    NEED(hh_scene_commit(s) == HH_OK);
                    e.edit(s);
                }
                stub_fail_at = k;
                const hh_status st = hh_scene_commit(s);
                const bool reached = stub_fail_at == 0;
                stub_fail_at = 0;
                if (reached) {
                    NEED(st != HH_OK);   // a failed call is reported
                    uint64_t stats[4];
                    NEED(hh_scene_bvh_stats(s, stats) == HH_ERR_NOT_READY);
                    NEED(hh_scene_commit(s) == HH_OK);
                    tried++;
                }
                check(ctx, s, what.c_str(), reached ? k : 0);
                hh_scene_destroy(s);
                hh_context_destroy(ctx);
                if (!reached) break;
            }
        }
    std::printf("%d failed commits repeated, %d faults\n", tried, faults);
    return faults ? 1 : 0;
}
