// Captured launch sequences of a context: one per shape of pass, at most 64 at a
// time, kept over commits and for other surfaces of the same size.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../include/helios_hip.h"
#include "hip_stub.hpp"

#define NEED(x)                                                        \
    do {                                                               \
        if (!(x)) {                                                    \
            std::printf("line %d: %s (%d sequences alive, %d launches)\n", __LINE__, #x, stub_graphs_alive, stub_graph_launches); \
            std::exit(1);                                              \
        }                                                              \
    } while (0)

int main() {
    hh_context ctx;
    hh_scene s;
    hh_integrator it;
    NEED(hh_context_create(0, &ctx) == HH_OK);
    NEED(hh_scene_create(ctx, &s) == HH_OK);
    const hh_sky_params sky{3.0f, 0.1f, 1.15f, 16};
    NEED(hh_scene_set_sky(s, &sky) == HH_OK);
    NEED(hh_scene_commit(s) == HH_OK);
    NEED(hh_integrator_create(ctx, &it) == HH_OK);
    const hh_camera cam{{0, 0, 5}, {0, 0, 0, 1}, 60.0f, 0.1f, 100.0f, 1.0f, 0.0f};
    auto surface = [&](uint32_t w, uint32_t h) {
        hh_surface f;
        NEED(hh_surface_create(ctx, w, h, &f) == HH_OK);
        return f;
    };
    auto render = [&](hh_surface f) { NEED(hh_integrator_render(it, s, &cam, f) == HH_OK); };

    std::vector<hh_surface> surfs{surface(256, 256)};   // the largest first: buffers do not grow after it
    render(surfs[0]);
    NEED(stub_graphs_alive == 1 && stub_graph_launches == 1);
    render(surfs[0]);
    surfs.push_back(surface(256, 256));
    render(surfs[1]);
    NEED(stub_graphs_alive == 1 && stub_graph_launches == 3);   // other surface, same shape
    NEED(hh_scene_set_sky(s, &sky) == HH_OK);
    NEED(hh_scene_commit(s) == HH_OK);
    render(surfs[0]);
    NEED(stub_graphs_alive == 1 && stub_graph_launches == 4);   // kept over the commit

    int most = 0;
    for (uint32_t w = 8; w < 8 + 150; w++) {
        surfs.push_back(surface(w, 4));
        render(surfs.back());
        most = stub_graphs_alive > most ? stub_graphs_alive : most;
    }
    NEED(most == 64);
    NEED(stub_graph_launches == 154);
    for (hh_surface f : surfs) hh_surface_destroy(f);
    hh_integrator_destroy(it);
    hh_scene_destroy(s);
    hh_context_destroy(ctx);
    NEED(stub_graphs_alive == 0);
    return 0;
}
