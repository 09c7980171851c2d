#pragma once
#include <cstddef>

#include "../../helios_amd/csrc/gpu_scene.hpp"

constexpr unsigned char kStubPoison = 0xCD;   // what device memory holds until it is written
extern long stub_fail_at;                     // the call that fails (0: none)
extern long stub_calls;                       // calls that could have failed
extern int stub_graphs_alive, stub_graph_launches;
extern hh::SceneGPU stub_scene;               // the scene of the last frame launched or captured
// Whether every 16-byte unit of the range lies in one live allocation and was written.
bool stub_range_written(const void* p, size_t bytes);
