// A stand-in for the HIP runtime and the library's kernels, for tests of the
// host code in api.hip without a GPU: device memory is host memory filled with
// a poison byte, copies are memcpy, and each kernel launcher marks what its
// kernel would write. Every call that can fail on a GPU counts down
// `stub_fail_at`; the one that reaches zero fails.
//
// Only what the test programs reach is defined; the programs are linked with
// unresolved symbols allowed.
#include <cstdlib>
#include <cstring>
#include <map>

#define __bf16 uint16_t   // g++ has no such type; the denoiser's pointers are not used here
#include "../../helios_amd/csrc/internal.hpp"
#include "hip_stub.hpp"

long stub_fail_at = 0;
long stub_calls = 0;
int stub_graphs_alive = 0;
int stub_graph_launches = 0;
hh::SceneGPU stub_scene;

static std::map<char*, size_t> g_alloc;

static hipError_t may_fail() {
    stub_calls++;
    return stub_fail_at > 0 && --stub_fail_at == 0 ? hipErrorOutOfMemory : hipSuccess;
}

bool stub_range_written(const void* p, size_t bytes) {
    if (bytes == 0) return true;
    auto it = g_alloc.upper_bound((char*)p);
    if (it == g_alloc.begin()) return false;
    --it;
    if ((char*)p + bytes > it->first + it->second) return false;
    // a 16-byte unit still all poison was never written
    for (size_t i = 0; i + 16 <= bytes; i += 16) {
        bool poison = true;
        for (size_t k = 0; k < 16; k++) poison = poison && ((const unsigned char*)p)[i + k] == kStubPoison;
        if (poison) return false;
    }
    return true;
}

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    if (may_fail() != hipSuccess) return hipErrorOutOfMemory;
    *p = std::aligned_alloc(256, (n + 255) / 256 * 256);
    std::memset(*p, kStubPoison, n);
    g_alloc[(char*)*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (p && g_alloc.erase((char*)p) == 0) std::abort();   // freed twice, or never allocated
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    if (may_fail() != hipSuccess) return hipErrorUnknown;
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
    *v = 2;   // CUs: small launch buffers
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static char area[16];
    *p = area;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = (hipStream_t)std::malloc(1);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    std::free((void*)s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = (hipEvent_t)std::malloc(1);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    std::free((void*)e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    *g = (hipGraph_t)std::malloc(1);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    *x = (hipGraphExec_t)std::malloc(1);
    stub_graphs_alive++;
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
    stub_graph_launches++;
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x) {
    std::free((void*)x);
    stub_graphs_alive--;
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
    std::free((void*)g);
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) {
    static void* h = nullptr;
    return &h;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
}

namespace hh {
void BuildScratch::release() {}
void BuildScratch::release_ploc() {}
void BuildScratch::release_sah() {}
hipError_t launch_soup(hipStream_t, const SoupRange*, uint32_t, uint32_t n, const float4*, const uint32_t*, float4* tri,
                       float4* shade) {
    std::memset((void*)tri, 1, size_t(n) * 48);
    std::memset((void*)shade, 1, size_t(n) * 64);
    return may_fail();
}
// One node per mesh.
hipError_t build_blas_forest(hipStream_t, int width, int, const std::vector<int2>& meshes, uint32_t total, const float4*,
                             float4* tris, const float4*, float4* shade, void* nodes, uint32_t node_base, BuildScratch&,
                             uint32_t* num_nodes, float* boxes) {
    const size_t nb = width == 8 ? sizeof(WideNode<8>) : sizeof(WideNode<4>);
    std::memset((char*)nodes + node_base * nb, 2, meshes.size() * nb);
    std::memset((void*)tris, 2, size_t(total) * 48);
    std::memset((void*)shade, 2, size_t(total) * 64);
    *num_nodes = (uint32_t)meshes.size();
    for (size_t g = 0; g < meshes.size(); g++)
        for (int k = 0; k < 6; k++) boxes[6 * g + k] = k < 3 ? -1.0f : 1.0f;
    return may_fail();
}
// One node.
hipError_t build_tlas(hipStream_t, int width, uint32_t, const float*, const float*, void* nodes, uint32_t node_base,
                      BuildScratch&, uint32_t* num_nodes, bool, bool, bool) {
    const size_t nb = width == 8 ? sizeof(WideNode<8>) : sizeof(WideNode<4>);
    if (may_fail() != hipSuccess) return hipErrorOutOfMemory;
    std::memset((char*)nodes + node_base * nb, 3, nb);
    *num_nodes = 1;
    return hipSuccess;
}
hipError_t quantize_bvh4(hipStream_t, const void* src, void* dst, uint32_t n) {
    if (n == 0) return hipSuccess;
    if (may_fail() != hipSuccess) return hipErrorUnknown;
    if (!stub_range_written(src, n * sizeof(WideNode<4>))) return hipErrorInvalidValue;
    std::memset(dst, 4, n * sizeof(QNode4));
    return hipSuccess;
}
hipError_t launch_fill_f4(hipStream_t, float4* p, float4 v, uint32_t n) {
    if (may_fail() != hipSuccess) return hipErrorUnknown;
    for (uint32_t i = 0; i < n; i++) p[i] = v;
    return hipSuccess;
}
void sky_coefficients(float, float, float, const float*, float* out) { std::memset(out, 0, 30 * sizeof(float)); }
hipError_t launch_sky_bake(hipStream_t, float4* cube, uint32_t size, const float*, const float*) {
    if (may_fail() != hipSuccess) return hipErrorUnknown;
    std::memset((void*)cube, 5, size_t(6) * size * size * sizeof(float4));
    return hipSuccess;
}
hipError_t launch_frame(const LaunchCfg&, const SceneGPU*, const SceneGPU* scenes, const ViewGPU*, const ViewGPU*, uint32_t,
                        uint32_t, uint32_t, Wavefront&, bool) {
    stub_scene = scenes[0];
    return hipSuccess;
}
}  // namespace hh
