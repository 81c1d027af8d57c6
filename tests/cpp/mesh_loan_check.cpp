// Host side of the mesh extraction (mesh.hip, compiled for the host alone)
// against a stand-in HIP runtime that logs what is queued and fails where it
// is told to: memory that queued kernels may still write is lent to the next
// call only after the stream has been waited for, or not at all.
//
// Usage: mesh_loan_check <check that fails, 1..3, 0: none> <the wait fails, 0/1>
// Prints "ok", or what is wrong.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <string>

#include "../../semantic_icpslam_amd/csrc/sicp_internal.hpp"

namespace {
int g_checks = 0, g_fail_check = 0, g_queued = 0;
bool g_fail_wait = false;
void* g_counts = nullptr;  // first launch's argument: the counts in use
}  // namespace

// ---- the stand-in runtime: what launch_mesh calls ---------------------------
extern "C" {
void** __hipRegisterFatBinary(const void*) { return (void**)calloc(1, sizeof(void*)); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*,
                           void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* n, hipStream_t* s) {
    *g = *b = dim3(1);
    *n = 0;
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void** args, size_t, hipStream_t) {
    // the reset's only argument starts with the counts' address
    if (g_queued++ == 0) g_counts = *(void**)args[0];
    return hipSuccess;
}
hipError_t hipGetLastError() {
    return ++g_checks == g_fail_check ? hipErrorUnknown : hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    if (g_fail_wait) return hipErrorUnknown;
    g_queued = 0;
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
    *p = calloc(1, n);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = calloc(1, n);
    return hipSuccess;
}
hipError_t hipFree(void*) { return hipSuccess; }      // kept, so that no address comes back
hipError_t hipHostFree(void*) { return hipSuccess; }
}

namespace sicp {
int hip_fail(hipError_t, const char*) { return 2; }
int invalid(const char*) { return 1; }
int launch_mesh(sicp_map*, float*, float*, uint8_t*, uint32_t, uint32_t*, uint32_t*, hipStream_t);
}  // namespace sicp

static int wrong(const std::string& what) {
    std::printf("%s\n", what.c_str());
    return 1;
}

int main(int argc, char** argv) {
    if (argc != 3) return wrong("two arguments");
    sicp_map map;
    map.cfg = sicp_map_config{};
    map.cfg.num_blocks = 1000;
    uint32_t n = 0, total = 0;
    auto call = [&] {
        g_checks = 0;
        return sicp::launch_mesh(&map, nullptr, nullptr, nullptr, 0, &n, &total, nullptr);
    };
    if (call() != 0) return wrong("first call failed");
    void* const kept = g_counts;
    if (call() != 0 || g_counts != kept) return wrong("the memory is not kept");

    g_fail_check = std::atoi(argv[1]);
    g_fail_wait = std::atoi(argv[2]) != 0;
    const bool fails = g_fail_check != 0 || g_fail_wait;
    if ((call() != 0) != fails) return wrong("the failure does not reach the caller");
    const bool in_flight = g_queued != 0;
    g_fail_check = 0;
    g_fail_wait = false;
    g_queued = 0;
    if (call() != 0) return wrong("the call after a failed one fails");
    if (in_flight && g_counts == kept) return wrong("memory lent again under queued kernels");
    if (map.mesh_lent.load()) return wrong("the memory stays lent");
    std::printf("ok\n");
    return 0;
}
