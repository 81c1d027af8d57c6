// sicp_internal.hpp — host-side objects behind the opaque C ABI handles.
#pragma once

#include <atomic>
#include <vector>

#include "sicp_kernels.hpp"

struct sicp_map {
    sicp_map_config cfg;
    sicp::MapDev dev;
    sicp::MapCounters* ctr = nullptr;  // device
    sicp::AllocScratch alloc{};
    sicp_block* visible = nullptr;     // device, num_blocks
    uint32_t* unify_snap = nullptr;    // neighbour label pass: label snapshot, num_blocks * 512
    uint32_t* unify_mark = nullptr;    // per heap slot: the pass of its last snapshot; then the
                                       // pass under way and the last one that ended
    std::atomic<bool> mesh_lent{false};  // mesh extraction: the memory below is in a call's use
    uint32_t* mesh_counts = nullptr;   // device
    uint32_t* mesh_total = nullptr;    // pinned host
    std::vector<void*> owned;          // every other device allocation of the map
};

namespace sicp {

// Pinned host memory that a call's last kernel writes its results into, so the
// call ends with one synchronisation and no copy (a copy to pageable memory is
// a launch, a staging buffer and a wait of its own). Lent from a pool of at
// most kHostLoansKept idle buffers, one to a call at a time; more calls at
// once get buffers of their own, freed when they end. The idle ones are freed
// with the last map (host_loans_release): freed with each, the next step of
// every other caller took 65 us after a map's end, 46 with the copy. Usable from every device. Without memory for one,
// `ptr` stays null and the call copies. Measured per call: ICPStep at 160x120
// 35 us with the copy, 26 with the loan; RGBStep at 320x240 (two copies) 61,
// 39; a frame's result (three copies) 42 us less.
constexpr size_t kHostLoanBytes = 2048;
constexpr int kHostLoansKept = 16;
struct HostLoan {
    void* ptr = nullptr;
    HostLoan() = default;
    HostLoan(const HostLoan&) = delete;
    HostLoan& operator=(const HostLoan&) = delete;
    void take();
    // Waits for the stream, then copies its first `bytes`.
    int wait(void* dst, size_t bytes, hipStream_t s);
    ~HostLoan();
};
void host_loans_retain();  // a map begins
void host_loans_release();  // and ends

int map_alloc(const sicp_map_config& cfg, sicp_map** out);
void map_free(sicp_map* m);
// The neighbour label pass over the map's visible list (unify.hip), and its
// scratch, allocated with the map where every fusion runs the pass (no later
// call allocates then), else by the first pass.
int unify_scratch(sicp_map* map);
int launch_unify(sicp_map* map, const int* gate, hipStream_t s);
// `queue_cleared`: the hand-over queue count was cleared by launch_fuse_count
// on the same stream.
int launch_raycast_gated(MapDev m, View<float4> vmap, View<float4> nmap, View<float> zmin,
                         View<float> zmax, PoseArg pose, float invfx, float invfy, float cx,
                         float cy, const int* gate, const uint32_t* nonempty, hipStream_t s,
                         bool queue_cleared = false, RayTuning tune = RayTuning{});

// ICPStep over the four maps with `partials_dev` as the workgroups' partial
// rows (sicp_icp_step and its variants). `allocates` false: host results are
// copied instead of written to a HostLoan, whose pool may allocate.
int icp_step(sicp_image vcurr, sicp_image vlast, sicp_image ncurr, sicp_image nlast,
             const sicp_pose_f* curr, const sicp_pose_f* last, sicp_intrinsics K,
             void* partials_dev, float* sums_dev, float* host_sums, double* A_host,
             double* b_host, float* residual_host, bool k32, void* stream,
             bool allocates = true);
// The largest image sicp_icp_step_static takes (the kernels index pixels
// with 32-bit integers).
constexpr int64_t kIcpStaticMaxPixels = (int64_t)1 << 30;

// A pitched device image owned by the library.
template <class T> struct DevImage {
    void* ptr = nullptr;
    size_t pitch = 0;
    int cols = 0, rows = 0;
    int create(int c, int r, size_t elem = sizeof(T)) {
        cols = c;
        rows = r;
        hipError_t e = hipMallocPitch(&ptr, &pitch, (size_t)c * elem, (size_t)(r > 0 ? r : 1));
        if (e != hipSuccess) return hip_fail(e, "hipMallocPitch");
        return SICP_OK;
    }
    void release() {
        if (ptr) (void)hipFree(ptr);
        ptr = nullptr;
    }
    View<T> v() const { return View<T>{(char*)ptr, pitch, cols, rows}; }
    sicp_image img() const { return sicp_image{ptr, pitch, cols, rows}; }
};

}  // namespace sicp
