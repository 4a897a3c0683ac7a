// Internal declarations shared by the HIP sources of libcqx.so.
#pragma once

#include "cqx_internal.h"
#include "trace_ranges.h"
#include "traverse_core.h"
#include "walk_packed.h"

#include <hip/hip_runtime.h>

#include <memory>
#include <vector>

#define HIP_TRY(expr)                                                                                            \
    do {                                                                                                         \
        hipError_t e_ = (expr);                                                                                  \
        if (e_ != hipSuccess) return cqx::fail(CQX_ERR_HIP, "%s failed: %s", #expr, hipGetErrorString(e_));     \
    } while (0)

namespace cqx {

struct PtPlan; // path-tracer buffers and captured graph (pathtrace.hip)
void destroy_pt_plan(PtPlan* plan);
bool plan_holds(const PtPlan* plan, const cqx_dvolume* vol); // whether the plan's graphs walk this volume
struct DemoPlan; // buffers of the reference-shading mode (demo.hip)
void destroy_demo_plan(DemoPlan* plan);
struct DeviceEdits; // a volume's on-device edit state (edits_gpu.hip)
void destroy_device_edits(DeviceEdits* e);
void forget_nodes(DeviceEdits* e, uint64_t first); // nodes from `first` on are replaced (the device is idle)

// Best-effort release paths: an error here has nowhere useful to go.
inline void release(void* p) { (void)hipFree(p); }

constexpr uint32_t kDefaultMaxIters = 1u << 22;

} // namespace cqx

struct cqx_ctx {
    int device = 0;
    int cu_count = 0;
    int lds_per_block = 0;
    uint64_t* d_counter = nullptr; // work counters of the persistent kernel (8 queues, 128 B apart)
    void* scratch = nullptr;       // staging for cqx_intersect_host
    size_t scratch_bytes = 0;
    void* pinned = nullptr; // host memory the GPU reads and writes: rays and records of small cqx_intersect_host calls
    size_t pinned_bytes = 0;
    void* bins = nullptr; // ray binning: cell counts/offsets, then the order (u32) and cells (u16) of n rays
    size_t bins_bytes = 0;
    hipStream_t capture_stream = nullptr; // private stream for graph capture
    cqx::PtPlan* pt_plan = nullptr;
    cqx::DemoPlan* demo_plan = nullptr;
    void* batch_desc = nullptr; // descriptor table of the batched launch
    size_t batch_bytes = 0;
    void* noalloc_scratch = nullptr; // this device's static scratch (cqx_intersect_noalloc), not owned
    struct Tuned {
        int height; // SubDAG height of the volume tuned on
        int cls;    // batch-size class: floor(log2 n)
        cqx_launch_cfg cfg;
        float ms;
    };
    std::vector<Tuned> tuned; // autotuner cache
};

struct cqx_dvolume {
    uint32_t* nodes = nullptr;
    cqx_subdag* sub = nullptr;
    uint64_t node_count = 0;
    uint64_t capacity = 0; // nodes the device buffer holds (headroom for appended edits)
    uint64_t uploaded = 0; // nodes of the upload: these may have later ones as children, appended ones may not
    // The packed copy of the store (walk_packed.h): present for stores of at most 2^24 nodes, used
    // when packed_ok (the SubDAGs lie within its coordinate limit).
    uint32_t* packed = nullptr;
    uint64_t packed_capacity = 0;
    uint64_t packed_count = 0; // nodes [0, packed_count) of the copy are as the store's
    bool packed_ok = false;
    uint32_t root = 0;
    cqx_subdag hsub[8];
    int max_height = 0; // largest SubDAG start height (stack rows needed: max_height + 1)
    cqx::DeviceEdits* edits = nullptr; // index and buffers of on-device edits, made on first use
};

namespace cqx {

// Autotuner cache lookup: the tuned configuration for a volume of this SubDAG height and a batch of
// about n rays (or of the nearest tuned height and batch size, each within 2), or null.
const cqx_launch_cfg* tuned_cfg(const cqx_ctx* ctx, int height, uint64_t n);

// Device scratch a launch uses instead of the context's buffers: the persistent kernels' work
// counters (1 KiB) and the ray-binning buffers (bins_bytes long).
struct ScratchView {
    void* counters = nullptr;
    void* bins = nullptr;
    size_t bins_bytes = 0;
};

// Grows the context's staging buffer (host-buffer entry points) to at least `bytes`.
cqx_status ensure_scratch(cqx_ctx* ctx, size_t bytes);
// Brings the packed copy up to date after nodes [first, node_count), the SubDAGs or the buffers
// changed, waiting for what it packs (a copy that could not be had before may be packed whole, whatever
// `first` says, and launches on any stream read it), and drops the path tracer's plan if it is this
// volume's and its graph no longer fits. A copy that cannot be allocated is left out. Words hold their
// children's masks: where the change reaches into the upload, whose nodes may have changed ones as
// children, all are made anew, and a store cut short of its upload, or of the root that an undo went back
// to, is walked raw.
cqx_status refresh_packed(cqx_ctx* ctx, cqx_dvolume* vol, uint64_t first);

// Rays per wave of a one-ray-per-lane launch of n rays (at most 64).
uint32_t lanes_per_wave(uint64_t n);

// Ids per wave of a launch of at most n secondary rays whose count is on the device (launch_intersect's
// `dealt`).
uint32_t dealt_ids(uint64_t n);

// Whether the caller left every field open that shapes a launch (cfg null or those fields zero).
bool launch_open(const cqx_launch_cfg* cfg);

// Launches the traversal of `n` rays (or of *n_dev rays, at most n, when n_dev is not null).
// Counters and binning buffers are the context's, or `sv`'s when it is given (then nothing is
// allocated). `dealt` != 0, on a packed volume: that many ids per wave, dealt at launch (up to 64: one
// ray per lane), whatever cfg says of the shape.
cqx_status launch_intersect(cqx_ctx* ctx, const cqx_dvolume* vol, const cqx_ray* rays, uint64_t n,
                            const uint32_t* n_dev, uint32_t flags, float max_footprint, cqx_hit* hits,
                            const cqx_launch_cfg* cfg, hipStream_t stream, const ScratchView* sv = nullptr,
                            uint32_t dealt = 0);

// Threads per block of the kernels that compact lists with block_slots.
constexpr uint32_t kCompactBlock = 1024;

// Stream compaction of N entries per thread into one list: a thread with take[l] set gets slot[l], its
// entry's index in the list. A block's slots are claimed with one atomicAdd on *count, and hold its
// entries l by l, each in thread order. One atomic per wave on a counter that every block uses
// serialises at the memory side (13 ns each on one counter), which made it the largest cost of a shading
// pass over millions of rays; per block it is 16 times rarer. (A claim per l instead made 36 of the 39 us
// of the reference shading's first pass over 900 blocks.) Entries keep no order across blocks. Call once
// per kernel, from every thread of a kBlock-thread block (it synchronises the block).
template <uint32_t kBlock, int N>
__device__ __forceinline__ void block_slots(const bool (&take)[N], uint32_t* count, uint32_t (&slot)[N])
{
    static_assert(kBlock % 64 == 0 && N * (kBlock / 64) <= 64, "whole waves, a lane of one wave per (l, wave)");
    constexpr uint32_t kWaves = kBlock / 64;
    __shared__ uint32_t part[N * kWaves]; // counts by l and wave, then their first slots
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint64_t mask[N];
#pragma unroll
    for (int l = 0; l < N; l++) {
        mask[l] = __ballot(take[l]);
        if (lane == 0) part[l * kWaves + wave] = uint32_t(__popcll(mask[l]));
    }
    __syncthreads();
    if (wave == 0) {
        const uint32_t own = lane < N * kWaves ? part[lane] : 0u;
        uint32_t sum = own;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t v = __shfl_up(sum, off);
            sum += int(lane) >= off ? v : 0u;
        }
        const uint32_t all = __shfl(sum, 63);
        uint32_t base = 0;
        if (lane == 0 && all) base = atomicAdd(count, all);
        base = __shfl(base, 0);
        if (lane < N * kWaves) part[lane] = base + sum - own;
    }
    __syncthreads();
    const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
    for (int l = 0; l < N; l++) slot[l] = part[l * kWaves + wave] + uint32_t(__popcll(mask[l] & below));
}

} // namespace cqx
