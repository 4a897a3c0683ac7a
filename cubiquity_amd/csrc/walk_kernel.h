// The kernel of the packed walk (walk_packed.h), over the rays of a Source:
//   kUniform          one volume: the parameters are the kernel's, the same for every lane
//   P, fetch          a ray id's ray and where its record goes (and, per lane, its volume)
//   Out, record       the record's type, and writing it from a finished ray's state
//   deal              the ids of wave w in a dealt launch
#pragma once

#include "device_internal.h"

namespace {

using namespace cqxd;

constexpr int kQueues = 8;
constexpr int kCounterStride = 16; // queue counters 128 bytes apart: one cache line each
constexpr int kFlagWord = 8;       // the sampled flag of gated launches, in the first counter's line
static_assert(kFlagWord < kCounterStride && kFlagWord % kCounterStride != 0, "a word no counter uses");

// Records are written once: streaming (non-temporal) stores keep them from displacing node lines in L2.
__device__ __forceinline__ void store_record(cqx_hit* dst, const cqx_hit& h)
{
    const uint32_t* s = reinterpret_cast<const uint32_t*>(&h);
    uint32_t* d = reinterpret_cast<uint32_t*>(dst);
#pragma unroll
    for (int i = 0; i < 8; i++) __builtin_nontemporal_store(s[i], d + i);
}

// A source whose ids are [0, n), with cqx_hit records.
struct OneRange {
    using Out = cqx_hit;
    __device__ __forceinline__ void deal(uint64_t w, uint32_t chunk, uint64_t n, uint64_t& next, uint64_t& end) const
    {
        const uint64_t at = w * chunk;
        next = at < n ? at : n;
        end = at + chunk < n ? at + chunk : n;
    }
    __device__ __forceinline__ void record(const PackedParams& P, const PackedRay& S, cqx_hit* dst) const
    {
        cqx_hit out;
        emit_packed(P, S, out);
        store_record(dst, out);
    }
};

template <typename Source>
__device__ __forceinline__ const PackedParams& uniform_params(const Source& s, const PackedParams& lane)
{
    if constexpr (Source::kUniform) return s.P;
    else return lane;
}

__device__ __forceinline__ void setup_packed(PackedRay& S, const float* r)
{
    float v[6];
#pragma unroll
    for (int i = 0; i < 6; i++) v[i] = __builtin_nontemporal_load(r + i);
    ray_setup_packed(S, v[0], v[1], v[2], v[3], v[4], v[5]);
}

// The lane's stack_base(): its wave's `rows` rows of the workgroup's LDS, its own word of each.
__device__ __forceinline__ uint32_t lane_stack(char* rows_lds, uint32_t rows, uint32_t top)
{
    // the low 32 bits of a generic LDS address are the LDS address
    const uint32_t lds = uint32_t(reinterpret_cast<uintptr_t>(rows_lds));
    uint32_t base = stack_base(lds + (threadIdx.x >> 6) * rows * kRowBytes + (threadIdx.x & 63u) * 4u, top);
    opaque(base); // one register, not its terms added at each use
    return base;
}

// Up to `steps` steps of the wave's walking lanes: the plain rays' step when every walking lane may
// take it (its ray plain, its iterations far enough from the cap), the general one otherwise.
template <bool kLod>
__device__ __forceinline__ void walk_burst(const PackedParams& P, PackedRay& S, char* lds, uint32_t base, uint32_t steps)
{
    const bool walking = S.phase == kWalk;
    const uint32_t room = P.max_iters >= 2u * steps ? P.max_iters - 2u * steps : 0u;
    const bool odd = walking && (!S.plain || S.iters > room || P.max_iters < 2u * steps);
    if (__ballot(odd)) {
        for (uint32_t k = 0; k < steps; k++)
            if (S.phase == kWalk) walk_step_packed_any(P, S, lds, base);
    } else {
        for (uint32_t k = 0; k < steps; k++)
            if (__builtin_amdgcn_inverse_ballot_w64(__builtin_amdgcn_ballot_w64(S.phase == kWalk)))
                walk_step_packed<kLod>(P, S, lds, base);
    }
}

__device__ __forceinline__ uint64_t uniform64(uint64_t v)
{
    return uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(v)))) |
           uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(v >> 32)))) << 32;
}

// What a wave does is the same in all forms; they differ in where its ray ids come from.
//   kDealt          wave w owns `chunk` ids or fewer (Source::deal): no counters, no claims, the
//                   hardware's dispatcher balances the load. With chunk <= 64 and refill 64 it is one
//                   ray per lane.
//   kClaimed        persistent waves claim `chunk` ids at a time from the queues' counters
//   kSampled        dealt, one ray per lane, where the sampled flag at `gate` is set (k_sample_rays), and
//                   otherwise claimed by the first `want` workgroups; the rest end at once, in the slots
//                   that those leave free (as a launch of its own they took 17 us of 1.87 ms at 2^24 rays)
// With `gate`, a kDealt launch runs only when the flag equals `want`.
// At 64 VGPRs 8 waves fit a SIMD; the batched form's per-lane parameters take 72 and 7 waves (1.2 M rays of
// 24 volumes 185 us with 6 waves, 183 with 7, 191 with 8 and registers spilled; 15 M of 64 1232, 1176, 1267).
enum WalkForm { kClaimed, kDealt, kSampled };

template <typename Source, bool kLod, WalkForm kForm>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(Source::kUniform ? 8 : 7)))
k_walk(Source src, uint64_t n, const uint32_t* __restrict__ n_dev, unsigned long long* __restrict__ counters,
       uint32_t regroup, uint32_t refill, uint32_t rows, uint32_t chunk, const unsigned long long* __restrict__ gate,
       uint32_t want)
{
    extern __shared__ char lds_rows[];
    bool dealt = kForm == kDealt;
    if constexpr (kForm == kSampled) {
        dealt = *gate != 0;
        if (dealt) refill = chunk = 64u;
        else if (blockIdx.x >= want) return;
    } else if constexpr (kForm == kDealt) {
        if (gate && *gate != want) return;
    }
    if (n_dev) {
        const uint64_t nd = *n_dev;
        n = nd < n ? nd : n;
    }
    PackedParams P;
    typename Source::Out* dst = nullptr;
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t base;
    if constexpr (Source::kUniform) base = lane_stack(lds_rows, rows, src.P.top);
    else base = lane_stack(lds_rows, rows, src.top);

    PackedRay S;
    S.phase = kIdle;
    __shared__ cqx_subdag lds_sub[8];
    const cqx_subdag* tab = lds_sub;
    uint32_t occ = 0u; // occupied octants of the launch's (a lane's) volume
    if constexpr (Source::kUniform) {
        occ = src.P.sub[0].pad1;
        if (threadIdx.x < 8) lds_sub[threadIdx.x] = src.P.sub[threadIdx.x];
        __syncthreads();
    }
    const uint64_t per_q = (n + kQueues - 1) / kQueues;
    uint32_t qc = blockIdx.x % kQueues; // current queue
    uint32_t drained = 0;               // queues found empty so far
    uint64_t c_next = 0, c_end = 0;     // ray ids claimed by this wave
    if (kForm != kClaimed && dealt) {
        const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
        src.deal(uint64_t(blockIdx.x) * (blockDim.x >> 6) + wave, chunk, n, c_next, c_end);
        drained = kQueues;
    }

    for (;;) {
        // A service pass runs once `refill` lanes wait, or none walks: misses of lanes that left their
        // last SubDAG, records of the finished lanes, new rays for the idle ones, then the next SubDAG
        // of every lane between SubDAGs (one copy of that code, for new and continuing rays; a ray
        // that turns out to miss there has its record written by the next pass).
        const uint64_t walking = __ballot(S.phase == kWalk);
        const uint32_t nwait = 64u - uint32_t(__popcll(walking));
        if (nwait >= refill || walking == 0) {
            resolve_leave(S, occ);
            if (is_finished(S.phase)) {
                src.record(uniform_params(src, P), S, dst);
                S.phase = kIdle;
            }
            while (c_next == c_end && drained < kQueues) {
                const uint64_t q_begin = per_q * qc;
                const uint64_t q_end = q_begin + per_q < n ? q_begin + per_q : n;
                const uint64_t q_len = q_end > q_begin ? q_end - q_begin : 0;
                unsigned long long claim = 0;
                if (lane == 0) claim = atomicAdd(&counters[qc * kCounterStride], (unsigned long long)chunk);
                claim = uniform64(claim);
                if (claim < q_len) {
                    c_next = q_begin + claim;
                    c_end = q_begin + (claim + chunk < q_len ? claim + chunk : q_len);
                } else {
                    qc = (qc + 1) % kQueues;
                    drained++;
                }
            }
            const uint64_t idle = __ballot(S.phase == kIdle);
            if (S.phase == kIdle) {
                const uint32_t rank = __builtin_amdgcn_mbcnt_hi(uint32_t(idle >> 32),
                                                                __builtin_amdgcn_mbcnt_lo(uint32_t(idle), 0u));
                const uint64_t k = c_next + rank;
                if (k < c_end) {
                    const float* r;
                    src.fetch(k, P, r, dst);
                    setup_packed(S, r);
                    if constexpr (!Source::kUniform) {
                        tab = P.sub;
                        occ = P.sub[0].pad1;
                    }
                }
            }
            const uint64_t nidle = uint64_t(__popcll(idle));
            c_next = c_next + nidle < c_end ? c_next + nidle : c_end;
            if (drained == kQueues && c_next == c_end && __ballot(S.phase != kIdle) == 0) break;
            enter_octants_packed(tab, uniform_params(src, P), S, lds_rows, base, occ);
        }
        walk_burst<kLod>(uniform_params(src, P), S, lds_rows, base, regroup);
    }
}

// The packed walk's parameters over an eligible volume; `lod`: whether the footprint test can end a walk
// before the leaves.
inline PackedParams packed_params(const cqx_dvolume* vol, uint32_t surf, uint32_t max_iters, float max_footprint, bool& lod)
{
    PackedParams P{};
    P.packed = vol->packed;
    P.sub = vol->sub;
    P.surf = surf;
    P.max_iters = max_iters;
    P.top = uint32_t(vol->max_height);
    P.fp_disabled = footprint_is_disabled(max_footprint) ? 1u : 0u;
    P.max_footprint = max_footprint;
    lod_thresholds(max_footprint, P.lod_hi, P.lod_lo);
    lod = !std::isinf(P.lod_hi);
    return P;
}

} // namespace
