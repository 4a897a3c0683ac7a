// Path tracer and its path-replay adjoint on the gfx950 traversal.
//
// Shading model (no reference counterpart: the reference's CPU and GLSL tracers use sun + sky
// shadow rays and one bounce, src/application/commands/view/pathtracing_demo.cpp:81-190; the
// conventions kept from them are the hit position o + d t, the bounce-ray origin offset along the
// face normal, pathtracing_demo.cpp:139, and the light-blue background (0.8, 0.8, 1.0), :124):
//   * per path (pixel p, sample s): PCG32 with initstate (seed << 32) + p and stream s;
//   * camera ray through (x + u, y + v) (two draws), pinhole, y down;
//   * at each hit: L += beta * emission[m]; if fewer than `bounces` scatterings so far, sample a
//     cosine-weighted direction about the face normal (two draws), beta *= albedo[m];
//   * a ray that escapes adds beta * sky; a path ends after `bounces` scatterings.
// Lambertian BRDF albedo/pi with cosine-weighted sampling makes the throughput weight albedo.
// sin/cos of 2 pi u use the quadrant reduction + Taylor polynomials below and sqrt is correctly
// rounded, so the same arithmetic on the CPU reproduces every path bit for bit.
//
// Forward, two forms with identical per-path arithmetic:
//   wavefront  camera pass (rays, walk and first vertex in one kernel), then per bounce (walk, shade)
//              over compacted lists of the surviving paths, captured once in a hipGraph per plan and
//              replayed; path counts live on the device. On volumes without a packed copy, or with a
//              launch shaped by the caller: generate -> (intersect, shade) x (bounces + 1)
//   megakernel one lane per path, grid-stride
// Both write per-path radiance; k_pt_resolve sums the samples of a pixel in sample order.
// Adjoint (path replay): runs the wavefront pass again (each path's PCG stream makes it trace the
// same paths), which records one byte per path vertex (its material) and how the path ended; then
// a sweep kernel rebuilds each path's throughputs in the forward's FP32 order and runs backwards,
//   G_K = sky if escaped else 0;  G_j = E_j + A_j G_{j+1};
//   dV/dE_j = beta_j,  dV/dA_j = beta_j G_{j+1},
// scaled by dL/dpixel / spp; partial sums in LDS, reduced over blocks in FP64.
#include "walk_kernel.h"

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstring>
#include <new>

using namespace cqxd;
using cqx::fail;
using cqx::release;

namespace {

constexpr int kMaxVertices = 65; // bounces + 1 <= 65 (at most 64 bounces)
// Path record of the wavefront pass: vmat[j * P + p] is
// the material of path p's vertex j, vstat[p] its vertex count K, plus kEscaped when the path
// ended in the sky. Paths that end by an anomaly or a failed scatter have kEscaped clear.
constexpr uint32_t kEscaped = 0x80u;

struct PtDevParams {
    float eye[3];
    float fwd[3], right[3], up[3];
    float kx, ky, half_w, half_h;
    float sky[3];
    float offset;
    float max_footprint;
    uint32_t width, height, spp, bounces;
    uint32_t pad;
    uint64_t seed;
    float* image;            // the render's output
    float albedo[256 * 3];   // by material id
    float emission[256 * 3]; // by material id
};

// A call's parameters as kernel arguments (at most 4 KiB): all but the material tables, then the
// materials [first, first + kArgMaterials).
constexpr uint32_t kArgMaterials = 128;
constexpr uint32_t kHeadWords = offsetof(PtDevParams, albedo) / 4;
struct PtArgs {
    uint32_t head[kHeadWords];
    uint32_t first;
    float albedo[kArgMaterials * 3];
    float emission[kArgMaterials * 3];
};
static_assert(sizeof(PtArgs) < 4000 && 2 * kArgMaterials == 256, "two launches hold the tables");

// ---- PCG32 (O'Neill 2014) ---------------------------------------------------------------------
struct Pcg {
    uint64_t state, inc;
};

__device__ __forceinline__ uint32_t pcg_next(Pcg& r)
{
    const uint64_t old = r.state;
    r.state = old * 6364136223846793005ULL + r.inc;
    const uint32_t xs = uint32_t(((old >> 18u) ^ old) >> 27u);
    const uint32_t rot = uint32_t(old >> 59u);
    return (xs >> rot) | (xs << ((-rot) & 31));
}

__device__ __forceinline__ Pcg pcg_seed(uint64_t initstate, uint64_t initseq)
{
    Pcg r;
    r.state = 0;
    r.inc = (initseq << 1u) | 1u;
    pcg_next(r);
    r.state += initstate;
    pcg_next(r);
    return r;
}

// A generator's state after `k` steps from (inc + initstate), where pcg_seed's second step starts:
// mul * (inc + initstate) + add * inc with mul = M^k, add = 1 + M + ... + M^(k-1). A path that reaches
// depth d has drawn 2 numbers for its camera ray and 2 per scatter, so its generator at depth d follows
// from its pixel and sample: no state is stored.
struct PcgJump {
    uint64_t mul, add;
};

inline PcgJump pcg_jump(uint32_t depth)
{
    PcgJump j{ 1, 0 };
    for (uint32_t k = 0; k < 1 + 2 + 2 * depth; k++) {
        j.add = j.add * 6364136223846793005ULL + 1u;
        j.mul *= 6364136223846793005ULL;
    }
    return j;
}

// uniform in [0, 1) with 24 random bits (exact conversion and scaling)
__device__ __forceinline__ float pcg_uniform(Pcg& r) { return float(pcg_next(r) >> 8) * (1.0f / 16777216.0f); }

// cos and sin of 2 pi u for u in [0, 1): quadrant q = floor(4u), theta = (4u - q) pi/2 in [0, pi/2),
// Taylor polynomials of degree 11 (sin) and 12 (cos), then the quadrant rotation.
__device__ __forceinline__ void sincos_2pi(float u, float& c, float& s)
{
    const float u4 = u * 4.0f;
    const float q = floorf(u4);
    const float th = (u4 - q) * 1.57079632679489662f;
    const float t2 = th * th;
    const float sp = th * (1.0f + t2 * (-1.66666667e-1f + t2 * (8.33333333e-3f + t2 * (-1.98412698e-4f +
                     t2 * (2.75573192e-6f + t2 * -2.50521084e-8f)))));
    const float cp = 1.0f + t2 * (-0.5f + t2 * (4.16666667e-2f + t2 * (-1.38888889e-3f + t2 * (2.48015873e-5f +
                     t2 * (-2.75573192e-7f + t2 * 2.08767570e-9f)))));
    const int qi = int(q);
    if (qi == 0) { c = cp; s = sp; }
    else if (qi == 1) { c = -sp; s = cp; }
    else if (qi == 2) { c = -cp; s = -sp; }
    else { c = sp; s = -cp; }
}

__device__ __forceinline__ void camera_ray(const PtDevParams& d, uint32_t x, uint32_t y, float jx, float jy,
                                           float* o, float* dir)
{
    const float cx = ((float(x) + jx) - d.half_w) * d.kx;
    const float cy = ((float(y) + jy) - d.half_h) * d.ky;
    float v[3];
    for (int a = 0; a < 3; a++) v[a] = (d.fwd[a] + d.right[a] * cx) - d.up[a] * cy;
    const float len = sqrtf((v[0] * v[0] + v[1] * v[1]) + v[2] * v[2]);
    for (int a = 0; a < 3; a++) {
        o[a] = d.eye[a];
        dir[a] = v[a] / len;
    }
}

// Face normal (components -1, -0, +0, +1) from a hit record's normal code.
__device__ __forceinline__ void decode_normal(uint32_t info, float* n)
{
    for (int a = 0; a < 3; a++) {
        const uint32_t code = (info >> (9 + 2 * a)) & 3u;
        const float mag = (code & 1u) ? 1.0f : 0.0f;
        n[a] = (code & 2u) ? -mag : mag;
    }
}

// Cosine-weighted direction about the face normal n and the next ray's origin
// (pos + n * offset). Orthonormal basis after Duff et al., "Building an Orthonormal Basis,
// Revisited", JCGT 6(1), 2017. Returns false for a degenerate (zero) normal.
__device__ __forceinline__ bool scatter(const PtDevParams& d, Pcg& rng, const float* pos, const float* n, float* o,
                                        float* dir)
{
    const float nl = sqrtf((n[0] * n[0] + n[1] * n[1]) + n[2] * n[2]);
    if (!(nl > 0.0f)) return false;
    const float nx = n[0] / nl, ny = n[1] / nl, nz = n[2] / nl;
    const float u1 = pcg_uniform(rng);
    const float u2 = pcg_uniform(rng);
    const float r = sqrtf(u1);
    float c, s;
    sincos_2pi(u2, c, s);
    const float lx = r * c, ly = r * s, lz = sqrtf(1.0f - u1);
    const float sign = copysignf(1.0f, nz);
    const float a = -1.0f / (sign + nz);
    const float b = nx * ny * a;
    const float t0 = 1.0f + sign * nx * nx * a, t1 = sign * b, t2 = -sign * nx;
    const float u0 = b, uu1 = sign + ny * ny * a, u2b = -ny;
    dir[0] = (t0 * lx + u0 * ly) + nx * lz;
    dir[1] = (t1 * lx + uu1 * ly) + ny * lz;
    dir[2] = (t2 * lx + u2b * ly) + nz * lz;
    for (int k = 0; k < 3; k++) o[k] = pos[k] + n[k] * d.offset;
    return true;
}

__device__ __forceinline__ void path_start(const PtDevParams& d, uint64_t p, Pcg& rng, float* o, float* dir,
                                           uint32_t& pixel)
{
    pixel = uint32_t(p / d.spp);
    const uint32_t s = uint32_t(p % d.spp);
    rng = pcg_seed((d.seed << 32) + uint64_t(pixel), uint64_t(s));
    const float jx = pcg_uniform(rng);
    const float jy = pcg_uniform(rng);
    camera_ray(d, pixel % d.width, pixel / d.width, jx, jy, o, dir);
}

// ---- wavefront kernels -----------------------------------------------------------------------

// The paths still alive at a depth: ray, path index and throughput per entry, in `parts` parts of `pcap`
// slots, part k filled from its start up to count[k]. A kernel that writes a list claims its slots with
// one atomicAdd per wave or block on the part's count. On one counter those claims serialise, at 13 ns
// each: with 1024-thread blocks they alone were the 189 us of the first shading pass over 14.7 M paths.
// Over 64 parts, each with its count on a cache line of its own, they overlap. The camera pass, whose
// waves claim for 64 paths each, has a part per group of paths instead (path_group), so that rays of a
// neighbourhood stay together in the next walk. Only the packed walk can be dealt such lists (PathRays):
// other launches take one part.
//
// Units of a list are dealt in turn to the 8 XCDs (a unit is a workgroup), and the units past a part's
// count are empty, so equal rows of the parts must not fall on equal XCDs: with row u % per for unit u,
// the last of every 16 units empty, frames take 5 % longer (2.1 M paths 512^3 adjoint 675 us, 644 rotated;
// 14.7 M at 1024^3 2249, 2135).
constexpr uint32_t kParts = 64;
constexpr uint32_t kCountStride = 32; // words: 128 bytes
struct PathList {
    cqx_ray* rays;
    uint32_t* paths;
    float* beta; // [3][slots]
    uint32_t* count;
    uint32_t parts, stride; // stride: words from a part's count to the next
    uint64_t pcap, slots;   // slots >= parts * pcap
    // Unit u (of `size` slots) as its part and its first row there. The camera pass's groups one after the
    // other; kParts parts in turn, since consecutive groups of paths went to consecutive parts.
    __device__ __forceinline__ void unit(uint32_t u, uint32_t size, uint32_t& part, uint64_t& row) const
    {
        if (parts > kParts) {
            const uint32_t per = uint32_t((pcap + size - 1) / size);
            part = u / per;
            row = uint64_t((u + part) % per) * size;
        } else {
            part = (u + u / parts) % parts;
            row = uint64_t(u / parts) * size;
        }
    }
    uint32_t units(uint32_t size) const { return uint32_t(parts * ((pcap + size - 1) / size)); }
};

// Paths per part of the camera pass's list. Frame times (us) at groups of 256, 1024, 4096, 8192
// paths: 2.1 M paths 512^3 adjoint 721 / 674 / 646 / 653, 7.4 M at 1024^3 1420 / 1397 / 1392 / 1385, 14.7 M
// at 1024^3 2208 / 2209 / 2138 / 2150.
inline uint32_t path_group(uint64_t P)
{
    uint32_t g = 64;
    while (g < 4096 && uint64_t(g) * kParts < P) g *= 2;
    return g;
}

// The bounce rays of a depth for the packed walk, with records of 8 bytes (time, info): the shading pass
// needs no more. With them, the generators' states recomputed and radiance touched only where a vertex
// adds to it, a bounce moves 88 bytes per ray between its two kernels instead of 152; shading passes of
// the 14.7 M path frame at depths 1 to 4: 115, 70, 62, 35 -> 85, 50, 41, 26 us.
struct PathRays {
    static constexpr bool kUniform = true;
    using Out = uint64_t;
    PackedParams P;
    PathList list;
    uint64_t* __restrict__ hits;
    __device__ __forceinline__ void fetch(uint64_t id, PackedParams&, const float*& ray, Out*& out) const
    {
        ray = reinterpret_cast<const float*>(list.rays + id);
        out = hits + id;
    }
    __device__ __forceinline__ void deal(uint64_t w, uint32_t chunk, uint64_t, uint64_t& next, uint64_t& end) const
    {
        uint32_t part;
        uint64_t at;
        list.unit(uint32_t(w), chunk, part, at);
        const uint64_t count = list.count[uint64_t(part) * list.stride];
        const uint64_t first = part * list.pcap;
        next = first + (at < count ? at : count);
        end = first + (at + chunk < count ? at + chunk : count);
    }
    __device__ __forceinline__ void record(const PackedParams& T, const PackedRay& S, Out* dst) const
    {
        PackedHit h;
        h.t = 0.0f;
        h.info = S.phase == kAnomaly ? CQX_HIT_ANOMALY : 0u;
        if (S.phase == kHit) (void)packed_hit(T, S, h);
        __builtin_nontemporal_store(uint64_t(fbits(h.t)) | uint64_t(h.info) << 32, dst);
    }
};

// Starts a call: its parameters to the device and the path counts cleared, one launch for a copy from
// host memory and a clear (a kernel each).
__global__ void __launch_bounds__(256) k_pt_begin(PtArgs args, PtDevParams* __restrict__ dp, uint32_t* __restrict__ counts,
                                                  uint32_t n)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < kHeadWords) reinterpret_cast<uint32_t*>(dp)[i] = args.head[i];
    if (i < kArgMaterials * 3) {
        dp->albedo[args.first * 3 + i] = args.albedo[i];
        dp->emission[args.first * 3 + i] = args.emission[i];
    }
    for (uint32_t k = i; k < n; k += gridDim.x * 256) counts[k] = 0u;
}

// Camera rays of all paths. The paths' throughput (1) and radiance (0) are not stored: the shading pass
// at depth 0, which sees every path, starts from those values.
__global__ void k_pt_generate(const PtDevParams* __restrict__ dp, uint64_t P, cqx_ray* __restrict__ rays,
                              uint32_t* __restrict__ count)
{
    const uint64_t p = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (p == 0) *count = uint32_t(P);
    if (p >= P) return;
    const PtDevParams& d = *dp;
    Pcg rng;
    float o[3], dir[3];
    uint32_t pixel;
    path_start(d, p, rng, o, dir, pixel);
    cqx_ray r;
    for (int a = 0; a < 3; a++) {
        r.o[a] = o[a];
        r.d[a] = dir[a];
    }
    rays[p] = r;
}

// A path's vertex at `depth`: its contribution l, whether it goes on, and if so its next ray and its
// throughput b. kRadiance: the render (throughput and radiance). Without it, the adjoint's replay: the
// same paths, recording each vertex's material (vmat) and how the path ended (vstat) only.
template <bool kRadiance>
__device__ __forceinline__ bool shade_vertex(const PtDevParams& d, uint64_t P, uint32_t depth, const PcgJump& jump, uint32_t p,
                                             float t, uint32_t info, const float* o, const float* dir, float* b, float* l,
                                             cqx_ray& next, uint8_t* __restrict__ vmat, uint8_t* __restrict__ vstat)
{
    for (int a = 0; a < 3; a++) l[a] = 0.0f;
    if (info & CQX_HIT_ANOMALY) {
        // traversal gave up on this ray: the path ends without a contribution
        if (!kRadiance) vstat[p] = uint8_t(depth);
        return false;
    }
    if (!(info & CQX_HIT_FLAG)) {
        if (kRadiance)
            for (int a = 0; a < 3; a++) l[a] = b[a] * d.sky[a];
        else vstat[p] = uint8_t(depth | kEscaped);
        return false;
    }
    const uint32_t m = (info >> 16) & 0xffu;
    if (!kRadiance) vmat[depth * P + p] = uint8_t(m);
    if (kRadiance)
        for (int a = 0; a < 3; a++) l[a] = b[a] * d.emission[m * 3 + a];
    bool cont = false;
    if (depth < d.bounces) {
        float pos[3], nrm[3];
        for (int a = 0; a < 3; a++) pos[a] = o[a] + dir[a] * t;
        decode_normal(info, nrm);
        const uint32_t pixel = p / d.spp;
        Pcg rng;
        rng.inc = (uint64_t(p - pixel * d.spp) << 1u) | 1u;
        rng.state = jump.mul * (rng.inc + ((d.seed << 32) + uint64_t(pixel))) + jump.add * rng.inc;
        cont = scatter(d, rng, pos, nrm, next.o, next.d);
        if (kRadiance)
            for (int a = 0; a < 3; a++) b[a] = b[a] * d.albedo[m * 3 + a];
    }
    if (!kRadiance && !cont) vstat[p] = uint8_t(depth + 1);
    return cont;
}

template <bool kRadiance>
__device__ __forceinline__ void store_path(const PathList& list, uint64_t slot, const cqx_ray& next, uint32_t p, const float* b)
{
    list.rays[slot] = next;
    list.paths[slot] = p;
    if (kRadiance)
        for (int a = 0; a < 3; a++) list.beta[a * list.slots + slot] = b[a];
}

// The camera pass on a packed volume: a path's camera ray, its walk (one ray per lane, `ids` per wave)
// and its first vertex, in registers from one to the next: 14.7 M paths at 1024^3 in 582 us, with VALU
// issue the bound as in the other walks. As three kernels (rays written once and read twice, 32-byte
// records, claims on one counter) they took 66 + 573 + 189. A burst of 8, 12, 16 or 24 steps is the same to
// 0.5 %: no lane waits for a service pass here.
template <bool kRadiance, bool kLod>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(8)))
k_pt_camera(const PtDevParams* __restrict__ dp, uint64_t P, PackedParams T, uint32_t rows, uint32_t ids, PcgJump jump,
            PathList next, float* __restrict__ L, uint8_t* __restrict__ vmat, uint8_t* __restrict__ vstat)
{
    extern __shared__ char lds_rows[];
    __shared__ cqx_subdag lds_sub[8];
    __shared__ float keep[3][64]; // the rays' directions, during the walk
    const PtDevParams& d = *dp;
    const uint32_t lane = threadIdx.x;
    const uint32_t base = lane_stack(lds_rows, rows, T.top);
    const uint32_t occ = T.sub[0].pad1;
    if (lane < 8) lds_sub[lane] = T.sub[lane];
    __syncthreads();
    const uint64_t first = uint64_t(blockIdx.x) * ids, p = first + lane;
    const bool valid = lane < ids && p < P;
    PackedRay S;
    S.phase = kIdle;
    if (valid) {
        Pcg rng;
        float o[3], dir[3];
        uint32_t pixel;
        path_start(d, p, rng, o, dir, pixel);
        for (int a = 0; a < 3; a++) keep[a][lane] = dir[a];
        ray_setup_packed(S, o[0], o[1], o[2], dir[0], dir[1], dir[2]);
    }
    do {
        enter_octants_packed(lds_sub, T, S, lds_rows, base, occ);
        while (__ballot(S.phase == kWalk)) walk_burst<kLod>(T, S, lds_rows, base, 12);
        resolve_leave(S, occ);
    } while (__ballot(S.phase == kLeave));
    bool cont = false;
    cqx_ray ray;
    float b[3] = { 1.0f, 1.0f, 1.0f };
    if (valid) {
        PackedHit h;
        h.t = 0.0f;
        h.info = S.phase == kAnomaly ? CQX_HIT_ANOMALY : 0u;
        if (S.phase == kHit) (void)packed_hit(T, S, h);
        float dir[3], l[3];
        for (int a = 0; a < 3; a++) dir[a] = keep[a][lane];
        cont = shade_vertex<kRadiance>(d, P, 0u, jump, uint32_t(p), h.t, h.info, d.eye, dir, b, l, ray, vmat, vstat);
        if (kRadiance)
            for (int a = 0; a < 3; a++) L[a * P + p] = 0.0f + l[a];
    }
    const uint64_t alive = __ballot(cont);
    if (!alive) return;
    const uint32_t part = uint32_t(first / next.pcap);
    uint32_t at = 0;
    if (lane == 0) at = atomicAdd(next.count + uint64_t(part) * next.stride, uint32_t(__popcll(alive)));
    at = uint32_t(__builtin_amdgcn_readfirstlane(at));
    if (cont)
        store_path<kRadiance>(next, part * next.pcap + at + uint32_t(__popcll(alive & ((1ull << lane) - 1ull))), ray,
                              uint32_t(p), b);
}

// Threads of a shading block: claims on one counter need as few as possible, on kParts there is time.
template <typename Hit>
constexpr uint32_t kShadeBlock = sizeof(Hit) == sizeof(cqx_hit) ? cqx::kCompactBlock : 256u;

__device__ __forceinline__ void read_hit(const cqx_hit& h, float& t, uint32_t& info)
{
    t = h.t;
    info = h.info;
}
__device__ __forceinline__ void read_hit(const uint64_t& h, float& t, uint32_t& info)
{
    const uint64_t v = __builtin_nontemporal_load(&h);
    t = bitsf(uint32_t(v));
    info = uint32_t(v >> 32);
}

// The shading pass of a depth: a thread per slot, block b on part b % parts. Radiance is read and written
// only where the vertex adds to it (a sky ray, an emissive material): adding a zero would keep its bits.
template <bool kRadiance, typename Hit>
__global__ void __launch_bounds__(kShadeBlock<Hit>) k_pt_shade(const PtDevParams* __restrict__ dp, uint64_t P, uint32_t depth,
                                                               PcgJump jump, PathList cur, const Hit* __restrict__ hits,
                                                               PathList next, float* __restrict__ L,
                                                               uint8_t* __restrict__ vmat, uint8_t* __restrict__ vstat)
{
    const PtDevParams& d = *dp;
    uint32_t part;
    uint64_t row;
    cur.unit(blockIdx.x, kShadeBlock<Hit>, part, row);
    const uint64_t count = cur.count[uint64_t(part) * cur.stride];
    if (row >= count) return;
    const uint64_t i = part * cur.pcap + row + threadIdx.x;
    bool cont = false;
    uint32_t p = 0;
    cqx_ray ray;
    float b[3] = { 1.0f, 1.0f, 1.0f };
    if (row + threadIdx.x < count) {
        // depth 0 (on one part) holds every path in order, with throughput 1 and radiance 0
        p = depth == 0 ? uint32_t(i) : cur.paths[i];
        float t, l[3];
        uint32_t info;
        read_hit(hits[i], t, info);
        if (kRadiance && depth > 0)
            for (int a = 0; a < 3; a++) b[a] = cur.beta[a * cur.slots + i];
        const cqx_ray r = cur.rays[i];
        cont = shade_vertex<kRadiance>(d, P, depth, jump, p, t, info, r.o, r.d, b, l, ray, vmat, vstat);
        if (kRadiance) {
            if (depth == 0)
                for (int a = 0; a < 3; a++) L[a * P + p] = 0.0f + l[a];
            else if (l[0] != 0.0f || l[1] != 0.0f || l[2] != 0.0f)
                for (int a = 0; a < 3; a++) L[a * P + p] += l[a];
        }
    }
    if (depth >= d.bounces) return; // no path goes on
    const bool take[1] = { cont };
    const uint32_t to = part % next.parts;
    uint32_t slot[1];
    cqx::block_slots<kShadeBlock<Hit>>(take, next.count + to * next.stride, slot);
    if (cont) store_path<kRadiance>(next, to * next.pcap + slot[0], ray, p, b);
}

// Per-pixel mean of the samples, summed in sample order; channel blockIdx.y of 256 pixels per block.
// With `staged`, a block first copies its pixels' samples (contiguous in L) to LDS with coalesced reads,
// then each thread sums its pixel's row there (a word of padding per 32, so that rows of 2^k samples do
// not share banks); otherwise threads read L directly (spp too large for LDS). 1280x720x16: 75 us with
// the three channels in turn and without padding, 33 us so (177 MB at 5.3 TB/s, the rate of a copy).
constexpr uint32_t resolve_words(uint32_t samples) { return samples + (samples >> 5) + 1u; }

__global__ void __launch_bounds__(256) k_pt_resolve(const PtDevParams* __restrict__ dp, uint64_t P,
                                                    const float* __restrict__ L, uint32_t staged)
{
    extern __shared__ float tile[]; // resolve_words(256 * spp) when staged
    const PtDevParams& d = *dp;
    const uint32_t pixels = d.width * d.height, spp = d.spp, a = blockIdx.y;
    const uint32_t q0 = blockIdx.x * 256; // < pixels: the grid covers the pixels once
    const uint32_t q = q0 + threadIdx.x;
    const uint32_t npix = pixels - q0 < 256 ? pixels - q0 : 256;
    const float* const src = L + a * P + uint64_t(q0) * spp;
    float sum = 0.0f;
    if (staged) {
#pragma unroll 8
        for (uint32_t k = threadIdx.x; k < npix * spp; k += 256) tile[k + (k >> 5)] = __builtin_nontemporal_load(src + k);
        __syncthreads();
        if (q < pixels)
            for (uint32_t s = 0, k = threadIdx.x * spp; s < spp; s++, k++) sum += tile[k + (k >> 5)];
    } else if (q < pixels) {
        for (uint32_t s = 0; s < spp; s++) sum += src[uint64_t(threadIdx.x) * spp + s];
    }
    if (q < pixels) d.image[uint64_t(q) * 3 + a] = sum / float(spp);
}

void launch_resolve(const PtDevParams* dparams, uint32_t pixels, uint32_t spp, uint64_t P, const float* L, hipStream_t s)
{
    const bool staged = spp <= 64;
    hipLaunchKernelGGL(k_pt_resolve, dim3((pixels + 255) / 256, 3), dim3(256),
                       staged ? resolve_words(256 * spp) * sizeof(float) : 0, s, dparams, P, L, staged ? 1u : 0u);
}

// ---- megakernel forward ------------------------------------------------------------------------

__global__ void __launch_bounds__(256) k_pt_megakernel(const PtDevParams* __restrict__ dp, TraceParams T, uint64_t P,
                                                       float* __restrict__ L)
{
    extern __shared__ uint32_t lds_stack[];
    const PtDevParams& d = *dp;
    const uint32_t occ = occupied_octants(T.sub);
    const uint64_t stride_all = uint64_t(gridDim.x) * blockDim.x;
    for (uint64_t p = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; p < P; p += stride_all) {
        Pcg rng;
        float o[3], dir[3];
        uint32_t pixel;
        path_start(d, p, rng, o, dir, pixel);
        float b[3] = { 1.0f, 1.0f, 1.0f }, l[3] = { 0.0f, 0.0f, 0.0f };
        for (uint32_t depth = 0;; depth++) {
            cqx_hit h;
            trace_ray(T, o[0], o[1], o[2], dir[0], dir[1], dir[2], lds_stack + threadIdx.x, blockDim.x, h, occ);
            if (h.info & CQX_HIT_ANOMALY) break;
            if (!(h.info & CQX_HIT_FLAG)) {
                for (int a = 0; a < 3; a++) l[a] += b[a] * d.sky[a];
                break;
            }
            const uint32_t m = (h.info >> 16) & 0xffu;
            for (int a = 0; a < 3; a++) l[a] += b[a] * d.emission[m * 3 + a];
            if (depth >= d.bounces) break;
            float pos[3], nrm[3];
            for (int a = 0; a < 3; a++) pos[a] = o[a] + dir[a] * h.t;
            decode_normal(h.info, nrm);
            if (!scatter(d, rng, pos, nrm, o, dir)) break;
            for (int a = 0; a < 3; a++) b[a] = b[a] * d.albedo[m * 3 + a];
        }
        for (int a = 0; a < 3; a++) L[a * P + p] = l[a];
    }
}

// ---- adjoint (path replay) -----------------------------------------------------------------------

// The backward sweep over each path's recorded vertices. The throughputs beta_j are rebuilt as the
// forward pass formed them (beta_0 = 1, beta_{j+1} = beta_j * albedo[m_j], FP32 in that order).
// The sweep takes the vertices in segments of kSegment, last segment first: a segment's betas are
// rebuilt from beta_0 by the same products (so a path of up to 64 bounces needs registers for one
// segment only), then its vertices are swept from last to first.
//
// The gradient sums have a fixed order, so the result is the same bit for bit on every run: each
// wave takes 64 consecutive paths at a time, and no atomics are involved.
constexpr uint32_t kAdjointBlock = 256;
constexpr int kSegment = 4; // vertices per segment: a path of up to 3 bounces is one
constexpr uint32_t kAdjointWaves = kAdjointBlock / 64;
constexpr uint32_t kAccMaterials = 16;

// Up to kAccMaterials materials: each lane adds its paths' contributions, vertex by vertex in order,
// into its own column of sums in LDS (one row per material and component), and after its last path
// the wave sums each row in a fixed order (the tree of a butterfly over the lanes), a row per lane.
// One wave per workgroup, so that as many as the rows leave room for (6 per CU with 16 materials)
// share a CU. The sums lived in 96 registers before, each contribution added to all of them through
// selects, 192 instructions per vertex: 113 us for 2^21 paths of up to 4 vertices and 16 materials,
// 57 us so (and k_pt_reduce 10 us for 5, over four times the rows). The next paths' records are read while the current ones are swept.
struct SweepIn {
    uint32_t stat;
    uint32_t vm[kSegment]; // the first segment's materials; entries past the path's end are not used
    float delta[3];
};

__global__ void __launch_bounds__(64) k_pt_adjoint_lds(const PtDevParams* __restrict__ dp, uint64_t P,
                                                       const uint8_t* __restrict__ vmat,
                                                       const uint8_t* __restrict__ vstat,
                                                       const float* __restrict__ dimage, uint32_t M,
                                                       float* __restrict__ partials)
{
    extern __shared__ float acc[]; // [M * 6 rows: dA rgb, dE rgb per material][64 lanes]
    __shared__ float table[kAccMaterials + 1][6]; // albedo, emission by material; row 0 for ids not listed (zeros)
    const PtDevParams& d = *dp;
    const uint32_t lane = threadIdx.x, rows = M * 6, last = d.bounces;
    for (uint32_t k = lane; k < (M + 1) * 6; k += 64) {
        const uint32_t m = k / 6, c = k % 6;
        table[m][c] = m == 0 ? 0.0f : c < 3 ? d.albedo[m * 3 + c] : d.emission[m * 3 + (c - 3)];
    }
    for (uint32_t r = 0; r < rows; r++) acc[r * 64 + lane] = 0.0f;
    __syncthreads();
    const float inv_spp = 1.0f / float(d.spp);
    const uint64_t stride_all = uint64_t(gridDim.x) * 64;
    const auto load = [&](uint64_t p, SweepIn& in) {
        const bool valid = p < P;
        in.stat = valid ? vstat[p] : 0u;
#pragma unroll
        for (uint32_t i = 0; i < uint32_t(kSegment); i++) in.vm[i] = valid && i <= last ? vmat[uint64_t(i) * P + p] : 0u;
        const uint32_t pixel = valid ? uint32_t(p) / d.spp : 0u; // P < 2^32
#pragma unroll
        for (int a = 0; a < 3; a++) in.delta[a] = valid ? dimage[uint64_t(pixel) * 3 + a] * inv_spp : 0.0f;
    };
    // `base` is the same for the 64 lanes, so every lane runs every iteration
    uint64_t base = uint64_t(blockIdx.x) * 64;
    SweepIn cur;
    load(base + lane, cur);
    for (; base < P; base += stride_all) {
        const uint64_t p = base + lane;
        SweepIn ahead;
        load(p + stride_all, ahead);
        const int K = int(cur.stat & ~kEscaped);
        const bool escaped = (cur.stat & kEscaped) != 0;
        float G[3];
        for (int a = 0; a < 3; a++) G[a] = escaped ? d.sky[a] : 0.0f;
        // the wave's most vertices (a wave-uniform segment count)
        int kw = 0;
        while (__any(K > kw)) kw += kSegment;
        for (int j0 = kw - kSegment; j0 >= 0; j0 -= kSegment) {
            float b[3] = { 1.0f, 1.0f, 1.0f };
            for (int j = 0; j < j0 && j < K; j++) {
                const uint32_t m = vmat[uint64_t(j) * P + p];
                for (int a = 0; a < 3; a++) b[a] = b[a] * d.albedo[m * 3 + a];
            }
            uint32_t vm[kSegment];
            float vb[kSegment][3], va[kSegment][3];
#pragma unroll
            for (int i = 0; i < kSegment; i++) {
                const bool live = j0 + i < K;
                const uint32_t m = !live ? 0u : j0 == 0 ? cur.vm[i] : vmat[uint64_t(j0 + i) * P + p];
                vm[i] = m <= M ? m : 0u;
#pragma unroll
                for (int a = 0; a < 3; a++) {
                    va[i][a] = table[vm[i]][a];
                    vb[i][a] = b[a];
                    b[a] = b[a] * va[i][a];
                }
            }
#pragma unroll
            for (int i = kSegment - 1; i >= 0; i--) {
                if (j0 + i >= K) continue;
                const uint32_t m = vm[i];
                float* const row = acc + (m - 1) * 6 * 64 + lane;
                float c[6];
#pragma unroll
                for (int a = 0; a < 3; a++) {
                    const float w = cur.delta[a] * vb[i][a];
                    c[a] = w * G[a];
                    c[3 + a] = w;
                    G[a] = table[m][3 + a] + va[i][a] * G[a];
                }
                if (m)
#pragma unroll
                    for (int k = 0; k < 6; k++) row[k * 64] += c[k];
            }
        }
        cur = ahead;
    }
    __syncthreads();
    // Row r on lane r & 63: column j ^ lane at step j, so that the 64 lanes read 64 banks; the tree over
    // the columns (j and j ^ 32 first, then ^ 16, ..) is the same for every lane.
    for (uint32_t r = lane; r < rows; r += 64) {
        const float* const v = acc + r * 64;
        float t[6] = { 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f }; // partial sums waiting for their other half, by level
        float sum = 0.0f;
#pragma unroll
        for (uint32_t n = 0; n < 64; n++) {
            uint32_t j = 0; // n with its 6 bits reversed
#pragma unroll
            for (uint32_t k = 0; k < 6; k++) j |= ((n >> k) & 1u) << (5 - k);
            sum = v[j ^ lane];
#pragma unroll
            for (uint32_t k = 0; k < 6; k++) {
                if (!((n >> k) & 1u)) {
                    t[k] = sum;
                    break;
                }
                sum = t[k] + sum;
            }
        }
        partials[uint64_t(blockIdx.x) * rows + r] = sum;
    }
}

// More materials: vertex slot by vertex slot, the wave groups its lanes by material (the first
// remaining lane's material, then the next); a group's six contributions are summed over the wave by a
// fixed butterfly (lanes outside the group add 0) and lane 0 adds the sums to the wave's row of
// per-material totals in LDS; the block adds its waves' rows in wave order.
__global__ void __launch_bounds__(kAdjointBlock) k_pt_adjoint(const PtDevParams* __restrict__ dp, uint64_t P,
                                                              const uint8_t* __restrict__ vmat,
                                                              const uint8_t* __restrict__ vstat,
                                                              const float* __restrict__ dimage, uint32_t M,
                                                              float* __restrict__ partials)
{
    __shared__ float g[kAdjointWaves][256 * 6]; // per wave: [material][dA rgb, dE rgb]
    for (uint32_t k = threadIdx.x; k < kAdjointWaves * 256 * 6; k += blockDim.x) (&g[0][0])[k] = 0.0f;
    __syncthreads();
    const PtDevParams& d = *dp;
    const float inv_spp = 1.0f / float(d.spp);
    const uint32_t lane = threadIdx.x & 63u;
    float* const gw = g[threadIdx.x >> 6];
    const uint64_t stride_all = uint64_t(gridDim.x) * blockDim.x;
    // `base` is the same for the 64 lanes of a wave, so every lane runs every iteration
    for (uint64_t base = uint64_t(blockIdx.x) * blockDim.x + (threadIdx.x & ~63u); base < P; base += stride_all) {
        const uint64_t p = base + lane;
        const bool valid = p < P;
        const uint32_t stat = valid ? vstat[p] : 0u;
        const int K = int(stat & ~kEscaped);
        const bool escaped = (stat & kEscaped) != 0;
        const uint32_t pixel = valid ? uint32_t(p) / d.spp : 0u; // P < 2^32
        float delta[3];
        for (int a = 0; a < 3; a++) delta[a] = valid ? dimage[uint64_t(pixel) * 3 + a] * inv_spp : 0.0f;
        float G[3];
        for (int a = 0; a < 3; a++) G[a] = escaped ? d.sky[a] : 0.0f;
        // the wave's most vertices (a wave-uniform segment count)
        int kw = K;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const int o = __shfl_xor(kw, off);
            kw = o > kw ? o : kw;
        }
        for (int seg = (kw + kSegment - 1) / kSegment - 1; seg >= 0; seg--) {
            const int j0 = seg * kSegment;
            float b[3] = { 1.0f, 1.0f, 1.0f };
            for (int j = 0; j < j0 && j < K; j++) {
                const uint32_t m = vmat[uint64_t(j) * P + p];
                for (int a = 0; a < 3; a++) b[a] = b[a] * d.albedo[m * 3 + a];
            }
            uint32_t vm[kSegment];
            float vb[kSegment][3];
#pragma unroll
            for (int i = 0; i < kSegment; i++) {
                vm[i] = 0u;
                if (j0 + i < K) {
                    const uint32_t m = vmat[uint64_t(j0 + i) * P + p];
                    vm[i] = m;
                    for (int a = 0; a < 3; a++) {
                        vb[i][a] = b[a];
                        b[a] = b[a] * d.albedo[m * 3 + a];
                    }
                }
            }
#pragma unroll
            for (int i = kSegment - 1; i >= 0; i--) {
                const bool live = j0 + i < K;
                const uint32_t m = vm[i];
                float c[6] = { 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f };
                if (live) {
                    for (int a = 0; a < 3; a++) {
                        const float w = delta[a] * vb[i][a];
                        c[a] = w * G[a];
                        c[3 + a] = w;
                        G[a] = d.emission[m * 3 + a] + d.albedo[m * 3 + a] * G[a];
                    }
                }
                uint64_t todo = __ballot(live);
                while (todo) {
                    const uint32_t m0 = uint32_t(__shfl(int(m), __ffsll((unsigned long long)todo) - 1));
                    const bool in = live && m == m0;
                    todo &= ~__ballot(in);
#pragma unroll
                    for (int k = 0; k < 6; k++) {
                        float v = in ? c[k] : 0.0f;
#pragma unroll
                        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
                        if (lane == 0) gw[m0 * 6 + k] += v;
                    }
                }
            }
        }
    }
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < M * 6; k += blockDim.x) { // material ids 1..M
        float sum = 0.0f;
        for (uint32_t w = 0; w < kAdjointWaves; w++) sum += g[w][6 + k];
        partials[uint64_t(blockIdx.x) * M * 6 + k] = sum;
    }
}

// One workgroup per output value ((material - 1) * 6 + component): strided FP64 sums over the
// block partials (kWaves rows each, added in FP32 in order), then a fixed-order tree in LDS
// (deterministic for a given grid).
template <uint32_t kWaves>
__global__ void __launch_bounds__(256) k_pt_reduce(const float* __restrict__ partials, uint32_t blocks, uint32_t M,
                                                   float* __restrict__ d_albedo, float* __restrict__ d_emission)
{
    __shared__ double acc[256];
    const uint32_t k = blockIdx.x;
    double sum = 0.0;
    for (uint32_t b = threadIdx.x; b < blocks; b += blockDim.x) {
        float f = 0.0f;
#pragma unroll
        for (uint32_t w = 0; w < kWaves; w++) f += partials[(uint64_t(b) * kWaves + w) * M * 6 + k];
        sum += double(f);
    }
    acc[threadIdx.x] = sum;
    __syncthreads();
    for (uint32_t w = blockDim.x / 2; w > 0; w /= 2) {
        if (threadIdx.x < w) acc[threadIdx.x] += acc[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const uint32_t m = k / 6, c = k % 6;
        if (c < 3) d_albedo[m * 3 + c] = float(acc[0]);
        else d_emission[m * 3 + (c - 3)] = float(acc[0]);
    }
}

} // namespace

namespace cqx {

struct PtPlan {
    const cqx_dvolume* vol = nullptr;
    uint32_t width = 0, height = 0, spp = 0, bounces = 0;
    float max_footprint = -1.0f;
    cqx_launch_cfg cfg{};  // traversal launch of the bounce rays
    cqx_launch_cfg cfg0{}; // traversal launch of the camera rays (depth 0)
    bool open = false;     // the caller left the launch open
    uint64_t P = 0;
    uint32_t parts = 1; // shape of the path lists
    uint64_t pcap = 0;
    uint32_t groups = 0; // parts of the camera pass's list (packed)
    size_t count_words(uint32_t depth) const { return groups + size_t(depth) * parts * kCountStride; } // counts before depth's
    PtDevParams* dparams = nullptr;
    bool high = true; // dparams' tables past kArgMaterials are not known to be zero
    cqx_ray* rays[2] = { nullptr, nullptr };
    uint32_t* paths[2] = { nullptr, nullptr };
    float* beta[2] = { nullptr, nullptr };
    void* hits = nullptr; // cqx_hit, or 8-byte records on a packed volume
    float* L = nullptr;
    uint32_t* counts = nullptr; // per depth, kCountStride words per part
    uint8_t* vmat = nullptr;  // (bounces + 1) x P vertex materials
    uint8_t* vstat = nullptr; // P path records (vertex count, escaped)
    float* partials = nullptr;
    size_t partial_floats = 0;
    hipGraph_t graph = nullptr;        // the render: radiance, no path record
    hipGraphExec_t exec = nullptr;
    hipGraph_t graph_replay = nullptr; // the adjoint's replay: path record, no radiance
    hipGraphExec_t exec_replay = nullptr;
};

bool plan_holds(const PtPlan* p, const cqx_dvolume* vol) { return p && p->vol == vol; }

void destroy_pt_plan(PtPlan* p)
{
    if (!p) return;
    if (p->exec) (void)hipGraphExecDestroy(p->exec);
    if (p->graph) (void)hipGraphDestroy(p->graph);
    if (p->exec_replay) (void)hipGraphExecDestroy(p->exec_replay);
    if (p->graph_replay) (void)hipGraphDestroy(p->graph_replay);
    release(p->dparams);
    for (int k = 0; k < 2; k++) {
        release(p->rays[k]);
        release(p->paths[k]);
        release(p->beta[k]);
    }
    release(p->hits);
    release(p->L);
    release(p->counts);
    release(p->vmat);
    release(p->vstat);
    release(p->partials);
    delete p;
}

} // namespace cqx

namespace {

using cqx::PtPlan;

cqx_status fill_params(const cqx_pt_params* pp, PtDevParams& d)
{
    std::memset(&d, 0, sizeof(d));
    if (!pp->width || !pp->height || !pp->spp) return fail(CQX_ERR_INVALID_ARG, "image size and spp must be positive");
    if (pp->bounces > 64) return fail(CQX_ERR_LIMIT, "at most 64 bounces");
    if (pp->n_materials > 255) return fail(CQX_ERR_INVALID_ARG, "at most 255 materials");
    if (pp->n_materials && (!pp->albedo || !pp->emission)) return fail(CQX_ERR_INVALID_ARG, "null material table");
    double f[3] = { pp->target[0] - pp->eye[0], pp->target[1] - pp->eye[1], pp->target[2] - pp->eye[2] };
    const double fl = std::sqrt(f[0] * f[0] + f[1] * f[1] + f[2] * f[2]);
    if (!(fl > 0)) return fail(CQX_ERR_INVALID_ARG, "eye equals target");
    for (double& c : f) c /= fl;
    double r[3] = { -f[2], 0.0, f[0] };
    const double rl = std::sqrt(r[0] * r[0] + r[2] * r[2]);
    if (!(rl > 0)) return fail(CQX_ERR_INVALID_ARG, "view direction parallel to +y");
    for (double& c : r) c /= rl;
    const double u[3] = { r[1] * f[2] - r[2] * f[1], r[2] * f[0] - r[0] * f[2], r[0] * f[1] - r[1] * f[0] };
    const double scale = 2.0 * std::tan(pp->fov_y_degrees * 3.14159265358979323846 / 360.0);
    const double aspect = double(pp->width) / double(pp->height);
    for (int a = 0; a < 3; a++) {
        d.eye[a] = float(pp->eye[a]);
        d.fwd[a] = float(f[a]);
        d.right[a] = float(r[a]);
        d.up[a] = float(u[a]);
        d.sky[a] = pp->sky[a];
    }
    d.kx = float(aspect * scale / pp->width);
    d.ky = float(scale / pp->height);
    d.half_w = 0.5f * float(pp->width);
    d.half_h = 0.5f * float(pp->height);
    d.offset = pp->bounce_offset;
    d.max_footprint = pp->max_footprint;
    d.width = pp->width;
    d.height = pp->height;
    d.spp = pp->spp;
    d.bounces = pp->bounces;
    d.seed = pp->seed;
    for (uint32_t m = 1; m <= pp->n_materials; m++)
        for (int a = 0; a < 3; a++) {
            d.albedo[m * 3 + a] = pp->albedo[(m - 1) * 3 + a];
            d.emission[m * 3 + a] = pp->emission[(m - 1) * 3 + a];
        }
    return CQX_OK;
}

template <typename T>
cqx_status alloc(T** p, size_t count)
{
    if (hipMalloc(reinterpret_cast<void**>(p), sizeof(T) * std::max<size_t>(count, 1)) != hipSuccess)
        return fail(CQX_ERR_OOM, "device allocation of %zu bytes failed", sizeof(T) * count);
    return CQX_OK;
}

// Returns the context's plan for this volume and image shape, (re)building it when anything
// differs. The wavefront buffers and graph are added on first use.
cqx_status get_plan(cqx_ctx* ctx, const cqx_dvolume* vol, const cqx_pt_params* pp, const cqx_launch_cfg* cfg,
                    PtPlan** out)
{
    cqx_launch_cfg c{};
    if (cfg) c = *cfg;
    c.bin_bits = 0; // the bounce launches read their ray count on the device: no binning prepass
    // "auto" (variant 0): the camera rays (depth 0, coherent: a pixel's samples are adjacent) one
    // per lane, 64 per workgroup; the bounce rays on persistent waves at 24 per CU (raw stores, and
    // when the caller shaped the launch), or on a packed volume dealt to the waves (dealt_ids).
    // Only the fields the caller left at zero take these values.
    const bool open = cqx::launch_open(cfg);
    cqx_launch_cfg c0 = c;
    if (c.variant == 0) {
        c0.variant = 1;
        if (!c0.block) c0.block = 64;
        if (!c.waves_per_cu) c.waves_per_cu = 24;
    }
    PtPlan* p = ctx->pt_plan;
    if (p && p->vol == vol && p->width == pp->width && p->height == pp->height && p->spp == pp->spp &&
        p->bounces == pp->bounces && p->max_footprint == pp->max_footprint && p->open == open &&
        std::memcmp(&p->cfg, &c, sizeof(c)) == 0) {
        *out = p;
        return CQX_OK;
    }
    HIP_TRY(hipDeviceSynchronize());
    cqx::destroy_pt_plan(p);
    ctx->pt_plan = nullptr;
    p = new (std::nothrow) PtPlan;
    if (!p) return fail(CQX_ERR_OOM, "out of host memory");
    p->vol = vol;
    p->width = pp->width;
    p->height = pp->height;
    p->spp = pp->spp;
    p->bounces = pp->bounces;
    p->max_footprint = pp->max_footprint;
    p->cfg = c;
    p->cfg0 = c0;
    p->P = uint64_t(pp->width) * pp->height * pp->spp;
    p->open = open;
    cqx_status st = alloc(&p->dparams, 1);
    if (st == CQX_OK) st = alloc(&p->L, 3 * p->P);
    if (st != CQX_OK) {
        cqx::destroy_pt_plan(p);
        return st;
    }
    ctx->pt_plan = p;
    *out = p;
    return CQX_OK;
}

// The wavefront graph of the render (replay false, down to the image) or of the adjoint's replay (replay
// true), captured
// once per plan; the buffers they share are allocated with the first. On a packed volume whose launch
// the caller left open: camera pass, then (walk, shade) per bounce over lists in parts. Otherwise
// generate, then (intersect, shade) per depth.
template <bool kRadiance>
cqx_status capture(cqx_ctx* ctx, PtPlan* p, hipStream_t s)
{
    const uint64_t P = p->P;
    const bool packed = p->vol->packed_ok && p->open;
    uint8_t* const vmat = kRadiance ? nullptr : p->vmat;
    uint8_t* const vstat = kRadiance ? nullptr : p->vstat;
    const uint64_t slots = p->parts * p->pcap;
    const uint32_t group = path_group(P), groups = uint32_t((P + group - 1) / group);
    const auto list = [&](uint32_t depth) {
        const int k = int(depth & 1u);
        if (packed && depth == 1) return PathList{ p->rays[k], p->paths[k], p->beta[k], p->counts, groups, 1u, group, slots };
        return PathList{ p->rays[k], p->paths[k], p->beta[k], p->counts + p->count_words(depth), p->parts, kCountStride,
                         p->pcap, slots };
    };
    if (!packed) {
        hipLaunchKernelGGL(k_pt_generate, dim3(uint32_t((P + 255) / 256)), dim3(256), 0, s, p->dparams, P, p->rays[0], p->counts);
        cqx_hit* const hits = static_cast<cqx_hit*>(p->hits);
        constexpr uint32_t block = kShadeBlock<cqx_hit>;
        for (uint32_t depth = 0; depth <= p->bounces; depth++) {
            const cqx_status st =
                cqx::launch_intersect(ctx, p->vol, p->rays[depth & 1u], P, list(depth).count, CQX_SURFACE_PROPERTIES,
                                      p->max_footprint, hits, depth == 0 ? &p->cfg0 : &p->cfg, s);
            if (st != CQX_OK) return st;
            hipLaunchKernelGGL((k_pt_shade<kRadiance, cqx_hit>), dim3(uint32_t((P + block - 1) / block)), dim3(block), 0, s,
                               p->dparams, P, depth, pcg_jump(depth), list(depth), hits, list(depth + 1), p->L, vmat, vstat);
        }
        return CQX_OK;
    }
    bool lod = false;
    const PackedParams T = packed_params(p->vol, 1u, p->cfg.max_iters ? p->cfg.max_iters : cqx::kDefaultMaxIters,
                                         p->max_footprint, lod);
    const uint32_t rows = T.top + 1u, ids = cqx::lanes_per_wave(P);
    const size_t lds = size_t(rows) * kRowBytes;
    const dim3 camera(uint32_t((P + ids - 1) / ids));
    if (lod)
        hipLaunchKernelGGL((k_pt_camera<kRadiance, true>), camera, dim3(64), lds, s, p->dparams, P, T, rows, ids,
                           pcg_jump(0), list(1), p->L, vmat, vstat);
    else
        hipLaunchKernelGGL((k_pt_camera<kRadiance, false>), camera, dim3(64), lds, s, p->dparams, P, T, rows, ids,
                           pcg_jump(0), list(1), p->L, vmat, vstat);
    uint64_t* const hits = static_cast<uint64_t*>(p->hits);
    const uint32_t chunk = cqx::dealt_ids(P);
    constexpr uint32_t block = kShadeBlock<uint64_t>;
    for (uint32_t depth = 1; depth <= p->bounces; depth++) {
        const PathRays src{ T, list(depth), hits };
        const dim3 walk(src.list.units(chunk)), shade(src.list.units(block));
        const uint32_t refill = chunk > 64 ? 16u : 64u;
        if (lod)
            hipLaunchKernelGGL((k_walk<PathRays, true, kDealt>), walk, dim3(64), lds, s, src, P, nullptr, nullptr, 16u, refill,
                               rows, chunk, nullptr, 0u);
        else
            hipLaunchKernelGGL((k_walk<PathRays, false, kDealt>), walk, dim3(64), lds, s, src, P, nullptr, nullptr, 16u, refill,
                               rows, chunk, nullptr, 0u);
        hipLaunchKernelGGL((k_pt_shade<kRadiance, uint64_t>), shade, dim3(block), 0, s, p->dparams, P, depth,
                           pcg_jump(depth), list(depth), hits, list(depth + 1), p->L, vmat, vstat);
    }
    return CQX_OK;
}

cqx_status ensure_wavefront(cqx_ctx* ctx, PtPlan* p, bool replay)
{
    if (replay ? p->exec_replay : p->exec) return CQX_OK;
    cqx_status st = CQX_OK;
    if (!p->hits) {
        const bool packed = p->vol->packed_ok && p->open;
        const uint64_t group = path_group(p->P), groups = (p->P + group - 1) / group;
        p->parts = packed ? uint32_t(std::min<uint64_t>(kParts, groups)) : 1u;
        p->pcap = packed ? (groups + p->parts - 1) / p->parts * group : p->P;
        const uint64_t slots = p->parts * p->pcap;
        for (int k = 0; k < 2 && st == CQX_OK; k++) {
            st = alloc(&p->rays[k], slots);
            if (st == CQX_OK) st = alloc(&p->paths[k], slots);
            if (st == CQX_OK) st = alloc(&p->beta[k], 3 * slots);
        }
        p->groups = packed ? uint32_t(groups) : 0u;
        if (st == CQX_OK) st = alloc(&p->counts, p->count_words(p->bounces + 2));
        if (st == CQX_OK) {
            uint8_t* hits = nullptr;
            st = alloc(&hits, slots * (packed ? sizeof(uint64_t) : sizeof(cqx_hit)));
            p->hits = hits;
        }
        if (st != CQX_OK) { // all or none, so that a later call starts over
            for (int k = 0; k < 2; k++) {
                release(p->rays[k]);
                release(p->paths[k]);
                release(p->beta[k]);
                p->rays[k] = nullptr;
                p->paths[k] = nullptr;
                p->beta[k] = nullptr;
            }
            release(p->counts);
            p->counts = nullptr;
        }
    }
    if (st == CQX_OK && replay && !p->vstat) { // the adjoint's path record
        st = alloc(&p->vmat, (p->bounces + 1) * p->P);
        if (st == CQX_OK) st = alloc(&p->vstat, p->P);
    }
    if (st != CQX_OK) return st;
    hipStream_t s = ctx->capture_stream;
    HIP_TRY(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    const cqx_status cst = replay ? capture<false>(ctx, p, s) : capture<true>(ctx, p, s);
    if (!replay) launch_resolve(p->dparams, p->width * p->height, p->spp, p->P, p->L, s);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(s, &g);
    (replay ? p->graph_replay : p->graph) = g;
    if (cst != CQX_OK) return cst;
    if (e != hipSuccess || !g) return fail(CQX_ERR_HIP, "graph capture failed: %s", hipGetErrorString(e));
    HIP_TRY(hipGraphInstantiate(replay ? &p->exec_replay : &p->exec, g, nullptr, nullptr, 0));
    return CQX_OK;
}

cqx_status check(cqx_ctx* ctx, const cqx_dvolume* vol, const cqx_pt_params* pp)
{
    if (!ctx || !vol || !pp) return fail(CQX_ERR_INVALID_ARG, "null argument");
    HIP_TRY(hipSetDevice(ctx->device));
    const uint64_t P = uint64_t(pp->width) * pp->height * pp->spp;
    if (P == 0) return fail(CQX_ERR_INVALID_ARG, "empty image");
    if (P >= (uint64_t(1) << 32)) return fail(CQX_ERR_LIMIT, "at most 2^32 - 1 paths per call");
    return CQX_OK;
}

// Queues the call's parameters and the clearing of the path counts, ahead of its kernels. Material ids
// past the caller's are black; the upper half of the tables is written where it holds more than that.
void begin(PtPlan* p, const PtDevParams& host, uint32_t n_materials, hipStream_t s)
{
    const uint32_t words = p->counts ? uint32_t(p->count_words(p->bounces + 2)) : 0u;
    const uint32_t blocks = std::max(2u, std::min(64u, words / 256)); // 2: the material table's 384 words
    PtArgs args;
    std::memcpy(args.head, &host, sizeof(args.head));
    const bool high = n_materials >= kArgMaterials;
    const uint32_t halves = high || p->high ? 2 : 1;
    p->high = high;
    for (uint32_t half = 0; half < halves; half++) {
        args.first = half * kArgMaterials;
        std::memcpy(args.albedo, host.albedo + args.first * 3, sizeof(args.albedo));
        std::memcpy(args.emission, host.emission + args.first * 3, sizeof(args.emission));
        hipLaunchKernelGGL(k_pt_begin, dim3(blocks), dim3(256), 0, s, args, p->dparams, p->counts, words);
    }
}

TraceParams trace_params(const cqx_dvolume* vol, const cqx_pt_params* pp, const cqx_launch_cfg* cfg)
{
    TraceParams T;
    T.nodes = vol->nodes;
    T.sub = vol->sub;
    T.surf = 1;
    T.max_footprint = pp->max_footprint;
    T.max_iters = (cfg && cfg->max_iters) ? cfg->max_iters : cqx::kDefaultMaxIters;
    T.fp_disabled = footprint_is_disabled(pp->max_footprint) ? 1u : 0u;
    T.offset32 = vol->node_count <= (uint64_t(1) << 27) ? 1u : 0u;
    return T;
}

} // namespace

extern "C" {

cqx_status cqx_pathtrace(cqx_ctx* ctx, const cqx_dvolume* vol, const cqx_pt_params* pp, uint32_t mode,
                         const cqx_launch_cfg* cfg, float* image, void* stream_ptr)
{
    const cqx::TraceRange range("cqx_pathtrace");
    cqx_status st = check(ctx, vol, pp);
    if (st != CQX_OK) return st;
    if (!image) return fail(CQX_ERR_INVALID_ARG, "null image");
    if (mode > 1) return fail(CQX_ERR_INVALID_ARG, "mode must be 0 (wavefront) or 1 (megakernel)");
    PtDevParams host;
    st = fill_params(pp, host);
    if (st != CQX_OK) return st;
    PtPlan* p = nullptr;
    st = get_plan(ctx, vol, pp, cfg, &p);
    if (st != CQX_OK) return st;
    if (mode == 0) {
        st = ensure_wavefront(ctx, p, false);
        if (st != CQX_OK) return st;
    }
    hipStream_t s = hipStream_t(stream_ptr);
    host.image = image;
    begin(p, host, pp->n_materials, s);
    if (mode == 0) {
        const cqx::TraceRange bounces("wavefront graph: camera rays, then per bounce traversal and shading");
        HIP_TRY(hipGraphLaunch(p->exec, s));
    } else {
        const cqx::TraceRange mega("megakernel: one lane per path");
        const uint32_t block = 256;
        const size_t lds = size_t(vol->max_height + 1) * block * sizeof(uint32_t);
        if (lds > size_t(ctx->lds_per_block)) return fail(CQX_ERR_LIMIT, "stack needs %zu B of LDS", lds);
        const uint32_t waves = (cfg && cfg->waves_per_cu) ? cfg->waves_per_cu : 16u;
        const uint64_t want = (uint64_t(ctx->cu_count) * waves * 64 + block - 1) / block;
        const uint32_t blocks = uint32_t(std::max<uint64_t>(1, std::min<uint64_t>(want, (p->P + block - 1) / block)));
        hipLaunchKernelGGL(k_pt_megakernel, dim3(blocks), dim3(block), lds, s, p->dparams, trace_params(vol, pp, cfg),
                           p->P, p->L);
        launch_resolve(p->dparams, pp->width * pp->height, pp->spp, p->P, p->L, s);
    }
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(s));
    return CQX_OK;
}

cqx_status cqx_pathtrace_adjoint(cqx_ctx* ctx, const cqx_dvolume* vol, const cqx_pt_params* pp,
                                 const cqx_launch_cfg* cfg, const float* d_image, float* d_albedo, float* d_emission,
                                 void* stream_ptr)
{
    const cqx::TraceRange range("cqx_pathtrace_adjoint");
    cqx_status st = check(ctx, vol, pp);
    if (st != CQX_OK) return st;
    if (!d_image || !d_albedo || !d_emission) return fail(CQX_ERR_INVALID_ARG, "null buffer");
    if (pp->bounces + 1 > uint32_t(kMaxVertices))
        return fail(CQX_ERR_LIMIT, "the adjoint supports at most %d bounces", kMaxVertices - 1);
    if (pp->n_materials == 0) return fail(CQX_ERR_INVALID_ARG, "no materials to differentiate");
    PtDevParams host;
    st = fill_params(pp, host);
    if (st != CQX_OK) return st;
    PtPlan* p = nullptr;
    st = get_plan(ctx, vol, pp, cfg, &p);
    if (st == CQX_OK) st = ensure_wavefront(ctx, p, true);
    if (st != CQX_OK) return st;
    const uint32_t block = kAdjointBlock;
    const uint32_t blocks =
        uint32_t(std::max<uint64_t>(1, std::min<uint64_t>(uint64_t(ctx->cu_count) * 8, (p->P + block - 1) / block)));
    const bool in_lds = pp->n_materials <= kAccMaterials;
    const size_t need = size_t(blocks) * (in_lds ? kAdjointWaves : 1u) * pp->n_materials * 6;
    if (need > p->partial_floats) {
        HIP_TRY(hipDeviceSynchronize());
        release(p->partials);
        p->partials = nullptr;
        p->partial_floats = 0;
        st = alloc(&p->partials, need);
        if (st != CQX_OK) return st;
        p->partial_floats = need;
    }
    hipStream_t s = hipStream_t(stream_ptr);
    begin(p, host, pp->n_materials, s);
    // replay the paths (the replay graph records each path's vertices), then sweep them backwards
    {
        const cqx::TraceRange replay("adjoint: path replay (wavefront graph)");
        HIP_TRY(hipGraphLaunch(p->exec_replay, s));
    }
    {
        const cqx::TraceRange sweep("adjoint: backward sweep and reduction");
        if (in_lds) { // a wave per workgroup, with the paths that the 256-thread blocks' waves would take
            hipLaunchKernelGGL(k_pt_adjoint_lds, dim3(blocks * kAdjointWaves), dim3(64),
                               pp->n_materials * 6 * 64 * sizeof(float), s, p->dparams, p->P, p->vmat, p->vstat,
                               d_image, pp->n_materials, p->partials);
            hipLaunchKernelGGL(k_pt_reduce<kAdjointWaves>, dim3(pp->n_materials * 6), dim3(256), 0, s, p->partials,
                               blocks, pp->n_materials, d_albedo, d_emission);
        } else {
            hipLaunchKernelGGL(k_pt_adjoint, dim3(blocks), dim3(block), 0, s, p->dparams, p->P, p->vmat, p->vstat,
                               d_image, pp->n_materials, p->partials);
            hipLaunchKernelGGL(k_pt_reduce<1>, dim3(pp->n_materials * 6), dim3(256), 0, s, p->partials, blocks,
                               pp->n_materials, d_albedo, d_emission);
        }
    }
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(s));
    return CQX_OK;
}

} // extern "C"
