// The ESVO walk over the packed copy of a node store: the traversal every launch on an eligible
// volume runs (see packed_eligible), with the records of traverse_core.h bit for bit.
//
// What it is built around, measured on gfx950 (one instruction type in a loop, 8 waves per SIMD,
// cycles per wave instruction per SIMD):
//   * 2 cycles: v_add/sub/mul/fma_f32, v_mov, v_add/sub_u32, v_and/or/xor/not, right shifts, with
//     VGPR, inline-constant or literal operands;
//   * 4 cycles: compares, v_cndmask, min/max, int <-> float conversions, left shifts, bit-field and
//     other three-operand integer forms, and the 2-cycle ones with an SGPR operand.
// The walk is bound by these issue cycles (the step of traverse_core.h costs about 415 of them with
// its three paths live, 42 steps per ray on the 1024^3 benchmark), then by the L2's rate for
// scattered child reads (256 G reads/s for lines that hit L2). Hence:
//   * Packed words. Each child word of the copy holds the child's index << 8 | its occupancy mask
//     (bit c: its child c is not empty). The walk knows from the node's own word which children are
//     empty and reads memory for occupied ones only: 23 reads per ray instead of 43.
//   * One step = one advance over an empty child (with its pop), where the lane stands on one, then
//     the read of an occupied child and the descent into it: 28 steps per ray instead of 42.
//   * Positions are floats holding kBias + integer: exact for |p| <= 2^22, so plane positions need
//     float additions only, and the bits below the bias are those of the integer for the pop's
//     exclusive or and masks.
//   * Per-axis choices are sign masks (a float difference's sign bit shifted over the word) instead
//     of compare + select, and min/max of three values one instruction.
// Measured against the raw-store walk (MI355X, default launches): 1024^3, 2^24 incoherent rays 3.13 ->
// 1.85 ms; 4096^3, 4.0 M rays without surface properties 2.02 -> 0.98 ms; 1280x720 primary rays at
// 1024^3 with LOD 0.30 -> 0.084 ms; 1021 incoherent rays at 512^3 0.116 -> 0.041 ms; reads from L2 5.8e8 ->
// 2.7e8 per 2^24-ray launch.
// A step's instructions matter twice: as issue cycles where waves fill the chip, and, where they do not
// (small batches, the long rays a launch ends with), as the length of one wave's chain: about 170
// instructions and a read's latency a step. So the child's entry planes are computed while its word is
// in flight, a walk that left stands on node 0 instead of taking a branch of its own, and phases and the
// stack base stay in registers the compiler cannot remake in every branch: 144 -> 113 VALU instructions
// and 60 -> 37 scalar ones. By that alone, 1280x720 camera rays with LOD at 1024^3 99 -> 80 us, 65536 camera rays 37.5 ->
// 30 us, 1021 incoherent rays 51 -> 37 us, 2^24 2.07 -> 1.93 ms. (Reading the next word already at the end
// of a step, with its waits where they belong, took 12 to 20 more instructions and 4 to 12 % longer.)
// The sign masks and one-instruction minima need values without NaN, -0 and underflow: ray_plain() is true for rays where
// none can occur. A wave with another ray among its walking lanes takes walk_step_packed_any, which
// keeps the compare-selects of the reference.
#pragma once

#include "traverse_core.h"

#include <cmath>
#include <cstring>

namespace cqxd {

constexpr float kBias = 12582912.0f;         // 1.5 * 2^23
constexpr uint32_t kBiasBits = 0x4b400000u;  // its bits: as_uint(kBias + p) = kBiasBits + p
constexpr int32_t kPackedExtent = 1 << 22;   // SubDAG corners lie in [-2^22, 2^22]
constexpr uint32_t kPackedNodes = 1u << 24;  // node indices of a packed store
constexpr uint32_t kRowBytes = 64u * 4u;     // one stack row: a word per lane of the wave

struct PackedParams {
    const uint32_t* __restrict__ packed; // node_count x 8 packed words
    const cqx_subdag* __restrict__ sub;  // 8 SubDAGs: pad0 the node's packed word, pad1 the mask of the occupied ones
    uint32_t surf;
    uint32_t max_iters;
    uint32_t top;     // largest SubDAG height of the launch: the row of height h is top - h
    float lod_hi;     // child of size s and exit time t large: 0 <= t <= lod_hi * s or t <= lod_lo * s < 0
    float lod_lo;
    uint32_t fp_disabled;
    float max_footprint;
};

// Word for a child with index `index` whose occupancy mask is `mask` (0 for an empty child).
__host__ __device__ inline uint32_t packed_word(uint32_t index, uint32_t mask) { return index ? (index << 8) | mask : 0u; }

// The packed word of a child: its index and the occupancy mask of its node. Nodes that no root reaches are
// packed too, and their words are unchecked: one past the store's `node_count` nodes is packed as empty.
__device__ __forceinline__ uint32_t pack_child(const uint32_t* __restrict__ nodes, uint64_t node_count, uint32_t child)
{
    if (child == 0 || child >= node_count) return 0u;
    const uint4* q = reinterpret_cast<const uint4*>(nodes) + uint64_t(child) * 2;
    const uint4 a = q[0], b = q[1];
    const uint32_t mask = (a.x ? 1u : 0u) | (a.y ? 2u : 0u) | (a.z ? 4u : 0u) | (a.w ? 8u : 0u) | (b.x ? 16u : 0u) |
                          (b.y ? 32u : 0u) | (b.z ? 64u : 0u) | (b.w ? 128u : 0u);
    return packed_word(child, mask);
}

// The footprint test size / t > F (one correctly rounded division; size a power of two) as thresholds
// on t / size, which is exact: with u = t / size, RN(1 / u) > F holds for 0 <= u <= hi and for
// u <= lo < 0 (RN(1 / u) is monotonic on either side of 0). hi = infinity: for every u >= 0.
inline void lod_thresholds(float F, float& hi, float& lo)
{
    hi = -1.0f;
    lo = -INFINITY;
    const auto value = [](uint32_t b) { float f; std::memcpy(&f, &b, 4); return f; };
    if (F < 0.0f) { // u > 0: always; u < 0: |u| at least the smallest magnitude b with RN(-1 / |u|) > F
        hi = INFINITY;
        uint32_t a = 0u, b = 0x7f800000u;
        while (b - a > 1) {
            const uint32_t m = a + (b - a) / 2;
            (-1.0f / value(m) > F ? b : a) = m;
        }
        lo = -value(b);
    } else if (F < INFINITY) { // 0 <= u <= the largest magnitude a with RN(1 / u) > F
        uint32_t a = 0u, b = 0x7f800000u;
        while (b - a > 1) {
            const uint32_t m = a + (b - a) / 2;
            (1.0f / value(m) > F ? a : b) = m;
        }
        hi = value(a);
    }
}

// Whether a store with these SubDAGs can be walked packed: node indices below 2^24, positions whose
// biased floats are exact, and heights as the walk's child sizes state them.
inline bool packed_eligible(uint64_t node_count, const cqx_subdag (&sub)[8])
{
    if (node_count > kPackedNodes) return false;
    for (const cqx_subdag& s : sub) {
        if (s.node == 0) continue;
        if (s.height < 0 || s.height > 22 || (s.height == 0 && s.node >= kMaterialCount)) return false;
        for (int a = 0; a < 3; a++)
            if (s.lower[a] < -kPackedExtent || int64_t(s.lower[a]) + (int64_t(1) << s.height) > kPackedExtent) return false;
    }
    return true;
}

// A state of the walk (RayState of traverse_core.h, in the packed walk's terms).
struct PackedRay {
    float ox, oy, oz; // reflected, shifted origin
    float dx, dy, dz; // |direction|
    float ix, iy, iz; // 1 / |direction|
    uint32_t sign_bits;
    uint32_t oct;
    uint32_t node;    // packed word of the current node
    uint32_t word;    // the hit child's packed word once the phase is kHit
    float bx, by, bz; // lower corner of the current child, plus kBias
    float s;          // its size
    uint32_t cid;
    uint32_t sp;      // byte offset of the stack row of the current node's height
    uint32_t zstart;  // 32 - the SubDAG's height
    float last_exit;
    uint32_t entries, iters;
    uint32_t phase;
    uint32_t plain;   // ray_plain()
};

__device__ __forceinline__ uint32_t fbits(float f)
{
#if defined(__AMDGCN__)
    return __float_as_uint(f);
#else
    uint32_t u;
    std::memcpy(&u, &f, 4);
    return u;
#endif
}
__device__ __forceinline__ float bitsf(uint32_t u)
{
#if defined(__AMDGCN__)
    return __uint_as_float(u);
#else
    float f;
    std::memcpy(&f, &u, 4);
    return f;
#endif
}

// Minimum and maximum of values that are neither NaN nor -0, in one instruction.
__device__ __forceinline__ float plain_min3(float a, float b, float c)
{
#if defined(__AMDGCN__)
    float r;
    asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
#else
    return min3f(a, b, c);
#endif
}
__device__ __forceinline__ float plain_max3(float a, float b, float c)
{
#if defined(__AMDGCN__)
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
#else
    return max3f(a, b, c);
#endif
}
// max(x, smallest denormal)
__device__ __forceinline__ float at_least_denorm(float x)
{
#if defined(__AMDGCN__)
    float r;
    asm("v_max_f32 %0, 1, %1" : "=v"(r) : "v"(x)); // inline constant 1: the bits of 2^-149
    return r;
#else
    return smax(bitsf(1u), x);
#endif
}
// 1 / d correctly rounded for d in [1e-18, 1e18] (a normal result): the hardware's reciprocal (within
// 1 ulp) and two Newton corrections by fused multiply-adds, the last one Markstein's correctly
// rounding step; 24 issue cycles against 38 for the general division's scaling and fix-up. Equal to
// the division for every float of that range (test_plain_reciprocal.py compares all 1.0e9 on the GPU).
__device__ __forceinline__ float plain_rcp(float d)
{
#if defined(__AMDGCN__)
    float r = __builtin_amdgcn_rcpf(d);
    r = __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
    return __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
#else
    return 1.0f / d;
#endif
}
// A value the compiler knows nothing of: kept in its register instead of being made anew (a phase that
// is kWalk, a sum) in every branch.
__device__ __forceinline__ void opaque(uint32_t& v)
{
#if defined(__AMDGCN__)
    asm("" : "+v"(v));
#else
    (void)v;
#endif
}
// Keeps what is computed of a, b and c in the branch it stands in.
__device__ __forceinline__ void stay_here(float& a, float& b, float& c)
{
#if defined(__AMDGCN__)
    asm volatile("" : "+v"(a), "+v"(b), "+v"(c));
#else
    (void)a, (void)b, (void)c;
#endif
}
// Has a, b and c computed here, while a read issued before is in flight, rather than after its wait in
// the branch that uses them (where the compiler moves them).
__device__ __forceinline__ void in_flight(uint32_t& a, uint32_t& b, uint32_t& c)
{
#if defined(__AMDGCN__)
    asm volatile("" : "+v"(a), "+v"(b), "+v"(c));
    __builtin_amdgcn_sched_barrier(0);
#else
    (void)a, (void)b, (void)c;
#endif
}
// All bits set where a < b (0 otherwise), for a, b finite: with denormals a - b is negative exactly then.
__device__ __forceinline__ uint32_t less_mask(float a, float b) { return uint32_t(int32_t(fbits(a - b)) >> 31); }

// Rays whose walk meets no NaN, no -0 and no underflow: for coordinates p with |p| <= 2^22, p - o is
// 0 or at least 2^-25 in magnitude (o = fl(ray origin + 0.5) is a multiple of 2^-25) and at most
// 2^60, and 1/|d| within [2^-60, 2^60], so every (p - o) * (1/|d|) is +0 or a normal number.
__device__ __forceinline__ bool ray_plain(const PackedRay& S)
{
    const float o = (fabsf(S.ox) + fabsf(S.oy)) + fabsf(S.oz); // NaN and infinity stay
    const float d = (S.dx + S.dy) + S.dz;
    return (o <= 5.0e17f) & (d <= 1.0e18f) & (S.dx >= 1.0e-18f) & (S.dy >= 1.0e-18f) & (S.dz >= 1.0e-18f);
}

// The octants a ray crosses, in order (raytracing.cpp:424-434, :469-475).
struct OctantChain {
    float distx, disty, distz;
    uint32_t oct;
    uint32_t phase;
};

__device__ __forceinline__ OctantChain octant_chain(const PackedRay& S)
{
    OctantChain c;
    float ox = S.ox, oy = S.oy, oz = S.oz;
    stay_here(ox, oy, oz); // (three divisions that few lanes need: hoisted out of enter_octants_packed's loop otherwise)
    c.distx = (-ox) / S.dx;
    c.disty = (-oy) / S.dy;
    c.distz = (-oz) / S.dz;
    c.oct = 0;
    if (c.distx < 0.0f) { c.oct += 1; c.distx += kFltMax; }
    if (c.disty < 0.0f) { c.oct += 2; c.disty += kFltMax; }
    if (c.distz < 0.0f) { c.oct += 4; c.distz += kFltMax; }
    c.phase = kOctant;
    return c;
}

// Ray setup, raytracing.cpp:415-434. The octant distances are not kept: only a ray that has to go on
// to another octant needs them (octant_chain). A plain ray's first octant follows from the signs of
// its origin (o > 0 exactly when (-o) / d < 0).
__device__ __forceinline__ void ray_setup_packed(PackedRay& S, float rox, float roy, float roz, float rdx, float rdy,
                                                 float rdz)
{
    const bool sbx = rdx < 0.0f, sby = rdy < 0.0f, sbz = rdz < 0.0f;
    S.sign_bits = (sbx ? 1u : 0u) | (sby ? 2u : 0u) | (sbz ? 4u : 0u);
    S.ox = (rox + 0.5f) * (sbx ? -1.0f : 1.0f);
    S.oy = (roy + 0.5f) * (sby ? -1.0f : 1.0f);
    S.oz = (roz + 0.5f) * (sbz ? -1.0f : 1.0f);
    S.dx = fabsf(rdx);
    S.dy = fabsf(rdy);
    S.dz = fabsf(rdz);
    S.entries = 0;
    S.iters = 0;
    S.phase = kOctant;
    const bool plain = ray_plain(S);
    S.plain = plain ? 1u : 0u;
    if (plain) {
        S.ix = plain_rcp(S.dx);
        S.iy = plain_rcp(S.dy);
        S.iz = plain_rcp(S.dz);
        S.oct = (S.ox > 0.0f ? 1u : 0u) | (S.oy > 0.0f ? 2u : 0u) | (S.oz > 0.0f ? 4u : 0u);
    } else {
        S.ix = 1.0f / S.dx;
        S.iy = 1.0f / S.dy;
        S.iz = 1.0f / S.dz;
        S.oct = octant_chain(S).oct;
    }
}

// The stack word at byte offset `off`: on the GPU an LDS address (lds_address() + the offset in the
// workgroup's rows), so that no base is added on each access; `lds` is the host's buffer.
__device__ __forceinline__ void stack_store(char* lds, uint32_t off, uint32_t v)
{
#if defined(__AMDGCN__)
    *reinterpret_cast<__attribute__((address_space(3))) uint32_t*>(off) = v;
#else
    std::memcpy(lds + off, &v, 4);
#endif
}
__device__ __forceinline__ uint32_t stack_load(const char* lds, uint32_t off)
{
#if defined(__AMDGCN__)
    return *reinterpret_cast<const __attribute__((address_space(3))) uint32_t*>(off);
#else
    uint32_t v;
    std::memcpy(&v, lds + off, 4);
    return v;
#endif
}

// Node 0 in `rows` rows from `off` on: ancestors not pushed yet read as node 0, as in the reference's zeroed
// stack. Four rows at a time (two instructions), the last four overlapping those before.
__device__ __forceinline__ void stack_clear(char* lds, uint32_t off, uint32_t rows)
{
    const auto four = [&](uint32_t at) {
        for (uint32_t k = 0; k < 4; k++) stack_store(lds, at + k * kRowBytes, 0u);
    };
    if (rows < 4u) {
        for (uint32_t k = 0; k < rows; k++) stack_store(lds, off + k * kRowBytes, 0u);
        return;
    }
    for (uint32_t k = 4; k < rows; k += 4, off += 4u * kRowBytes) four(off);
    four(off + (((rows - 1u) & 3u) - 3u) * kRowBytes);
}

// A lane's stack base: row(h) = base + (32 - h) rows, for the column (first row) at `column`.
__device__ __forceinline__ uint32_t stack_base(uint32_t column, uint32_t top) { return column + (top - 32u) * kRowBytes; }

// Whether an occupied octant (occ: bit i for SubDAG i) can follow the ray's current one: a plain ray
// crosses octants by setting bits of `oct`, one after the other, so only supersets of it are ahead.
// Other rays: always true.
__device__ __forceinline__ bool octants_ahead(const PackedRay& S, uint32_t occ)
{
    const uint32_t o = S.oct ^ S.sign_bits;
    uint32_t m = occ & ~(1u << o);
    m &= (S.oct & 1u) ? ((o & 1u) ? 0xaau : 0x55u) : 0xffu;
    m &= (S.oct & 2u) ? ((o & 2u) ? 0xccu : 0x33u) : 0xffu;
    m &= (S.oct & 4u) ? ((o & 4u) ? 0xf0u : 0x0fu) : 0xffu;
    return !S.plain || m != 0;
}

// The slab test of the current octant's SubDAG and the walk's first child (raytracing.cpp:443-458,
// :220-250); the phase becomes kWalk, or kLeave when the ray misses the SubDAG. `base`: the lane's
// stack_base(); `tab`: the 8 SubDAGs with their packed root words (pad0).
__device__ __forceinline__ void octant_enter_packed(const cqx_subdag* tab, const PackedParams& P, PackedRay& S, char* lds,
                                                    uint32_t base)
{
    const cqx_subdag& sd = tab[S.oct ^ S.sign_bits];
    const int32_t height = sd.height;
    const float nsz = bitsf(uint32_t(127 + height) << 23); // 2^height
    // reflected lower corner: lower, or -lower - size
    const float lx = float(sd.lower[0]), ly = float(sd.lower[1]), lz = float(sd.lower[2]);
    const float px = (S.sign_bits & 1u) ? -lx - nsz : lx, py = (S.sign_bits & 2u) ? -ly - nsz : ly,
                pz = (S.sign_bits & 4u) ? -lz - nsz : lz;
    const float entry = max3f((px - S.ox) * S.ix, (py - S.oy) * S.iy, (pz - S.oz) * S.iz);
    const float exitt = min3f(((px + nsz) - S.ox) * S.ix, ((py + nsz) - S.oy) * S.iy, ((pz + nsz) - S.oz) * S.iz);
    S.phase = kLeave;
    if (!(entry < exitt)) return;
    stack_clear(lds, base + (32u - P.top) * kRowBytes, P.top + 1u);
    S.zstart = 32u - uint32_t(height);
    S.sp = base + S.zstart * kRowBytes;
    S.node = sd.pad0;
    const float half = height > 0 ? nsz * 0.5f : 0.0f;
    const float cx = px + half, cy = py + half, cz = pz + half;
    const bool behind = entry <= 0.0f; // findFirstChild, raytracing.cpp:178-196
    const bool bx = ((cx - S.ox) * S.ix < entry) | (behind & (S.ox >= cx));
    const bool by = ((cy - S.oy) * S.iy < entry) | (behind & (S.oy >= cy));
    const bool bz = ((cz - S.oz) * S.iz < entry) | (behind & (S.oz >= cz));
    S.cid = (bx ? 1u : 0u) | (by ? 2u : 0u) | (bz ? 4u : 0u);
    S.bx = kBias + (bx ? cx : px);
    S.by = kBias + (by ? cy : py);
    S.bz = kBias + (bz ? cz : pz);
    S.s = half;
    S.last_exit = exitt;
    S.entries++;
    S.phase = kWalk;
}

// Moves a lane that is between SubDAGs (kOctant: at its current octant; kLeave: past it) into the walk
// of the next SubDAG it enters, or to the end of its walk.
__device__ __forceinline__ void enter_octants_packed(const cqx_subdag* tab, const PackedParams& P, PackedRay& S, char* lds,
                                                     uint32_t base, uint32_t occ)
{
    while (S.phase == kOctant || S.phase == kLeave) {
        if (S.phase == kLeave || !((occ >> (S.oct ^ S.sign_bits)) & 1u)) {
            if (!octants_ahead(S, occ)) {
                S.phase = kMiss;
            } else {
                OctantChain c = octant_chain(S); // replayed up to the current octant: the same steps
                while (c.oct < S.oct && c.phase == kOctant) octant_advance(c);
                do octant_advance(c);
                while (c.phase == kOctant && !((occ >> (c.oct ^ S.sign_bits)) & 1u));
                S.oct = c.oct;
                S.phase = c.phase;
            }
        }
        if (S.phase == kOctant) octant_enter_packed(tab, P, S, lds, base);
    }
}

// What a service pass does first for a lane that left its SubDAG: with no occupied octant ahead its
// walk is a miss, and its record can be written in the same pass.
__device__ __forceinline__ void resolve_leave(PackedRay& S, uint32_t occ)
{
    if (S.phase != kLeave) return;
    // the usual volume has one occupied octant: the one just left
    if ((occ & (occ - 1u)) == 0 ? S.plain != 0 : !octants_ahead(S, occ)) S.phase = kMiss;
}

// The occupied child's word: slot cid ^ signBits of the current node.
__device__ __forceinline__ uint32_t packed_fetch(const PackedParams& P, const PackedRay& S, uint32_t slot)
{
    const uint32_t off = ((S.node >> 3) & ~31u) | (slot << 2); // index * 32 + slot * 4 < 2^29
    return *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(P.packed) + off);
}

// Exit times of the current child (its upper planes), and their minimum.
__device__ __forceinline__ float packed_exits(const PackedRay& S, float& t1x, float& t1y, float& t1z)
{
    t1x = (((S.bx - kBias) + S.s) - S.ox) * S.ix;
    t1y = (((S.by - kBias) + S.s) - S.oy) * S.iy;
    t1z = (((S.bz - kBias) + S.s) - S.oz) * S.iz;
    return plain_min3(t1x, t1y, t1z);
}

__device__ __forceinline__ uint32_t bit_at(uint32_t v, uint32_t m)
{
#if defined(__AMDGCN__)
    return __builtin_amdgcn_ubfe(v, m, 1u);
#else
    return (v >> m) & 1u;
#endif
}

// Pop to the highest boundary crossed (raytracing.cpp:339-364); obx.. the position before the
// advance. A walk that left the SubDAG stands on node 0, which has no children.
__device__ __forceinline__ void packed_pop(PackedRay& S, char* lds, uint32_t base, float obx, float oby, float obz)
{
    const uint32_t ux = fbits(S.bx), uy = fbits(S.by), uz = fbits(S.bz);
    const uint32_t diff = (ux ^ fbits(obx)) | (uy ^ fbits(oby)) | (uz ^ fbits(obz));
    const uint32_t z = uint32_t(__builtin_clz(diff)); // the highest bit is 31 - z; the node's height 32 - z
    const bool left = z < S.zstart;
    S.phase = left ? uint32_t(kLeave) : S.phase;
    opaque(S.phase); // one select
    S.node = 0u;
    if (left) return;
    S.sp = base + z * kRowBytes;
    S.node = stack_load(lds, S.sp);
    const uint32_t keep = uint32_t(int32_t(0x80000000u) >> z); // clears the bits below the boundary's
    const uint32_t m = 31u - z;
    S.cid = bit_at(ux, m) | (bit_at(uy, m) << 1) | (bit_at(uz, m) << 2);
    S.bx = bitsf(ux & keep);
    S.by = bitsf(uy & keep);
    S.bz = bitsf(uz & keep);
    S.s = bitsf((158u - z) << 23); // 2^(31 - z)
    S.last_exit = 0.0f;
    S.entries++;
}

// Whether the current child is occupied.
__device__ __forceinline__ bool on_occupied(const PackedRay& S) { return (S.node >> (S.cid ^ S.sign_bits)) & 1u; }

// The footprint test of a child of size s and exit time tcx by its thresholds: large when 0 <= tcx <=
// lod_hi * s, or tcx <= lod_lo * s (which is negative). Where tcx is not -0, tcx >= 0 or tcx <= -q
// says that the bits of -tcx, as an integer, are at least those of q >= 0: one compare.
template <bool kLod>
__device__ __forceinline__ bool large_at(const PackedParams& P, float tcx, float s)
{
    const bool large = (fbits(tcx) ^ 0x80000000u) >= fbits(-P.lod_lo * s);
    return kLod ? large & (tcx <= P.lod_hi * s) : large;
}

// One step of a plain ray (ray_plain) whose phase is kWalk: an advance if the current child is empty,
// then the descent into (or hit of) the current child if it is occupied. Counts up to two
// iterations; the caller keeps iters + 2 <= max_iters.
template <bool kLod>
__device__ __forceinline__ void walk_step_packed(const PackedParams& P, PackedRay& S, char* lds, uint32_t base)
{
    float t1x, t1y, t1z;
    if (!on_occupied(S)) {
        // Advance to the next sibling, raytracing.cpp:328-332: the axes whose exit is the minimum.
        S.iters++;
        const float tcx = packed_exits(S, t1x, t1y, t1z);
        const uint32_t fx = uint32_t(int32_t(fbits(t1x - tcx) - 1u) >> 31), fy = uint32_t(int32_t(fbits(t1y - tcx) - 1u) >> 31),
                       fz = uint32_t(int32_t(fbits(t1z - tcx) - 1u) >> 31);
        const float obx = S.bx, oby = S.by, obz = S.bz;
        S.bx = obx + bitsf(fbits(S.s) & fx);
        S.by = oby + bitsf(fbits(S.s) & fy);
        S.bz = obz + bitsf(fbits(S.s) & fz);
        const uint32_t flips = (fx & 1u) | (fy & 2u) | (fz & 4u);
        const uint32_t carry = S.cid & flips;
        S.cid ^= flips;
        if (carry) packed_pop(S, lds, base, obx, oby, obz);
    }
    opaque(S.cid); // tested anew: carrying the outcome past the branch takes more instructions
    if (on_occupied(S)) {
        S.word = packed_fetch(P, S, S.cid ^ S.sign_bits); // the last one read is the hit's
        S.iters++;
        const float tcx = packed_exits(S, t1x, t1y, t1z);
        const float half = S.s * 0.5f;
        const float px = S.bx - kBias, py = S.by - kBias, pz = S.bz - kBias;
        // entry time of the child; children behind the origin (entry <= 0) compare their centre
        // planes with "t <= 0", which is t < 2^-149 (findFirstChild, raytracing.cpp:178-196)
        const float tce = at_least_denorm(plain_max3((px - S.ox) * S.ix, (py - S.oy) * S.iy, (pz - S.oz) * S.iz));
        uint32_t mx = less_mask(((px + half) - S.ox) * S.ix, tce);
        uint32_t my = less_mask(((py + half) - S.oy) * S.iy, tce);
        uint32_t mz = less_mask(((pz + half) - S.oz) * S.iz, tce);
        in_flight(mx, my, mz);
        // (s >= 1.5: deeper than a valid DAG otherwise; packed_hit tells these from hits)
        const bool down = large_at<kLod>(P, tcx, S.s) & (S.word >= (kMaterialCount << 8)) & (S.s >= 1.5f);
        S.phase = down ? S.phase : uint32_t(kHit);
        opaque(S.phase);
        if (down) {
            if (tcx < S.last_exit) stack_store(lds, S.sp, S.node);
            S.last_exit = tcx;
            S.sp += kRowBytes;
            S.node = S.word;
            S.s = half;
            S.entries++;
            S.bx += bitsf(fbits(half) & mx);
            S.by += bitsf(fbits(half) & my);
            S.bz += bitsf(fbits(half) & mz);
            S.cid = (mx & 1u) | (my & 2u) | (mz & 4u);
        }
    }
}

// hasLargeFootprint with the reference's division (footprint_large of traverse_core.h).
__device__ __forceinline__ bool packed_footprint_large(const PackedParams& P, float size, float tcx)
{
    if (P.fp_disabled && size > 0.0f) return fbits(tcx) <= 0x7f800000u || tcx < -size;
    return (size / tcx) > P.max_footprint;
}

// One iteration of the walk (walk_step_on of traverse_core.h) of any ray, with the reference's
// compare-selects and its iteration cap.
__device__ __forceinline__ void walk_step_packed_any(const PackedParams& P, PackedRay& S, char* lds, uint32_t base)
{
    if (S.iters >= P.max_iters) {
        S.phase = kAnomaly;
        return;
    }
    S.iters++;
    const float px = S.bx - kBias, py = S.by - kBias, pz = S.bz - kBias;
    const float t1x = ((px + S.s) - S.ox) * S.ix, t1y = ((py + S.s) - S.oy) * S.iy, t1z = ((pz + S.s) - S.oz) * S.iz;
    const float tcx = min3f(t1x, t1y, t1z);
    const uint32_t slot = S.cid ^ S.sign_bits;
    if ((S.node >> slot) & 1u) {
        const uint32_t child = packed_fetch(P, S, slot);
        if (child < (kMaterialCount << 8) || !packed_footprint_large(P, S.s, tcx)) {
            S.word = child;
            S.phase = kHit;
            return;
        }
        if (S.s < 1.5f) {
            S.phase = kAnomaly;
            return;
        }
        const float tce = max3f((px - S.ox) * S.ix, (py - S.oy) * S.iy, (pz - S.oz) * S.iz);
        if (tcx < S.last_exit) stack_store(lds, S.sp, S.node);
        S.last_exit = tcx;
        S.sp += kRowBytes;
        S.node = child;
        const float half = S.s * 0.5f;
        S.s = half;
        S.entries++;
        const float cx = px + half, cy = py + half, cz = pz + half;
        const bool behind = tce <= 0.0f;
        const bool bx = ((cx - S.ox) * S.ix < tce) | (behind & (S.ox >= cx));
        const bool by = ((cy - S.oy) * S.iy < tce) | (behind & (S.oy >= cy));
        const bool bz = ((cz - S.oz) * S.iz < tce) | (behind & (S.oz >= cz));
        S.bx += bx ? half : 0.0f;
        S.by += by ? half : 0.0f;
        S.bz += bz ? half : 0.0f;
        S.cid = (bx ? 1u : 0u) | (by ? 2u : 0u) | (bz ? 4u : 0u);
        return;
    }
    const uint32_t flips = (t1x <= tcx ? 1u : 0u) | (t1y <= tcx ? 2u : 0u) | (t1z <= tcx ? 4u : 0u);
    const float obx = S.bx, oby = S.by, obz = S.bz;
    S.bx = obx + ((flips & 1u) ? S.s : 0.0f);
    S.by = oby + ((flips & 2u) ? S.s : 0.0f);
    S.bz = obz + ((flips & 4u) ? S.s : 0.0f);
    const uint32_t carry = S.cid & flips;
    S.cid ^= flips;
    if (carry) packed_pop(S, lds, base, obx, oby, obz);
}

// First voxel of the hit block entered by a plain ray (entered_voxel of traverse_core.h): floor(o + d t)
// clamped to the block, as floats (exact integers below 2^23).
__device__ __forceinline__ uint32_t entered_voxel_plain(float o, float d, float t, float lo, float hi, bool entry_axis)
{
    const float q = floorf(o + d * t);
#if defined(__AMDGCN__)
    const float c = __builtin_amdgcn_fmed3f(q, lo, hi);
#else
    const float c = smin(smax(q, lo), hi);
#endif
    return fbits((entry_axis ? lo : c) + kBias) - kBiasBits;
}

// The hit of a finished ray (phase kHit): its time and info word (with P.surf the normal and the nearest
// material, which takes the first occupied child from the node's mask: one read per level), and which
// axes it entered by. False (info CQX_HIT_ANOMALY) where the material's descent meets an empty node.
struct PackedHit {
    float t;
    uint32_t info;
    uint32_t entries; // with the material's descent
    bool ex, ey, ez;
};

__device__ __forceinline__ bool packed_hit(const PackedParams& P, const PackedRay& S, PackedHit& h)
{
    const uint32_t slot = S.cid ^ S.sign_bits;
    const float px = S.bx - kBias, py = S.by - kBias, pz = S.bz - kBias;
    const float t0x = (px - S.ox) * S.ix, t0y = (py - S.oy) * S.iy, t0z = (pz - S.oz) * S.iz;
    h.t = max3f(t0x, t0y, t0z);
    h.ex = h.t == t0x;
    h.ey = h.t == t0y;
    h.ez = h.t == t0z;
    h.entries = S.entries;
    if (S.plain && S.word >= (kMaterialCount << 8) && S.s < 1.5f) { // a walk that would go deeper than a valid DAG
        float t1x, t1y, t1z;
        const float tcx = packed_exits(S, t1x, t1y, t1z);
        if (large_at<true>(P, tcx, S.s)) {
            h.info = CQX_HIT_ANOMALY;
            return false;
        }
    }
    const float bsize = S.s > 0.0f ? S.s : 1.0f; // a SubDAG of height 0: the node itself, of side 1
    h.info = 1u | (slot << 1) | (((fbits(bsize) >> 23) - 127u) << 4);
    if (!P.surf) return true;
    uint32_t m = S.word;
    while (m >= (kMaterialCount << 8)) {
        h.entries++;
        const uint32_t mask = m & 0xffu;
        if (mask == 0) {
            h.info = CQX_HIT_ANOMALY;
            return false;
        }
        uint32_t ids = (0x76534210u | 0x88888888u) ^ (S.sign_bits * 0x11111111u);
        while (!((mask >> (ids & 7u)) & 1u)) ids >>= 4;
        m = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(P.packed) +
                                               (((m >> 3) & ~31u) | ((ids & 7u) << 2)));
    }
    // normal = vec3(equal(tEntry, childT0)) * -rayDirSign, raytracing.cpp:317-318: magnitude 1 on
    // the entry axes, and the sign bit of -rayDirSign on every axis (0 * -1 = -0)
    h.info |= (h.ex ? 1u << 9 : 0u) | (h.ey ? 1u << 11 : 0u) | (h.ez ? 1u << 13 : 0u);
    h.info |= (S.sign_bits & 1u) ? 0u : 1u << 10;
    h.info |= (S.sign_bits & 2u) ? 0u : 1u << 12;
    h.info |= (S.sign_bits & 4u) ? 0u : 1u << 14;
    h.info |= (m >> 8) << 16;
    return true;
}

// Record of a finished ray: emit_record of traverse_core.h from the packed walk's state.
__device__ __forceinline__ void emit_packed(const PackedParams& P, const PackedRay& S, cqx_hit& out)
{
    result_miss(out);
    out.entries = S.entries;
    out.iters = S.iters;
    out.info = S.phase == kAnomaly ? CQX_HIT_ANOMALY : 0u;
    if (S.phase != kHit) return;
    PackedHit h;
    const bool found = packed_hit(P, S, h);
    out.entries = h.entries;
    out.info = h.info;
    if (!found) return;
    const float px = S.bx - kBias, py = S.by - kBias, pz = S.bz - kBias;
    const float bsize = S.s > 0.0f ? S.s : 1.0f;
    uint32_t vx, vy, vz;
    if (S.plain) {
        const float ext = bsize - 1.0f;
        vx = entered_voxel_plain(S.ox, S.dx, h.t, px, px + ext, h.ex);
        vy = entered_voxel_plain(S.oy, S.dy, h.t, py, py + ext, h.ey);
        vz = entered_voxel_plain(S.oz, S.dz, h.t, pz, pz + ext, h.ez);
    } else {
        const int32_t size = int32_t(bsize);
        vx = uint32_t(entered_voxel(S.ox, S.dx, h.t, int32_t(px), size, h.ex));
        vy = uint32_t(entered_voxel(S.oy, S.dy, h.t, int32_t(py), size, h.ey));
        vz = uint32_t(entered_voxel(S.oz, S.dz, h.t, int32_t(pz), size, h.ez));
    }
    out.voxel[0] = int32_t(vx ^ (0u - (S.sign_bits & 1u)));
    out.voxel[1] = int32_t(vy ^ (0u - ((S.sign_bits >> 1) & 1u)));
    out.voxel[2] = int32_t(vz ^ (0u - (S.sign_bits >> 2)));
    out.t = h.t;
    out.node = S.node >> 8;
}

} // namespace cqxd
