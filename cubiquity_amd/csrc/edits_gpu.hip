// On-device sphere edits: the region-parallel algorithm of cqx_hv_edit_spheres_mt (edits.cpp) run
// on the device copy of a store, giving the same store byte for byte.
//
//   planning (host, plan_edits): the regions of side 2^hs each sphere's bounds touch, with their
//     spheres in order, and the levels above the regions in Morton order;
//   k_edit_regions: one wave per region descends to the region's node and applies its spheres in
//     order with fillBrush's arithmetic (voxelization.cpp:825-915; EditWalk::fill, here with an
//     explicit stack, each node's 8 children tested on the wave's 64 lanes at once and the 512 voxels
//     of a height-3 node in one step), interning changed nodes into the region's own list with its own
//     hash table; a node without listed children is first looked up in the device index over the
//     store. A list that outgrows its slice stops its region, which runs again with a larger one;
//   merge (k_merge_*): the lists laid end to end in region order and merged as merge_regions does:
//     level by level, the lowest list position among equal nodes is kept, the kept ones are
//     appended in list order;
//   k_top_*: the levels above the regions rebuilt bottom-up, each level's changed nodes interned in Morton
//     order (rebuild_levels);
//   k_find_subdags: the new root's SubDAGs (findSubDAG, raytracing.cpp:43-87).
// The index over the store (open addressing on the node hash; among equal nodes the lowest index)
// is built on a volume's first edit and extended with every appended node. Appended nodes only
// point at earlier nodes, and no node that existed before a call changes, so device copies and
// traversal launches of earlier versions stay valid (undo / redo switch roots).
#include "device_internal.h"

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>

using cqx::fail;
using cqx::release;

namespace {

constexpr uint32_t kMat = CQX_MATERIAL_COUNT;
constexpr uint32_t kEmptySlot = 0xffffffffu;
constexpr uint32_t kTopBlock = 1024;

struct DNode {
    uint32_t c[8];
};

__device__ __forceinline__ DNode load_node(const uint32_t* __restrict__ base, uint64_t i)
{
    const uint4* q = reinterpret_cast<const uint4*>(base + i * 8);
    const uint4 a = q[0], b = q[1];
    return DNode{ { a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w } };
}

// A node read at device scope (past the CU's L1): inside one kernel, what other waves appended or
// inserted with device-scope stores and atomics is seen.
__device__ __forceinline__ DNode load_node_coherent(const uint32_t* base, uint64_t i)
{
    DNode n;
#pragma unroll
    for (int c = 0; c < 8; c++) n.c[c] = __hip_atomic_load(base + i * 8 + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return n;
}

__device__ __forceinline__ void store_node(uint32_t* __restrict__ base, uint64_t i, const DNode& n)
{
    uint4* q = reinterpret_cast<uint4*>(base + i * 8);
    q[0] = make_uint4(n.c[0], n.c[1], n.c[2], n.c[3]);
    q[1] = make_uint4(n.c[4], n.c[5], n.c[6], n.c[7]);
}

__device__ __forceinline__ bool node_eq(const DNode& a, const DNode& b)
{
    bool e = true;
#pragma unroll
    for (int i = 0; i < 8; i++) e = e && a.c[i] == b.c[i];
    return e;
}

// The host interner's node hash (edits.cpp hash_node); any hash would do, this one is shared.
__device__ __forceinline__ uint64_t hash_node(const DNode& n)
{
    uint64_t h = 0x243f6a8885a308d3ULL;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        h ^= n.c[i];
        h *= 0x9fb21c651e98df25ULL;
        h ^= h >> 29;
    }
    return h;
}

// Adds store node j to the index: an empty slot is claimed with a compare-and-swap; where an equal
// node already sits, the lower index stays. kCoherent: for a kernel that appends nodes meanwhile.
template <bool kCoherent = false>
__device__ void index_insert(const uint32_t* __restrict__ nodes, uint32_t* __restrict__ slots, uint64_t mask, uint32_t j,
                             const DNode& n)
{
    for (uint64_t i = hash_node(n) & mask;; i = (i + 1) & mask) {
        const uint32_t cur = atomicCAS(&slots[i], kEmptySlot, j);
        if (cur == kEmptySlot) return;
        if (node_eq(kCoherent ? load_node_coherent(nodes, cur) : load_node(nodes, cur), n)) {
            atomicMin(&slots[i], j);
            return;
        }
    }
}

__global__ void __launch_bounds__(256) k_fill_u32(uint32_t* __restrict__ p, uint64_t count, uint32_t v)
{
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += uint64_t(gridDim.x) * blockDim.x)
        p[i] = v;
}

__global__ void __launch_bounds__(256) k_index_insert(const uint32_t* __restrict__ nodes, uint64_t from, uint64_t to,
                                                      uint32_t* __restrict__ slots, uint64_t mask)
{
    for (uint64_t j = from + uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; j < to;
         j += uint64_t(gridDim.x) * blockDim.x)
        index_insert(nodes, slots, mask, uint32_t(j), load_node(nodes, j));
}

// ---- the region walk ------------------------------------------------------------------------------

struct DRegionKey {
    uint32_t x, y, z;
};

// What a call's kernels leave for the host, read in one copy where the host needs it.
struct EditReport {
    uint64_t listed;    // nodes the regions listed
    uint64_t kept;      // of them, the distinct ones
    uint32_t outgrown;  // a region outgrew its slice
    uint32_t next_run;  // the region walk's work counter
    uint32_t count;     // store size after the levels above the regions
    uint32_t root;
    uint32_t deep;      // k_find_subdags: a single-child chain deeper than the tree
    uint32_t fresh[29]; // per level above the regions: whether it has new nodes
    cqx_subdag sub[8];
};

// SphereBrush (voxelization.h:91-126) in FP32, as SphereBrushF in edits.cpp.
struct Brush {
    float cx, cy, cz, r2;
    float lo[3], hi[3];

    __device__ explicit Brush(const cqx_sphere_edit& e)
    {
        cx = e.centre[0];
        cy = e.centre[1];
        cz = e.centre[2];
        r2 = e.radius * e.radius;
        const float c[3] = { cx, cy, cz };
        for (int a = 0; a < 3; a++) {
            lo[a] = c[a] - e.radius;
            hi[a] = c[a] + e.radius;
        }
    }

    // SphereBrush::contains: FP32 squared distance truncated to int64 (out of range and NaN give
    // INT64_MIN, as the x86-64 conversion does), compared as float with r2, strictly.
    __device__ bool contains(float x, float y, float z) const
    {
        const float dx = x - cx, dy = y - cy, dz = z - cz;
        const float sum = dx * dx + dy * dy + dz * dz;
        // within int64's range the truncated sum is a float itself: float(int64_t(sum)) = truncf(sum)
        const bool fits = sum >= -9.2233720368547758e18f && sum < 9.2233720368547758e18f;
        return (fits ? truncf(sum) : -9.2233720368547758e18f) < r2;
    }

    // SphereBrushF::box_outside: contains() is false everywhere in the box, with margins for its
    // FP32 rounding; FP64 arithmetic, the same operations in the same order.
    __device__ bool box_outside(float x0, float y0, float z0, float x1, float y1, float z1) const
    {
        const double c[3] = { cx, cy, cz }, lo3[3] = { x0, y0, z0 }, hi3[3] = { x1, y1, z1 };
        double dmin = 0.0, dmax = 0.0;
        for (int a = 0; a < 3; a++) {
            const double below = lo3[a] - c[a], above = c[a] - hi3[a];
            const double nearest = below > 0.0 ? below : (above > 0.0 ? above : 0.0);
            const double p = fabs(lo3[a] - c[a]), q = fabs(hi3[a] - c[a]);
            const double farthest = (p < q) ? q : p; // std::max
            dmin += nearest * nearest;
            dmax += farthest * farthest;
        }
        return dmax < 1e18 && dmin > double(r2) * (1.0 + 1e-5) + 16.0;
    }
};

struct RegionArgs {
    const uint32_t* nodes;  // the store (read-only during the walk)
    const uint32_t* index;  // index over the store
    uint64_t index_mask;
    uint32_t root;
    int hs;
    uint32_t base; // store size when the call began: list entries are base + position
    const cqx_sphere_edit* edits;
    const DRegionKey* keys;
    const uint64_t* first;    // keys + 1 offsets into edit_ids
    const uint32_t* edit_ids;
    const uint32_t* run; // the regions this launch runs, heaviest first
    uint32_t n_run;
    uint32_t* next_run;  // work counter: the next entry of `run` to take (zero at launch)
    const uint64_t* pool_off; // each region's slice: pool nodes [pool_off, pool_off + cap)
    const uint32_t* cap;      // power of two
    uint32_t* pool;           // listed nodes, 8 words each
    uint32_t* table;          // each region's hash table: 2 x cap slots from 2 x pool_off
    uint32_t* counts;
    uint32_t* results;
    uint32_t* overflow;
};

// The walk of one region (one wave): lane l stands for child c = l / 8 of the node it is at and, of
// that child, corner or child k = l % 8; the height-2 children of a node of height 3 are one step together
// (bricks). Above that the walk is depth first with the children's children read as soon as a node is
// entered, so that entering a child waits for no memory. What is interned, and in which order, is the
// recursion's. The phase lasts as long as its longest walk, a chain of dependent reads: 1000 spheres in a
// 2048^3 volume 2.62 ms with a step per node, 0.69 ms with a step per height-2 node, 0.35 ms now (0.63 ms where
// most new nodes are in neither the store nor the list, 0.73 before).
struct Region {
    const RegionArgs& A;
    uint64_t poff;
    uint32_t cap;
    uint32_t count = 0;

    __device__ uint32_t child(uint32_t node, uint32_t c) const
    {
        if (node < kMat) return node;
        if (node >= A.base) return A.pool[(poff + (node - A.base)) * 8 + c];
        return A.nodes[uint64_t(node) * 8 + c];
    }
};

// A value that is the same in every active lane, as a scalar.
__device__ __forceinline__ uint32_t uni(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// Orders what lanes of the wave stored before what its lanes load after (a wave's memory
// operations reach its L1 and LDS in order).
__device__ __forceinline__ void wave_fence()
{
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Bits 0, 8, .., 56 of b as bits 0..7.
__device__ __forceinline__ uint32_t byte_bits(uint64_t b)
{
    return uint32_t(((b & 0x0101010101010101ull) * 0x0102040810204080ull) >> 56);
}
// Bit c: every bit, or any bit, of byte c set.
__device__ __forceinline__ uint32_t bytes_all(uint64_t b)
{
    b &= b >> 4;
    b &= b >> 2;
    return byte_bits(b & (b >> 1));
}
__device__ __forceinline__ uint32_t bytes_any(uint64_t b)
{
    b |= b >> 4;
    b |= b >> 2;
    return byte_bits(b | (b >> 1));
}

// A hash table of node indices probed for each group's node: 8 slots at a time, one per lane.
// `found` receives the index where one holds an equal node, else kEmptySlot, and `at` the first
// empty slot on the way. `look`: the groups that search (the same in a group's lanes).
__device__ __forceinline__ void probe_groups(const uint32_t* __restrict__ slots, uint64_t mask, const uint32_t* __restrict__ nodes,
                                             const DNode& n, uint64_t hash, bool look, uint32_t lane, uint32_t& found,
                                             uint64_t& at)
{
    const uint32_t c8 = lane & 56u, k = lane & 7u;
    uint64_t i = hash & mask;
    while (__ballot(look)) {
        const uint32_t s = look ? slots[(i + k) & mask] : kEmptySlot;
        const uint32_t empty = uint32_t(__ballot(look && s == kEmptySlot) >> c8) & 0xffu;
        const uint32_t first = empty ? uint32_t(__builtin_ctz(empty)) : 8u;
        const bool eq = look && k < first && node_eq(load_node(nodes, s), n);
        const uint32_t match = uint32_t(__ballot(eq) >> c8) & 0xffu;
        const uint32_t hit = uint32_t(__shfl(int(s), int(c8 + (match ? uint32_t(__builtin_ctz(match)) : 0u))));
        if (look) {
            if (match) found = hit;
            else if (empty) at = (i + first) & mask;
            else i += 8;
            look = !match && !empty;
        }
    }
}

// RegionStore::intern of each group's node (`w`: word k of group c's node) whose bit is set in
// `active`, in group order: 8 equal material children collapse; a node without listed children
// that is in the store is shared; otherwise the region's list keeps one copy of each node. The
// group's node index in all its lanes; false when the list outgrew its slice. kNew: the nodes are known not to
// collapse and not to be in the store.
template <bool kNew = false>
__device__ bool intern_groups(Region& R, uint32_t w, uint32_t active, uint32_t lane, uint32_t& result)
{
    const RegionArgs& A = R.A;
    const uint32_t c8 = lane & 56u, c = lane >> 3, k = lane & 7u;
    DNode n;
    bool uniform = true, listed = false;
#pragma unroll
    for (uint32_t i = 0; i < 8; i++) {
        n.c[i] = uint32_t(__shfl(int(w), int(c8 + i)));
        uniform = uniform && n.c[i] == n.c[0];
        listed = listed || n.c[i] >= A.base;
    }
    uniform = uniform && n.c[0] < kMat;
    const bool need = ((active >> c) & 1u) && !uniform;
    uint32_t r = uniform ? n.c[0] : kEmptySlot;
    const uint64_t hash = hash_node(n);
    uint64_t at = 0;
    if (!kNew) probe_groups(A.index, A.index_mask, A.nodes, n, hash, need && !listed, lane, r, at);
    uint32_t* const tab = A.table + R.poff * 2;
    const uint64_t tmask = uint64_t(R.cap) * 2 - 1;
    uint32_t local = kEmptySlot;
    const bool look = need && r == kEmptySlot;
    probe_groups(tab, tmask, A.pool + R.poff * 8, n, hash, look, lane, local, at);
    if (look && local != kEmptySlot) r = A.base + local;
    uint32_t fresh = byte_bits(__ballot(look && local == kEmptySlot));
    uint64_t mine = ~0ull; // lane j: the slot of the j-th node added here
    uint32_t added = 0;
    while (fresh) { // each group's node not listed yet, once per distinct node
        const uint32_t g = uint32_t(__builtin_ctz(fresh));
        bool eq = true;
#pragma unroll
        for (uint32_t i = 0; i < 8; i++) eq = eq && n.c[i] == uint32_t(__builtin_amdgcn_readlane(int(w), int(8 * g + i)));
        const uint32_t same = byte_bits(__ballot(eq)) & fresh;
        if (R.count >= R.cap) return false;
        const uint32_t idx = R.count++;
        uint64_t slot = uint64_t(uint32_t(__builtin_amdgcn_readlane(int(uint32_t(at)), int(8 * g)))) |
                        uint64_t(uint32_t(__builtin_amdgcn_readlane(int(uint32_t(at >> 32)), int(8 * g)))) << 32;
        // a node added just now may sit there: on to the next empty slot
        bool first = true;
        while (__ballot(mine == slot) || (!first && tab[slot] != kEmptySlot)) {
            slot = (slot + 1) & tmask;
            first = false;
        }
        if (c == g) A.pool[(R.poff + idx) * 8 + k] = w;
        if (lane == 0) tab[slot] = idx;
        if (lane == added) mine = slot;
        added++;
        if ((same >> c) & 1u) r = A.base + idx;
        fresh &= ~same;
    }
    wave_fence();
    result = r;
    return true;
}

// Interns one node, its child c's index in the lanes of group c.
__device__ bool intern_one(Region& R, uint32_t out, uint32_t lane, uint32_t& result)
{
    const uint32_t w = uint32_t(__shfl(int(out), int((lane & 7u) * 8u)));
    if (!intern_groups(R, w, 1u, lane, result)) return false;
    result = uni(result);
    return true;
}

// The children of a node (lower corner lo, children of side `side`) against the brush, as masks over
// the children: those to be filled and those to be walked. False when no child's float box overlaps
// the brush bounds (geometry.h:346-357): the node stays.
__device__ __forceinline__ bool test_children(const Brush& b, uint32_t mat, uint32_t child, uint32_t side, int32_t lx,
                                              int32_t ly, int32_t lz, uint32_t lane, uint32_t& fill, uint32_t& walk)
{
    const uint32_t c = lane >> 3, k = lane & 7u;
    const int32_t x0 = int32_t(uint32_t(lx) + side * (c & 1u)), y0 = int32_t(uint32_t(ly) + side * ((c >> 1) & 1u)),
                  z0 = int32_t(uint32_t(lz) + side * (c >> 2));
    const float fx0 = float(x0), fy0 = float(y0), fz0 = float(z0);
    const float fx1 = float(int32_t(uint32_t(x0) + (side - 1))), fy1 = float(int32_t(uint32_t(y0) + (side - 1))),
                fz1 = float(int32_t(uint32_t(z0) + (side - 1)));
    const bool ok = !(b.hi[0] < fx0 || b.lo[0] > fx1) && !(b.hi[1] < fy0 || b.lo[1] > fy1) &&
                    !(b.hi[2] < fz0 || b.lo[2] > fz1);
    fill = walk = 0;
    const uint64_t okb = __ballot(ok);
    if (okb == 0) return false;
    const bool corner = b.contains((k & 1u) ? fx1 : fx0, (k & 2u) ? fy1 : fy0, (k & 4u) ? fz1 : fz0);
    const uint32_t all = bytes_all(__ballot(corner));
    const uint32_t live = byte_bits(__ballot(ok && child != mat));
    fill = live & all;
    walk = live & ~all;
    // (a child with all corners inside is not outside the sphere)
    if (walk) walk &= ~byte_bits(__ballot(b.box_outside(fx0, fy0, fz0, fx1, fy1, fz1)));
    return true;
}

// Index of a store node with this content, or kEmptySlot: a lane's own search, two slots' nodes at a time.
__device__ uint32_t store_find(const RegionArgs& A, const DNode& n)
{
    for (uint64_t i = hash_node(n) & A.index_mask;; i += 2) {
        const uint32_t s0 = A.index[i & A.index_mask], s1 = A.index[(i + 1) & A.index_mask];
        if (s0 == kEmptySlot) return kEmptySlot;
        const DNode a = load_node(A.nodes, s0), b = load_node(A.nodes, s1 == kEmptySlot ? s0 : s1);
        if (node_eq(a, n)) return s0;
        if (s1 == kEmptySlot) return kEmptySlot;
        if (node_eq(b, n)) return s1;
    }
}

// fillBrush on the children in `walk` of a node of height 3 (lower corner lo), height-2 nodes ("bricks"):
// lane l stands for child c = l % 8 of brick l / 8, `kid`; `out` holds the brick's node in its 8 lanes and
// receives the new one. A lane tests its child and the child's 8 voxels and searches the store for the
// new node, for all bricks at once; what is not there goes into the region's list brick by brick, in
// the recursion's order, and if everything is, the bricks' own nodes are interned together. A step per
// brick instead (its 8 children by 8 lanes each) was a chain of 5 reads a brick, against 2 to 3 now and, with
// nothing new, 5 for all 8.
__device__ bool bricks(Region& R, const Brush& b, uint32_t mat, uint32_t walk, uint32_t kid, int32_t lx, int32_t ly,
                       int32_t lz, uint32_t lane, uint32_t& out, uint32_t& changed)
{
    const RegionArgs& A = R.A;
    const uint32_t g = lane >> 3, c = lane & 7u;
    const uint32_t x0 = uint32_t(lx) + 4u * (g & 1u) + 2u * (c & 1u), y0 = uint32_t(ly) + 4u * ((g >> 1) & 1u) + 2u * ((c >> 1) & 1u),
                   z0 = uint32_t(lz) + 4u * (g >> 2) + 2u * (c >> 2);
    const float fx[2] = { float(int32_t(x0)), float(int32_t(x0 + 1u)) }, fy[2] = { float(int32_t(y0)), float(int32_t(y0 + 1u)) },
                fz[2] = { float(int32_t(z0)), float(int32_t(z0 + 1u)) };
    uint32_t next = kid;   // the child's new node
    bool fresh = false;    // not settled: in neither the store nor, yet, the list
    DNode n;
    const bool ok = ((walk >> g) & 1u) && kid != mat && !(b.hi[0] < fx[0] || b.lo[0] > fx[1]) &&
                    !(b.hi[1] < fy[0] || b.lo[1] > fy[1]) && !(b.hi[2] < fz[0] || b.lo[2] > fz[1]);
    if (ok) {
        uint32_t inside = 0;
#pragma unroll
        for (uint32_t k = 0; k < 8; k++) inside |= (b.contains(fx[k & 1u], fy[(k >> 1) & 1u], fz[k >> 2]) ? 1u : 0u) << k;
        if (inside == 0xffu) next = mat;
        else if (!b.box_outside(fx[0], fy[0], fz[0], fx[1], fy[1], fz[1])) {
            if (kid < kMat)
                for (uint32_t& w : n.c) w = kid;
            else n = kid >= A.base ? load_node(A.pool, R.poff + (kid - A.base)) : load_node(A.nodes, kid);
            bool differs = false, uniform = true, listed = false;
#pragma unroll
            for (uint32_t k = 0; k < 8; k++) {
                const float x = fx[k & 1u], y = fy[(k >> 1) & 1u], z = fz[k >> 2];
                const bool in = !(b.hi[0] < x || b.lo[0] > x) && !(b.hi[1] < y || b.lo[1] > y) && !(b.hi[2] < z || b.lo[2] > z);
                if (in && ((inside >> k) & 1u) && n.c[k] != mat) {
                    n.c[k] = mat;
                    differs = true;
                }
                uniform = uniform && n.c[k] == n.c[0];
                listed = listed || n.c[k] >= A.base;
            }
            if (differs) {
                next = uniform && n.c[0] < kMat ? n.c[0] : listed ? kEmptySlot : store_find(A, n);
                fresh = next == kEmptySlot;
            }
        }
    }
    if (__ballot(fresh) == 0) { // word c of brick g's node is `next`
        const uint32_t differ = bytes_any(__ballot(next != kid && ((walk >> g) & 1u)));
        if (!differ) return true;
        uint32_t r;
        if (!intern_groups(R, next, differ, lane, r)) return false;
        if ((differ >> g) & 1u) out = r; // (a brick that changed is another node)
        changed = 1u;
        return true;
    }
    for (; walk; walk &= walk - 1u) {
        const uint32_t at = uint32_t(__builtin_ctz(walk));
        const uint32_t add = uint32_t(__ballot(fresh) >> (8u * at)) & 0xffu; // children of brick `at`
        if (add) { // to lane (group c', word k) from lane 8 at + c'
            uint32_t w = 0, r;
#pragma unroll
            for (uint32_t k = 0; k < 8; k++) {
                const uint32_t v = uint32_t(__shfl(int(n.c[k]), int(8u * at + g)));
                w = k == c ? v : w;
            }
            if (!intern_groups<true>(R, w, add, lane, r)) return false;
            const uint32_t mine = uint32_t(__shfl(int(r), int(8u * c)));
            if (g == at && fresh) next = mine;
        }
        if ((__ballot(next != kid) >> (8u * at) & 0xffu) == 0) continue;
        uint32_t r;
        const uint32_t w = uint32_t(__shfl(int(next), int(8u * at + c)));
        if (!intern_groups(R, w, 1u, lane, r)) return false;
        r = uni(r); // of group 0
        if (g == at) out = r;
        changed = 1u;
    }
    return true;
}

// A node of height 3 or more on the way down, saved while a child of it is walked.
struct Frame {
    uint32_t kid[64]; // child c's children
    uint32_t out[8];
    uint32_t node;
    int32_t lo[3];
    uint32_t walk;    // children still to be walked
    uint32_t at;      // the one being walked
    uint32_t changed;
};

// EditWalk::fill (edits.cpp) on the region's node (height hs >= 5, lower corner lo); false when the
// list outgrew its slice.
__device__ bool fill(Region& R, const Brush& b, uint32_t mat, uint32_t node, uint32_t height, int32_t lx, int32_t ly,
                     int32_t lz, Frame* st, uint32_t lane, uint32_t& result)
{
    const uint32_t c = lane >> 3, k = lane & 7u;
    uint32_t out = R.child(node, c), walk, set, kid = 0, changed;
    result = node;
    if (!test_children(b, mat, out, 1u << (height - 1), lx, ly, lz, lane, set, walk)) return true;
    uint32_t sp = 0;
    const auto enter = [&] { // the node's children tested: what is filled, and the next level's reads
        changed = set ? 1u : 0u;
        if ((set >> c) & 1u) out = mat;
        if ((walk >> c) & 1u) kid = R.child(out, k);
    };
    enter();
    for (;;) {
        if (walk == 0) {
            uint32_t res = node;
            if (changed && !intern_one(R, out, lane, res)) return false;
            if (sp == 0) {
                result = res;
                return true;
            }
            const Frame& f = st[--sp];
            height++;
            kid = f.kid[lane];
            out = f.out[c];
            node = uni(f.node);
            lx = int32_t(uni(uint32_t(f.lo[0])));
            ly = int32_t(uni(uint32_t(f.lo[1])));
            lz = int32_t(uni(uint32_t(f.lo[2])));
            walk = uni(f.walk);
            changed = uni(f.changed);
            const uint32_t at = uni(f.at);
            const bool differs = __ballot(c == at && out != res) != 0;
            if (c == at) out = res;
            changed |= differs ? 1u : 0u;
            continue;
        }
        if (height == 3) {
            if (!bricks(R, b, mat, walk, kid, lx, ly, lz, lane, out, changed)) return false;
            walk = 0;
            continue;
        }
        const uint32_t at = uint32_t(__builtin_ctz(walk));
        walk &= walk - 1u;
        const uint32_t side = 1u << (height - 1);
        const uint32_t child = uint32_t(__builtin_amdgcn_readlane(int(out), int(8 * at)));
        const uint32_t grand = uint32_t(__shfl(int(kid), int(8 * at + c))); // the child's child c
        const int32_t cx = int32_t(uint32_t(lx) + side * (at & 1u)), cy = int32_t(uint32_t(ly) + side * ((at >> 1) & 1u)),
                      cz = int32_t(uint32_t(lz) + side * (at >> 2));
        uint32_t cset, cwalk;
        if (!test_children(b, mat, grand, side >> 1, cx, cy, cz, lane, cset, cwalk)) continue;
        Frame& f = st[sp++];
        f.kid[lane] = kid;
        if (k == 0) f.out[c] = out;
        if (lane == 0) {
            f.node = node;
            f.lo[0] = lx;
            f.lo[1] = ly;
            f.lo[2] = lz;
            f.walk = walk;
            f.at = at;
            f.changed = changed;
        }
        wave_fence();
        node = child;
        height--;
        lx = cx;
        ly = cy;
        lz = cz;
        out = grand;
        set = cset;
        walk = cwalk;
        enter();
    }
}

// The node at height h that holds key k (granularity 2^h), by descent from the root.
__device__ uint32_t node_at(const uint32_t* __restrict__ nodes, uint32_t root, int h, const DRegionKey& k)
{
    if (h >= 32) return root;
    uint32_t node = root;
    const uint32_t ux = k.x << h, uy = k.y << h, uz = k.z << h;
    for (int level = 32; level > h && node >= kMat; level--) {
        const uint32_t c = ((ux >> (level - 1)) & 1u) | (((uy >> (level - 1)) & 1u) << 1) |
                           (((uz >> (level - 1)) & 1u) << 2);
        node = nodes[uint64_t(node) * 8 + c];
    }
    return node;
}

__global__ void __launch_bounds__(64) k_edit_regions(RegionArgs A)
{
    extern __shared__ Frame st[]; // hs - 3: nodes of heights hs .. 4 while a child is walked
    const uint32_t lane = threadIdx.x;
    for (;;) { // one region per wave, taken from the work counter: the heaviest start first
        uint32_t t = 0;
        if (lane == 0) t = atomicAdd(A.next_run, 1u);
        t = uint32_t(__shfl(int(t), 0));
        if (t >= A.n_run) break;
        const uint32_t r = A.run[t];
        Region R{ A, A.pool_off[r], A.cap[r] };
        uint32_t* const tab = A.table + R.poff * 2;
        for (uint64_t i = lane; i < uint64_t(R.cap) * 2; i += 64) tab[i] = kEmptySlot;
        wave_fence();
        const DRegionKey k = A.keys[r];
        uint32_t node = node_at(A.nodes, A.root, A.hs, k);
        const int32_t lx = int32_t((k.x << A.hs) - 0x80000000u), ly = int32_t((k.y << A.hs) - 0x80000000u),
                      lz = int32_t((k.z << A.hs) - 0x80000000u);
        uint32_t over = 0;
        for (uint64_t j = A.first[r]; j < A.first[r + 1]; j++) {
            const cqx_sphere_edit e = A.edits[A.edit_ids[j]];
            const Brush b(e);
            uint32_t next;
            if (!fill(R, b, e.material, node, uint32_t(A.hs), lx, ly, lz, st, lane, next)) {
                over = 1;
                break;
            }
            node = next;
        }
        if (lane == 0) {
            A.results[r] = node;
            A.counts[r] = R.count;
            A.overflow[r] = over;
        }
        wave_fence();
    }
}

// ---- merge of the regions' lists (merge_regions, edits.cpp) ----------------------------------------

struct MergeArgs {
    uint32_t base;
    uint32_t nr;
    const uint64_t* pool_off;
    const uint32_t* pool;
    const uint32_t* counts;
    const uint64_t* off; // list position of each region's first node (exclusive scan of counts)
    uint64_t total;
    uint32_t* src;      // position -> pool node
    uint32_t* region;   // position -> region
    uint8_t* level;     // position -> level (1 + deepest listed child)
    uint32_t* key;      // position -> 8 words: the node with listed children as base + their kept position
    uint64_t* slot_of;  // position -> its slot in the merge table
    uint32_t* rep;      // position -> kept position of its node
    uint32_t* table;    // merge table
    uint64_t table_mask;
};

// The lists laid end to end, with each node's level: a wave per region, 64 nodes at a time. A node's listed
// children come before it: those of earlier rows have their levels, those among the 64 are settled in as
// many turns as their chain is long (at most the region's height). One thread a region, a node at a
// time, took 114 to 200 us of an edit of 1000 spheres at 2048^3, 10 us now.
__global__ void __launch_bounds__(64) k_merge_flatten(MergeArgs M)
{
    const uint32_t lane = threadIdx.x;
    for (uint32_t r = blockIdx.x; r < M.nr; r += gridDim.x) {
        const uint64_t o = M.off[r], poff = M.pool_off[r];
        const uint32_t count = M.counts[r];
        for (uint32_t row = 0; row < count; row += 64) {
            const uint32_t l = row + lane;
            const bool have = l < count;
            DNode n{};
            if (have) n = load_node(M.pool, poff + l);
            uint32_t lv = 0;
#pragma unroll
            for (int c = 0; c < 8; c++) {
                const uint32_t x = n.c[c] - M.base; // list position of a listed child
                if (have && n.c[c] >= M.base && x < row) lv = max(lv, uint32_t(M.level[o + x]) + 1u);
            }
            for (bool more = true; __ballot(more);) {
                more = false;
#pragma unroll
                for (int c = 0; c < 8; c++) {
                    const uint32_t x = n.c[c] - M.base;
                    const uint32_t under = uint32_t(__shfl(int(lv), int(x & 63u))) + 1u;
                    if (have && n.c[c] >= M.base && x >= row && under > lv) {
                        lv = under;
                        more = true;
                    }
                }
            }
            if (have) {
                M.src[o + l] = uint32_t(poff + l);
                M.region[o + l] = r;
                M.level[o + l] = uint8_t(lv);
            }
            wave_fence();
        }
    }
}

// Level `lv`: the keys (listed children replaced by base + their kept positions, which lower
// levels have settled).
__global__ void __launch_bounds__(256) k_merge_keys(MergeArgs M, uint32_t lv)
{
    for (uint64_t g = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; g < M.total; g += uint64_t(gridDim.x) * blockDim.x) {
        if (M.level[g] != lv) continue;
        DNode k = load_node(M.pool, M.src[g]);
        const uint64_t o = M.off[M.region[g]];
        for (int c = 0; c < 8; c++)
            if (k.c[c] >= M.base) k.c[c] = M.base + M.rep[o + (k.c[c] - M.base)];
        store_node(M.key, g, k);
    }
}

// Level `lv`: the lowest position of each set of equal keys ends up in their slot.
__global__ void __launch_bounds__(256) k_merge_insert(MergeArgs M, uint32_t lv)
{
    for (uint64_t g = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; g < M.total; g += uint64_t(gridDim.x) * blockDim.x) {
        if (M.level[g] != lv) continue;
        const DNode k = load_node(M.key, g);
        for (uint64_t i = hash_node(k) & M.table_mask;; i = (i + 1) & M.table_mask) {
            const uint32_t cur = atomicCAS(&M.table[i], kEmptySlot, uint32_t(g));
            if (cur == kEmptySlot || node_eq(load_node(M.key, cur), k)) {
                if (cur != kEmptySlot) atomicMin(&M.table[i], uint32_t(g));
                M.slot_of[g] = i;
                break;
            }
        }
    }
}

__global__ void __launch_bounds__(256) k_merge_rep(MergeArgs M, uint32_t lv)
{
    for (uint64_t g = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; g < M.total; g += uint64_t(gridDim.x) * blockDim.x)
        if (M.level[g] == lv) M.rep[g] = M.table[M.slot_of[g]];
}

// Exclusive prefix sums in one workgroup of 1024 threads (each thread a contiguous run).
__device__ void block_exclusive_scan_u64(uint64_t* __restrict__ v, uint64_t n, uint64_t* __restrict__ total)
{
    __shared__ uint64_t part[1024];
    const uint32_t t = threadIdx.x, T = blockDim.x;
    const uint64_t per = (n + T - 1) / T;
    const uint64_t b = uint64_t(t) * per < n ? uint64_t(t) * per : n, e = b + per < n ? b + per : n;
    uint64_t s = 0;
    for (uint64_t i = b; i < e; i++) s += v[i];
    part[t] = s;
    __syncthreads();
    for (uint32_t d = 1; d < T; d <<= 1) {
        const uint64_t x = t >= d ? part[t - d] : 0;
        __syncthreads();
        part[t] += x;
        __syncthreads();
    }
    uint64_t run = part[t] - s;
    for (uint64_t i = b; i < e; i++) {
        const uint64_t x = v[i];
        v[i] = run;
        run += x;
    }
    if (t == T - 1) *total = part[t];
    __syncthreads();
}

__global__ void __launch_bounds__(1024) k_scan_u64(uint64_t* v, uint64_t n, uint64_t* total)
{
    block_exclusive_scan_u64(v, n, total);
}

// Exclusive prefix sums over many workgroups: tiles of kScanTile values, 4 consecutive values per
// thread. k_scan_tile_sums sums each tile, the tile sums are scanned in one workgroup, and
// k_scan_tiles scans each tile from its tile's offset.
constexpr uint32_t kScanBlock = 1024, kScanTile = 4 * kScanBlock;

__device__ uint64_t block_sum_u64(uint64_t s)
{
    __shared__ uint64_t part[kScanBlock / 64];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if ((threadIdx.x & 63u) == 0) part[threadIdx.x >> 6] = s;
    __syncthreads();
    uint64_t t = 0;
    for (uint32_t w = 0; w < blockDim.x / 64; w++) t += part[w];
    return t;
}

__global__ void __launch_bounds__(kScanBlock) k_scan_tile_sums(const uint64_t* __restrict__ v, uint64_t n,
                                                               uint64_t* __restrict__ sums)
{
    const uint64_t first = uint64_t(blockIdx.x) * kScanTile + uint64_t(threadIdx.x) * 4;
    uint64_t s = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) s += first + k < n ? v[first + k] : 0u;
    const uint64_t t = block_sum_u64(s);
    if (threadIdx.x == 0) sums[blockIdx.x] = t;
}

__global__ void __launch_bounds__(kScanBlock) k_scan_tiles(uint64_t* __restrict__ v, uint64_t n,
                                                           const uint64_t* __restrict__ offsets)
{
    __shared__ uint64_t part[kScanBlock];
    const uint64_t first = uint64_t(blockIdx.x) * kScanTile + uint64_t(threadIdx.x) * 4;
    uint64_t x[4], s = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        x[k] = first + k < n ? v[first + k] : 0u;
        s += x[k];
    }
    const uint32_t t = threadIdx.x;
    part[t] = s;
    __syncthreads();
    for (uint32_t d = 1; d < blockDim.x; d <<= 1) {
        const uint64_t y = t >= d ? part[t - d] : 0;
        __syncthreads();
        part[t] += y;
        __syncthreads();
    }
    uint64_t run = offsets[blockIdx.x] + part[t] - s;
#pragma unroll
    for (int k = 0; k < 4; k++)
        if (first + k < n) {
            v[first + k] = run;
            run += x[k];
        }
}

__global__ void __launch_bounds__(256) k_region_counts(const uint32_t* __restrict__ c, const uint32_t* __restrict__ overflow,
                                                       uint64_t* __restrict__ o, uint32_t n, EditReport* __restrict__ rep)
{
    bool over = false;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        o[i] = c[i];
        over = over || overflow[i];
    }
    if (over) rep->outgrown = 1u;
}

__global__ void __launch_bounds__(64) k_edit_begin(EditReport* __restrict__ rep)
{
    if (threadIdx.x == 0) {
        rep->outgrown = 0u;
        rep->next_run = 0u;
    }
    if (threadIdx.x < sizeof(rep->fresh) / 4) rep->fresh[threadIdx.x] = 0u;
}

__global__ void __launch_bounds__(256) k_merge_kept(MergeArgs M, uint64_t* kept)
{
    for (uint64_t g = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; g < M.total; g += uint64_t(gridDim.x) * blockDim.x)
        kept[g] = M.rep[g] == uint32_t(g) ? 1u : 0u;
}

// The kept nodes into the store at base + their rank (fin), listed children mapped to the store
// indices of their kept nodes; the regions' results mapped the same way.
__global__ void __launch_bounds__(256) k_merge_write(MergeArgs M, const uint64_t* __restrict__ fin, uint32_t* __restrict__ nodes,
                                                     uint32_t* __restrict__ results)
{
    for (uint64_t g = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; g < M.total; g += uint64_t(gridDim.x) * blockDim.x) {
        if (M.rep[g] != uint32_t(g)) continue;
        DNode k = load_node(M.pool, M.src[g]);
        const uint64_t o = M.off[M.region[g]];
        for (int c = 0; c < 8; c++)
            if (k.c[c] >= M.base) k.c[c] = M.base + uint32_t(fin[M.rep[o + (k.c[c] - M.base)]]);
        store_node(nodes, M.base + fin[g], k);
    }
    for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < M.nr; r += gridDim.x * blockDim.x) {
        const uint32_t x = results[r];
        if (x >= M.base) results[r] = M.base + uint32_t(fin[M.rep[M.off[r] + (x - M.base)]]);
    }
}

// ---- the levels above the regions (rebuild_levels, edits.cpp) ---------------------------------------

struct TopArgs {
    uint32_t* nodes;
    uint32_t* index;
    uint64_t index_mask;
    uint32_t root;
    int hs;
    uint32_t levels;          // 32 - hs
    const uint32_t* lvl_off;  // levels + 2 entry offsets: level l is [lvl_off[l], lvl_off[l + 1])
    const DRegionKey* keys;   // per entry
    const uint32_t* cbeg;     // per entry of level >= 1: its children, entries [cbeg, cend) of level l - 1
    const uint32_t* cend;
    const uint32_t* morton_regions; // level 0 entry -> region
    const uint32_t* results;        // region -> new node
    uint32_t* res;        // per entry: the node after the edits
    uint32_t* cand;       // per entry: 1 when it is a new node to intern
    uint32_t* ckey;       // per entry: 8 words
    uint32_t* crep;       // per entry: the first entry of its level with the same node
    uint64_t* cslot;
    uint32_t* table;      // per level: 2 x pow2 slots from tab_off[l]
    const uint64_t* tab_off;
    uint32_t count;       // store size after the merge
    EditReport* rep;
    uint32_t* old;        // per entry of level >= 1: the node it held before the edits

    // The new node of entry j of level l.
    __device__ uint32_t result(uint32_t l, uint32_t j) const { return l == 0 ? results[morton_regions[j]] : res[j]; }
};

// Index of a store node with this content, or kEmptySlot, while nodes are appended and inserted: 4
// slots are read at once, since a probe is a chain of memory latencies.
__device__ uint32_t index_find(const uint32_t* nodes, const uint32_t* slots, uint64_t mask, const DNode& n)
{
    for (uint64_t i = hash_node(n) & mask;; i += 4) {
        uint32_t s[4];
#pragma unroll
        for (int j = 0; j < 4; j++)
            s[j] = __hip_atomic_load(slots + ((i + j) & mask), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (s[j] == kEmptySlot) return kEmptySlot;
            if (node_eq(load_node_coherent(nodes, s[j]), n)) return s[j];
        }
    }
}

// The levels of at most 64 entries ("small"; with a level every one above it is), on one wave with an
// entry per lane, their schedule, old nodes and results in LDS and equal new nodes found by comparing
// lanes. Above a volume's own height a level holds an entry or a few and depends on the one below, so
// the time is a chain of memory latencies: per level one read going down, and going up the index slots,
// a node and the insertion, the old node's words being read a level ahead. At 2048^3, 1000 spheres of
// radius 2 to 16 (4700 regions, 24 of the 27 levels small): 780 us with every level on the
// workgroup (5 barriers and as many passes through memory each, fences at device scope), 65 us the small ones so.
constexpr uint32_t kTopLevels = 28; // 32 - hs for hs >= 5, and level 0
struct SmallTop {
    uint32_t off[kTopLevels + 1]; // lvl_off
    uint32_t first;               // the lowest small level, >= 1
    uint32_t kids[kTopLevels * 64]; // of small entry e (at e - off[first]): cbeg | octant in the parent << 26 | count << 29
    uint32_t old[kTopLevels * 64];  // the node it held before the edits
    uint32_t below[64];
};

__device__ __forceinline__ uint32_t key_octant(const DRegionKey& k)
{
    return (k.x & 1u) | (k.y & 1u) << 1 | (k.z & 1u) << 2;
}

// The schedule into LDS, by the whole workgroup; ends with a barrier.
__device__ void top_stage(const TopArgs& A, SmallTop& S, uint32_t t, uint32_t T)
{
    if (t < A.levels + 2) S.off[t] = A.lvl_off[t];
    __syncthreads();
    if (t == 0) {
        uint32_t l = 1;
        while (S.off[l + 1] - S.off[l] > 64) l++;
        S.first = l;
    }
    __syncthreads();
    const uint32_t b = S.off[S.first], n = S.off[A.levels + 1] - b;
    for (uint32_t i = t; i < n; i += T) {
        const uint32_t cb = A.cbeg[b + i];
        S.kids[i] = (cb - S.off[S.first - 1]) | key_octant(A.keys[b + i]) << 26 | (A.cend[b + i] - cb - 1) << 29;
    }
    __syncthreads();
}

// Old nodes of the small levels and of the level below them, top down.
__device__ void top_small_down(const TopArgs& A, SmallTop& S, uint32_t lane)
{
    const uint32_t b0 = S.off[S.first];
    if (lane == 0) S.old[S.off[A.levels] - b0] = A.root;
    wave_fence();
    for (uint32_t l = A.levels; l >= S.first && l >= 2; l--) {
        const uint32_t e = S.off[l] + lane;
        if (e < S.off[l + 1]) {
            const uint32_t p = S.old[e - b0], k = S.kids[e - b0];
            DNode in;
            if (p >= kMat) in = load_node(A.nodes, p);
            else
                for (uint32_t& x : in.c) x = p;
            const uint32_t cb = (k & 0x3ffffffu) + S.off[S.first - 1];
            for (uint32_t j = cb; j <= cb + (k >> 29); j++) {
                const uint32_t id = l > S.first ? (S.kids[j - b0] >> 26) & 7u : key_octant(A.keys[j]);
                uint32_t x = 0;
#pragma unroll
                for (uint32_t c = 0; c < 8; c++) x = c == id ? in.c[c] : x;
                if (l > S.first) S.old[j - b0] = x;
                else A.old[j] = x;
            }
        }
        wave_fence();
    }
}

// The small levels bottom up; `base` is the store's size.
__device__ void top_small_up(const TopArgs& A, SmallTop& S, uint32_t base, uint32_t lane)
{
    const uint32_t b0 = S.off[S.first], c0 = S.off[S.first - 1];
    const auto old_node = [&](uint32_t l, uint32_t& old, DNode& n) {
        const uint32_t e = S.off[l] + lane;
        old = l <= A.levels && e < S.off[l + 1] ? S.old[e - b0] : 0u;
        if (old >= kMat) n = load_node(A.nodes, old);
        else
            for (uint32_t& x : n.c) x = old;
    };
    uint32_t old, top = 0;
    DNode out;
    old_node(S.first, old, out);
    for (uint32_t l = S.first; l <= A.levels; l++) {
        const uint32_t e = S.off[l] + lane;
        const bool have = e < S.off[l + 1];
        uint32_t next_old;
        DNode next;
        old_node(l + 1, next_old, next);
        uint32_t r = old;
        bool fresh = false, changed = false;
        if (have) {
            const uint32_t k = S.kids[e - b0], cb = (k & 0x3ffffffu) + c0;
            for (uint32_t j = cb; j <= cb + (k >> 29); j++) {
                const uint32_t id = l > S.first ? (S.kids[j - b0] >> 26) & 7u : key_octant(A.keys[j]);
                const uint32_t x = l > S.first ? S.below[j - S.off[l - 1]] : A.result(l - 1, j);
#pragma unroll
                for (uint32_t c = 0; c < 8; c++)
                    if (c == id && out.c[c] != x) {
                        out.c[c] = x;
                        changed = true;
                    }
            }
        }
        if (changed) { // Interner::intern: collapse, else the store's node, else new
            bool uniform = out.c[0] < kMat;
#pragma unroll
            for (int c = 1; c < 8; c++) uniform = uniform && out.c[c] == out.c[0];
            r = uniform ? out.c[0] : index_find(A.nodes, A.index, A.index_mask, out);
            fresh = r == kEmptySlot;
        }
        // new nodes appended in entry order, equal ones once
        uint64_t todo = __ballot(fresh);
        while (todo) {
            const int g = __ffsll((unsigned long long)todo) - 1;
            bool eq = fresh;
#pragma unroll
            for (int c = 0; c < 8; c++) eq = eq && out.c[c] == uint32_t(__builtin_amdgcn_readlane(int(out.c[c]), g));
            todo &= ~__ballot(eq);
            if (eq) r = base;
            if (int(lane) == g) store_node(A.nodes, base, out);
            else if (eq) fresh = false; // the first of the equal ones inserts it
            base++;
        }
        wave_fence();
        if (fresh) index_insert<true>(A.nodes, A.index, A.index_mask, r, out);
        if (have) S.below[lane] = r;
        wave_fence();
        top = r;
        old = next_old;
        out = next;
    }
    if (lane == 0) {
        A.rep->count = base;
        A.rep->root = top; // the top level has one entry
    }
}

// The levels of more than 64 entries ("large", the lowest ones) are spread over the chip, a launch per step
// and level, and the new nodes of a level, if any, appended by one workgroup. At 2048^3, 1000 spheres, with
// four large levels: 130 us for the whole, against 200 us with every level on one workgroup, whose threads
// took 5 entries of a level one after the other; where the nodes are new, 290 us against 436.

// Old nodes of the small levels and of the level below them, for the launches of the large ones.
__global__ void __launch_bounds__(kTopBlock) k_top_begin(TopArgs A)
{
    __shared__ SmallTop small;
    const uint32_t t = threadIdx.x;
    if (t == 0) A.rep->count = A.count;
    top_stage(A, small, t, blockDim.x);
    if (t < 64) top_small_down(A, small, t);
    __syncthreads();
    const uint32_t b = small.off[small.first], n = small.off[A.levels + 1] - b;
    for (uint32_t i = t; i < n; i += blockDim.x) A.old[b + i] = small.old[i];
}

// Old nodes of level l - 1, from those of level l.
__global__ void __launch_bounds__(256) k_top_old(TopArgs A, uint32_t l, uint32_t begin, uint32_t end)
{
    const uint32_t i = begin + blockIdx.x * 256u + threadIdx.x;
    if (i >= end) return;
    const uint32_t p = A.old[i], ce = A.cend[i];
    for (uint32_t j = A.cbeg[i]; j < ce; j++) A.old[j] = p < kMat ? p : A.nodes[uint64_t(p) * 8 + key_octant(A.keys[j])];
}

// The nodes of level l after the edits, where the store has them; the others as candidates.
__global__ void __launch_bounds__(64) k_top_build(TopArgs A, uint32_t l, uint32_t begin, uint32_t end)
{
    const uint32_t i = begin + blockIdx.x * 64u + threadIdx.x;
    if (i >= end) return;
    const uint32_t old = A.old[i];
    DNode out;
    if (old >= kMat) out = load_node(A.nodes, old);
    else
        for (uint32_t& x : out.c) x = old;
    bool changed = false;
    const uint32_t ce = A.cend[i];
    for (uint32_t j = A.cbeg[i]; j < ce; j++) {
        const uint32_t id = key_octant(A.keys[j]), x = A.result(l - 1, j);
#pragma unroll
        for (uint32_t c = 0; c < 8; c++)
            if (c == id && out.c[c] != x) {
                out.c[c] = x;
                changed = true;
            }
    }
    uint32_t r = old, cand = 0;
    if (changed) { // Interner::intern: collapse, else the store's node, else new
        bool uniform = out.c[0] < kMat;
        for (int c = 1; c < 8; c++) uniform = uniform && out.c[c] == out.c[0];
        if (uniform) r = out.c[0];
        else {
            r = index_find(A.nodes, A.index, A.index_mask, out);
            if (r == kEmptySlot) {
                cand = 1;
                store_node(A.ckey, i, out);
                A.rep->fresh[l] = 1u;
            }
        }
    }
    A.res[i] = r;
    A.cand[i] = cand;
}

// Equal new nodes of level l: the first in Morton order is kept.
__global__ void __launch_bounds__(64) k_top_unique(TopArgs A, uint32_t l, uint32_t begin, uint32_t end)
{
    if (!A.rep->fresh[l]) return;
    const uint32_t i = begin + blockIdx.x * 64u + threadIdx.x;
    if (i >= end || !A.cand[i]) return;
    const uint64_t tmask = (A.tab_off[l + 1] - A.tab_off[l]) - 1;
    uint32_t* const tab = A.table + A.tab_off[l];
    const DNode k = load_node(A.ckey, i);
    for (uint64_t s = hash_node(k) & tmask;; s = (s + 1) & tmask) {
        const uint32_t cur = atomicCAS(&tab[s], kEmptySlot, i);
        if (cur == kEmptySlot || node_eq(load_node(A.ckey, cur), k)) {
            if (cur != kEmptySlot) atomicMin(&tab[s], i);
            A.cslot[i] = s;
            break;
        }
    }
}

// The kept nodes of level l appended in order: one workgroup, a scan over the level in chunks of its size
// (each wave ranks its lanes by ballot, then adds the counts of the waves before it).
__global__ void __launch_bounds__(kTopBlock) k_top_append(TopArgs A, uint32_t l, uint32_t begin, uint32_t end)
{
    if (!A.rep->fresh[l]) return;
    __shared__ uint32_t wave_kept[kTopBlock / 64];
    const uint32_t t = threadIdx.x, T = blockDim.x, lane = t & 63u, w = t >> 6;
    const uint32_t* const tab = A.table + A.tab_off[l];
    uint32_t base = A.rep->count;
    for (uint32_t c0 = begin; c0 < end; c0 += T) {
        const uint32_t i = c0 + t;
        uint32_t first = kEmptySlot;
        if (i < end && A.cand[i]) A.crep[i] = first = tab[A.cslot[i]];
        const bool keep = first == i;
        const uint64_t bal = __ballot(keep);
        if (lane == 0) wave_kept[w] = uint32_t(__popcll(bal));
        __syncthreads();
        uint32_t before = 0, all = 0;
        for (uint32_t v = 0; v < T / 64; v++) {
            before += v < w ? wave_kept[v] : 0u;
            all += wave_kept[v];
        }
        if (keep) A.res[i] = base + before + uint32_t(__popcll(bal & ((1ull << lane) - 1ull)));
        base += all;
        __syncthreads();
    }
    if (t == 0) A.rep->count = base;
}

// The kept nodes into the store and its index; the others take the index of theirs.
__global__ void __launch_bounds__(64) k_top_write(TopArgs A, uint32_t l, uint32_t begin, uint32_t end)
{
    if (!A.rep->fresh[l]) return;
    const uint32_t i = begin + blockIdx.x * 64u + threadIdx.x;
    if (i >= end || !A.cand[i]) return;
    if (A.crep[i] == i) store_node(A.nodes, A.res[i], load_node(A.ckey, i));
    else A.res[i] = A.res[A.crep[i]];
}
__global__ void __launch_bounds__(64) k_top_index(TopArgs A, uint32_t l, uint32_t begin, uint32_t end)
{
    if (!A.rep->fresh[l]) return;
    const uint32_t i = begin + blockIdx.x * 64u + threadIdx.x;
    if (i < end && A.cand[i] && A.crep[i] == i) index_insert(A.nodes, A.index, A.index_mask, A.res[i], load_node(A.ckey, i));
}

// The small levels; `begun`: k_top_begin and the large levels' launches came before.
__global__ void __launch_bounds__(kTopBlock) k_top_small(TopArgs A, uint32_t begun)
{
    __shared__ SmallTop small;
    const uint32_t t = threadIdx.x;
    top_stage(A, small, t, blockDim.x);
    if (begun) {
        const uint32_t b = small.off[small.first], n = small.off[A.levels + 1] - b;
        for (uint32_t i = t; i < n; i += blockDim.x) small.old[i] = A.old[b + i];
        __syncthreads();
    } else if (t < 64) top_small_down(A, small, t);
    if (t < 64) top_small_up(A, small, begun ? A.rep->count : A.count, t);
}

// findSubDAG (raytracing.cpp:43-87) of every root child, as cqx::find_subdags, one thread each, with
// the packed walk's pads (pad0 the node's packed word, pad1 the mask of the occupied SubDAGs). Each
// level is one 32-byte read of the node: 27 us on one thread with a read per child.
__global__ void __launch_bounds__(64) k_find_subdags(const uint32_t* __restrict__ nodes, uint32_t root,
                                                     cqx_subdag* __restrict__ out, EditReport* __restrict__ rep)
{
    if (root == kEmptySlot) root = rep->root; // the one k_top_small left there
    const uint32_t c = threadIdx.x;
    bool deep = false;
    cqx_subdag s{};
    if (c < 8) {
        int height = 32;
        uint32_t lower[3] = { 0x80000000u, 0x80000000u, 0x80000000u };
        uint32_t only = c, node = 0, count = 1;
        uint32_t next = root < kMat ? root : nodes[uint64_t(root) * 8 + only];
        while (count == 1 && !deep) {
            if (height == 0) {
                deep = true;
                break;
            }
            height--;
            node = next;
            for (int a = 0; a < 3; a++) lower[a] ^= ((only >> a) & 1u) << height;
            const DNode n = load_node(nodes, node); // a material node's children are itself
            count = 0;
#pragma unroll
            for (uint32_t i = 0; i < 8; i++) {
                if (n.c[i] > 0) {
                    next = n.c[i];
                    count++;
                    only = i;
                }
            }
        }
        s.lower[0] = int32_t(lower[0]);
        s.lower[1] = int32_t(lower[1]);
        s.lower[2] = int32_t(lower[2]);
        s.height = height;
        s.node = node;
        s.pad0 = cqxd::pack_child(nodes, kEmptySlot, node); // a node of the store: reached from its root
    }
    const uint64_t occupied = __ballot(c < 8 && s.node > 0), failed = __ballot(deep);
    s.pad1 = uint32_t(occupied);
    if (c == 0) rep->deep = failed ? 1u : 0u;
    if (c < 8 && !failed) out[c] = rep->sub[c] = s;
}

uint32_t grid_for(uint64_t n, const cqx_ctx* ctx, uint32_t block)
{
    const uint64_t want = (n + block - 1) / block;
    return uint32_t(std::max<uint64_t>(1, std::min<uint64_t>(want, uint64_t(ctx->cu_count) * 16)));
}

uint64_t pow2_at_least(uint64_t x)
{
    uint64_t p = 1;
    while (p < x) p <<= 1;
    return p;
}

} // namespace

namespace cqx {

// Device buffers of a volume's edits, kept between calls (grown as needed).
struct DeviceEdits {
    uint32_t* index = nullptr; // index over the store
    uint64_t index_cap = 0;
    uint64_t indexed = 0; // store nodes [256, indexed) are in the index
    struct Buf {
        void* p = nullptr;
        size_t bytes = 0;
    };
    Buf bufs[40];
    struct Staged {
        Buf dev, host; // host: pinned memory
    };
    Staged staged[2]; // the plans of the regions and of the levels above them (Stage)
    Buf report;       // device: EditReport
    std::vector<uint32_t> roots{ 0 }; // history (checkpoint / undo / redo), as the host volume's
    size_t current = 0;
};

// The index names nodes by what they held: with one of them replaced or cut off it is made anew by the
// next edit, which would otherwise take a node past the store's end for one of its own.
void forget_nodes(DeviceEdits* e, uint64_t first)
{
    if (!e || first >= e->indexed) return;
    release(e->index);
    e->index = nullptr;
    e->index_cap = e->indexed = 0;
}

void destroy_device_edits(DeviceEdits* e)
{
    if (!e) return;
    release(e->index);
    for (auto& b : e->bufs) release(b.p);
    for (auto& st : e->staged) {
        release(st.dev.p);
        if (st.host.p) (void)hipHostFree(st.host.p);
    }
    release(e->report.p);
    delete e;
}

} // namespace cqx

namespace {

// Buffer slots of DeviceEdits::bufs.
enum : int {
    kBufRun, kBufPoolOff, kBufCap, kBufCounts, kBufResults, kBufOverflow, kBufPool, kBufTable, kBufOff, kBufSrc, kBufRegion,
    kBufLevel, kBufKey, kBufSlotOf, kBufRep, kBufMergeTable, kBufFin, kBufRes, kBufCand, kBufCkey, kBufTopTable,
    kBufCslot, kBufScanSums, kBufOld
};

// Buffer `slot` of the volume's edit state with at least `bytes` (contents not kept when grown).
template <typename T>
cqx_status buf(cqx::DeviceEdits* E, int slot, size_t count, T** out)
{
    const size_t bytes = std::max<size_t>(256, count * sizeof(T));
    auto& b = E->bufs[slot];
    if (b.bytes < bytes) {
        release(b.p);
        b.p = nullptr;
        b.bytes = 0;
        if (hipMalloc(&b.p, bytes) != hipSuccess) return fail(CQX_ERR_OOM, "edit buffer of %zu bytes failed", bytes);
        b.bytes = bytes;
    }
    *out = static_cast<T*>(b.p);
    return CQX_OK;
}

// Exclusive prefix sums of v[0, n) in place and their total in *total, on the null stream.
cqx_status scan_u64(cqx_ctx* ctx, cqx::DeviceEdits* E, uint64_t* v, uint64_t n, uint64_t* total);

template <typename T>
cqx_status upload(cqx::DeviceEdits* E, int slot, const std::vector<T>& v, T** out)
{
    cqx_status st = buf(E, slot, v.size(), out);
    if (st != CQX_OK) return st;
    if (!v.empty()) HIP_TRY(hipMemcpy(*out, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return CQX_OK;
}

// A plan on its way to the device: its arrays put next to each other in pinned memory, and copied in
// one piece (a copy each was 12 us of the host's time, 16 of them a call).
struct Stage {
    size_t used = 0;
    char* host = nullptr;
    char* dev = nullptr;
    std::vector<char> plain; // where pinned memory cannot be had

    cqx_status reserve(cqx::DeviceEdits::Staged& s, size_t bytes)
    {
        if (s.dev.bytes < bytes) {
            const size_t want = std::max(bytes, s.dev.bytes + s.dev.bytes / 2);
            release(s.dev.p);
            if (s.host.p) (void)hipHostFree(s.host.p);
            s = {};
            if (hipMalloc(&s.dev.p, want) != hipSuccess) {
                s.dev.p = nullptr;
                return fail(CQX_ERR_OOM, "edit buffer of %zu bytes failed", want);
            }
            s.dev.bytes = want;
            if (hipHostMalloc(&s.host.p, want, hipHostMallocDefault) != hipSuccess) {
                s.host.p = nullptr;
                (void)hipGetLastError();
            }
        }
        if (!s.host.p) plain.resize(bytes);
        host = s.host.p ? static_cast<char*>(s.host.p) : plain.data();
        dev = static_cast<char*>(s.dev.p);
        return CQX_OK;
    }
    static size_t room(size_t bytes) { return (bytes + 255) / 256 * 256; }
    // Space for `count` values: the host's in *h, the device address they will have returned.
    template <typename T>
    T* put(size_t count, T** h)
    {
        *h = reinterpret_cast<T*>(host + used);
        T* const d = reinterpret_cast<T*>(dev + used);
        used += room(count * sizeof(T));
        return d;
    }
    template <typename T>
    T* put(const std::vector<T>& v)
    {
        T* h = nullptr;
        T* const d = put(v.size(), &h);
        if (!v.empty()) std::memcpy(h, v.data(), v.size() * sizeof(T));
        return d;
    }
    // Queues the copy of what was put.
    cqx_status send() const
    {
        if (plain.empty()) HIP_TRY(hipMemcpyAsync(dev, host, used, hipMemcpyHostToDevice, nullptr));
        else HIP_TRY(hipMemcpy(dev, host, used, hipMemcpyHostToDevice));
        return CQX_OK;
    }
};

cqx_status report_buffer(cqx::DeviceEdits* E, EditReport** out)
{
    auto& b = E->report;
    if (!b.p) {
        if (hipMalloc(&b.p, sizeof(EditReport)) != hipSuccess) {
            b.p = nullptr;
            return fail(CQX_ERR_OOM, "edit buffer of %zu bytes failed", sizeof(EditReport));
        }
        b.bytes = sizeof(EditReport);
    }
    *out = static_cast<EditReport*>(b.p);
    return CQX_OK;
}

cqx_status scan_u64(cqx_ctx*, cqx::DeviceEdits* E, uint64_t* v, uint64_t n, uint64_t* total)
{
    const uint64_t tiles = (n + kScanTile - 1) / kScanTile;
    if (tiles <= 4) { // a few values per thread: one launch instead of three
        hipLaunchKernelGGL(k_scan_u64, dim3(1), dim3(1024), 0, 0, v, n, total);
    } else {
        if (tiles > 0x7fffffffull) return fail(CQX_ERR_LIMIT, "scan of %llu values", (unsigned long long)n);
        uint64_t* sums = nullptr;
        cqx_status st = buf(E, kBufScanSums, tiles, &sums);
        if (st != CQX_OK) return st;
        hipLaunchKernelGGL(k_scan_tile_sums, dim3(uint32_t(tiles)), dim3(kScanBlock), 0, 0, v, n, sums);
        hipLaunchKernelGGL(k_scan_u64, dim3(1), dim3(1024), 0, 0, sums, tiles, total);
        hipLaunchKernelGGL(k_scan_tiles, dim3(uint32_t(tiles)), dim3(kScanBlock), 0, 0, v, n, sums);
    }
    HIP_TRY(hipGetLastError());
    return CQX_OK;
}

// The index covers every store node (grown to keep its load at most a half).
cqx_status ensure_index(cqx_ctx* ctx, cqx_dvolume* vol, uint64_t will_hold)
{
    cqx::DeviceEdits* E = vol->edits;
    if (2 * will_hold > E->index_cap) {
        const uint64_t cap = pow2_at_least(std::max<uint64_t>(1024, 2 * will_hold + will_hold / 2));
        release(E->index);
        E->index = nullptr;
        E->index_cap = 0;
        E->indexed = 0;
        if (hipMalloc(&E->index, cap * 4) != hipSuccess)
            return fail(CQX_ERR_OOM, "edit index of %llu slots failed", (unsigned long long)cap);
        E->index_cap = cap;
        hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(cap, ctx, 256)), dim3(256), 0, 0, E->index, cap, kEmptySlot);
        E->indexed = kMat;
    }
    if (vol->node_count > E->indexed) {
        hipLaunchKernelGGL(k_index_insert, dim3(grid_for(vol->node_count - E->indexed, ctx, 256)), dim3(256), 0, 0,
                           vol->nodes, E->indexed, vol->node_count, E->index, E->index_cap - 1);
        E->indexed = vol->node_count;
    }
    HIP_TRY(hipGetLastError());
    return CQX_OK;
}

// The device store holds at least `count` nodes (grown by copying; pointers change).
cqx_status ensure_store(cqx_ctx* ctx, cqx_dvolume* vol, uint64_t count)
{
    if (count <= vol->capacity) return CQX_OK;
    const uint64_t cap = std::max<uint64_t>(count, vol->capacity + vol->capacity / 2);
    uint32_t* p = nullptr;
    if (hipMalloc(&p, size_t(cap) * 32) != hipSuccess) return fail(CQX_ERR_OOM, "device store growth failed");
    if (hipMemcpy(p, vol->nodes, size_t(vol->node_count) * 32, hipMemcpyDeviceToDevice) != hipSuccess) {
        release(p);
        return fail(CQX_ERR_HIP, "device store copy failed");
    }
    HIP_TRY(hipDeviceSynchronize());
    release(vol->nodes);
    vol->nodes = p;
    vol->capacity = cap;
    if (ctx->pt_plan) { // its captured graph holds the old pointer
        cqx::destroy_pt_plan(ctx->pt_plan);
        ctx->pt_plan = nullptr;
    }
    return CQX_OK;
}

// The volume's root and SubDAGs from the report that k_find_subdags left; nodes from first_new on are new.
cqx_status set_root(cqx_ctx* ctx, cqx_dvolume* vol, uint32_t root, uint64_t first_new, EditReport& rep)
{
    if (rep.deep) return fail(CQX_ERR_INVALID_DAG, "single-child chain deeper than the tree");
    int max_height = 0;
    for (cqx_subdag& s : rep.sub) {
        if (s.node > 0) max_height = std::max(max_height, int(s.height));
        s.pad0 = s.pad1 = 0; // the packed walk's, on the device copy only
    }
    if (ctx->pt_plan && max_height != vol->max_height) { // its graph holds the stack size
        cqx::destroy_pt_plan(ctx->pt_plan);
        ctx->pt_plan = nullptr;
    }
    vol->root = root;
    std::memcpy(vol->hsub, rep.sub, sizeof(rep.sub));
    vol->max_height = max_height;
    return cqx::refresh_packed(ctx, vol, first_new);
}

// Makes `root`, a node of the store, the volume's root.
cqx_status switch_root(cqx_ctx* ctx, cqx_dvolume* vol, uint32_t root)
{
    EditReport* d_rep = nullptr;
    const cqx_status st = report_buffer(vol->edits, &d_rep);
    if (st != CQX_OK) return st;
    HIP_TRY(hipDeviceSynchronize()); // launches in flight may read the SubDAGs
    hipLaunchKernelGGL(k_find_subdags, dim3(1), dim3(64), 0, 0, vol->nodes, root, vol->sub, d_rep);
    HIP_TRY(hipGetLastError());
    EditReport rep;
    HIP_TRY(hipMemcpy(&rep, d_rep, sizeof(rep), hipMemcpyDeviceToHost));
    return set_root(ctx, vol, root, vol->node_count, rep);
}

cqx_status check_args(cqx_ctx* ctx, cqx_dvolume* vol)
{
    if (!ctx || !vol) return fail(CQX_ERR_INVALID_ARG, "null argument");
    HIP_TRY(hipSetDevice(ctx->device));
    if (!vol->edits) {
        vol->edits = new (std::nothrow) cqx::DeviceEdits;
        if (!vol->edits) return fail(CQX_ERR_OOM, "out of host memory");
        vol->edits->roots[0] = vol->root;
    }
    return CQX_OK;
}

} // namespace

extern "C" {

cqx_status cqx_volume_edit_spheres(cqx_ctx* ctx, cqx_dvolume* vol, const cqx_sphere_edit* edits, uint64_t n,
                                   uint64_t* first_new)
{
    const cqx::TraceRange range("cqx_volume_edit_spheres");
    cqx_status st = check_args(ctx, vol);
    if (st != CQX_OK) return st;
    if (n && !edits) return fail(CQX_ERR_INVALID_ARG, "null edits");
    if (first_new) *first_new = vol->node_count;
    if (n == 0) return CQX_OK;
    for (uint64_t i = 0; i < n; i++) {
        if (edits[i].material >= kMat) return fail(CQX_ERR_INVALID_ARG, "edit %llu: material >= 256", (unsigned long long)i);
        if (!(edits[i].radius >= 0.0f)) return fail(CQX_ERR_INVALID_ARG, "edit %llu: bad radius", (unsigned long long)i);
    }
    const int hs = n >= 16 ? cqx::region_height(edits, n) : -1;
    if (hs < 0)
        return fail(CQX_ERR_LIMIT, "on-device edits take batches of at least 16 spheres, each within 2^23 voxels of the "
                                   "origin and with radius < 2^20 / 2; apply this batch with cqx_hv_edit_spheres");
    using clock = std::chrono::steady_clock;
    const auto ms_since = [](clock::time_point t) {
        return std::chrono::duration<double, std::milli>(clock::now() - t).count();
    };
    clock::time_point t_phase = clock::now();
    double ms[4] = { 0, 0, 0, 0 }; // plan, regions, merge, levels above
    int attempts = 0;
    cqx::EditPlan plan;
    try {
        cqx::plan_regions(edits, n, hs, plan);
    } catch (const std::bad_alloc&) {
        return fail(CQX_ERR_OOM, "out of host memory while planning edits");
    }
    if (vol->root >= vol->node_count) // an undo past an update that cut the store
        return fail(CQX_ERR_INVALID_DAG, "root %u is not in the store of %llu nodes", vol->root,
                    (unsigned long long)vol->node_count);
    cqx::DeviceEdits* E = vol->edits;
    HIP_TRY(hipDeviceSynchronize()); // launches in flight may read the store or the index
    const uint64_t base = vol->node_count;
    const uint32_t nr = uint32_t(plan.keys.size());
    st = ensure_index(ctx, vol, base);
    if (st != CQX_OK) return st;
    EditReport* d_rep = nullptr;
    if ((st = report_buffer(E, &d_rep)) != CQX_OK) return st;

    // ---- regions ----
    Stage stage;
    if ((st = stage.reserve(E->staged[0], Stage::room(n * sizeof(cqx_sphere_edit)) + Stage::room(nr * sizeof(DRegionKey)) +
                                              Stage::room((size_t(nr) + 1) * 8) + Stage::room(plan.edit_ids.size() * 4) +
                                              2 * Stage::room(size_t(nr) * 4) + Stage::room(size_t(nr) * 8))) != CQX_OK)
        return st;
    cqx_sphere_edit* h_edits;
    DRegionKey* h_keys;
    uint32_t *h_run, *h_cap;
    uint64_t* h_pool_off;
    const cqx_sphere_edit* const d_edits = stage.put(n, &h_edits);
    const DRegionKey* const d_keys = stage.put(nr, &h_keys);
    const uint64_t* const d_first = stage.put(plan.first);
    const uint32_t* const d_edit_ids = stage.put(plan.edit_ids);
    uint32_t* d_run = stage.put(nr, &h_run);
    uint32_t* d_cap = stage.put(nr, &h_cap);
    uint64_t* d_pool_off = stage.put(nr, &h_pool_off);
    std::memcpy(h_edits, edits, n * sizeof(cqx_sphere_edit));
    for (uint32_t r = 0; r < nr; r++) h_keys[r] = { plan.keys[r].x, plan.keys[r].y, plan.keys[r].z };
    std::vector<uint32_t> cap(nr), run(nr);
    std::vector<uint64_t> pool_off(nr);
    std::vector<float> work(nr);
    uint64_t pool_total = 0;
    // First slice of each region's list: per sphere about twice the voxels of its largest cross
    // section the region can hold (a sphere changes nodes along its surface, a few per voxel
    // column), so that few regions have to run again.
    // CQX_EDIT_FIRST_SLICE=<nodes> fixes the first slices instead (the tests use it to make
    // regions outgrow them).
    const char* fixed_slice = std::getenv("CQX_EDIT_FIRST_SLICE");
    const double fixed = fixed_slice ? std::atof(fixed_slice) : 0.0;
    const double side = std::ldexp(1.0, hs);
    float most = 0.0f;
    for (uint32_t r = 0; r < nr; r++) {
        double est = 64.0;
        for (uint64_t j = plan.first[r]; j < plan.first[r + 1]; j++) {
            const double rad = edits[plan.edit_ids[j]].radius;
            est += 2.0 * std::min(3.14159265 * rad * rad, side * side) + 16.0;
        }
        work[r] = float(est);
        most = std::max(most, work[r]);
        if (fixed >= 1.0) est = fixed;
        cap[r] = uint32_t(pow2_at_least(uint64_t(std::min(est, 1048576.0))));
        pool_off[r] = pool_total;
        pool_total += cap[r];
    }
    // the wave that takes the heaviest region (most sphere surface) early finishes early: the
    // phase then lasts about as long as its heaviest region or its average load per wave. Sorted
    // into 1024 classes of work: the order within one does not matter.
    {
        uint32_t at[1025] = {};
        const auto cls = [&](uint32_t r) { return 1023u - uint32_t(std::min(1023.0f, work[r] * (1023.0f / most))); };
        for (uint32_t r = 0; r < nr; r++) at[cls(r) + 1]++;
        for (int k = 0; k < 1024; k++) at[k + 1] += at[k];
        for (uint32_t r = 0; r < nr; r++) run[at[cls(r)]++] = r;
    }
    std::memcpy(h_run, run.data(), nr * 4);
    std::memcpy(h_cap, cap.data(), nr * 4);
    std::memcpy(h_pool_off, pool_off.data(), nr * 8);
    uint32_t *d_counts, *d_results, *d_overflow, *d_pool, *d_table;
    uint64_t* d_off;
    if ((st = stage.send()) != CQX_OK || (st = buf(E, kBufCounts, nr, &d_counts)) != CQX_OK ||
        (st = buf(E, kBufResults, nr, &d_results)) != CQX_OK || (st = buf(E, kBufOverflow, nr, &d_overflow)) != CQX_OK ||
        (st = buf(E, kBufOff, nr + 1, &d_off)) != CQX_OK)
        return st;
    ms[0] = ms_since(t_phase);
    t_phase = clock::now();
    // A region whose list outgrows its slice runs again with a slice 8 times larger, placed after
    // the others; the pool keeps what the finished regions listed.
    EditReport rep{};
    for (int attempt = 0; !run.empty(); attempt++) {
        if (attempt > 6) return fail(CQX_ERR_LIMIT, "an edit region listed more nodes than the retries allow");
        if (base + uint64_t(*std::max_element(cap.begin(), cap.end())) >= 0xfffffffeull)
            return fail(CQX_ERR_LIMIT, "store too large for on-device edits");
        // pool and tables: grown keeping their contents
        auto& pb = E->bufs[kBufPool];
        auto& tb = E->bufs[kBufTable];
        const size_t pool_bytes = size_t(pool_total) * 32, table_bytes = size_t(pool_total) * 8;
        for (auto* bb : { &pb, &tb }) {
            const size_t need = bb == &pb ? pool_bytes : table_bytes;
            if (bb->bytes < need) {
                void* q = nullptr;
                const size_t want = std::max(need, bb->bytes + bb->bytes / 2);
                if (hipMalloc(&q, want) != hipSuccess) return fail(CQX_ERR_OOM, "edit pool of %zu bytes failed", want);
                if (attempt > 0 && bb->p) HIP_TRY(hipMemcpy(q, bb->p, bb->bytes, hipMemcpyDeviceToDevice));
                release(bb->p);
                bb->p = q;
                bb->bytes = want;
            }
        }
        d_pool = static_cast<uint32_t*>(pb.p);
        d_table = static_cast<uint32_t*>(tb.p);
        if (attempt > 0 && ((st = upload(E, kBufRun, run, &d_run)) != CQX_OK ||
                            (st = upload(E, kBufPoolOff, pool_off, &d_pool_off)) != CQX_OK ||
                            (st = upload(E, kBufCap, cap, &d_cap)) != CQX_OK))
            return st;
        hipLaunchKernelGGL(k_edit_begin, dim3(1), dim3(64), 0, 0, d_rep);
        RegionArgs A{ vol->nodes, E->index, E->index_cap - 1, vol->root, hs, uint32_t(base), d_edits, d_keys, d_first,
                      d_edit_ids, d_run, uint32_t(run.size()), &d_rep->next_run, d_pool_off, d_cap, d_pool, d_table, d_counts,
                      d_results, d_overflow };
        const uint32_t waves = uint32_t(std::min<uint64_t>(run.size(), uint64_t(ctx->cu_count) * 32));
        hipLaunchKernelGGL(k_edit_regions, dim3(waves), dim3(64), sizeof(Frame) * size_t(std::max(hs - 3, 1)), 0, A);
        hipLaunchKernelGGL(k_region_counts, dim3(grid_for(nr, ctx, 256)), dim3(256), 0, 0, d_counts, d_overflow, d_off, nr,
                           d_rep);
        HIP_TRY(hipGetLastError());
        if ((st = scan_u64(ctx, E, d_off, uint64_t(nr), &d_rep->listed)) != CQX_OK) return st;
        if (attempt == 0) { // the levels above are planned while the regions run
            try {
                cqx::plan_levels(plan);
            } catch (const std::bad_alloc&) {
                return fail(CQX_ERR_OOM, "out of host memory while planning edits");
            }
        }
        HIP_TRY(hipMemcpy(&rep, d_rep, offsetof(EditReport, next_run), hipMemcpyDeviceToHost));
        std::vector<uint32_t> again;
        if (rep.outgrown) {
            std::vector<uint32_t> over(nr);
            HIP_TRY(hipMemcpy(over.data(), d_overflow, nr * 4, hipMemcpyDeviceToHost));
            for (uint32_t r : run)
                if (over[r]) {
                    again.push_back(r);
                    cap[r] *= 8;
                    pool_off[r] = pool_total;
                    pool_total += cap[r];
                }
            cqx::log_debug("device edits: %zu of %zu regions outgrew their node lists; running them again",
                           again.size(), run.size());
        }
        run.swap(again);
        attempts = attempt + 1;
    }
    const uint64_t total = rep.listed;
    ms[1] = ms_since(t_phase);
    t_phase = clock::now();

    // ---- merge ----
    if (base + total >= 0xfffffffeull) return fail(CQX_ERR_LIMIT, "store too large for on-device edits");
    uint64_t kept_total = 0, *d_fin = nullptr;
    MergeArgs M{};
    if (total) {
        uint64_t* d_slot_of;
        uint32_t *d_src, *d_region, *d_key, *d_rep_of, *d_mtable;
        uint8_t* d_level;
        const uint64_t mcap = pow2_at_least(std::max<uint64_t>(1024, 2 * total));
        if ((st = buf(E, kBufSrc, total, &d_src)) != CQX_OK || (st = buf(E, kBufRegion, total, &d_region)) != CQX_OK ||
            (st = buf(E, kBufLevel, total, &d_level)) != CQX_OK || (st = buf(E, kBufKey, total * 8, &d_key)) != CQX_OK ||
            (st = buf(E, kBufSlotOf, total, &d_slot_of)) != CQX_OK || (st = buf(E, kBufRep, total, &d_rep_of)) != CQX_OK ||
            (st = buf(E, kBufMergeTable, mcap, &d_mtable)) != CQX_OK || (st = buf(E, kBufFin, total + 1, &d_fin)) != CQX_OK)
            return st;
        M = MergeArgs{ uint32_t(base), nr, d_pool_off, d_pool, d_counts, d_off, total, d_src, d_region, d_level, d_key,
                       d_slot_of, d_rep_of, d_mtable, mcap - 1 };
        hipLaunchKernelGGL(k_merge_flatten, dim3(std::min<uint32_t>(nr, uint32_t(ctx->cu_count) * 32)), dim3(64), 0, 0, M);
        hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(mcap, ctx, 256)), dim3(256), 0, 0, d_mtable, mcap, kEmptySlot);
        const uint32_t g = grid_for(total, ctx, 256);
        for (uint32_t lv = 0; lv < uint32_t(hs); lv++) { // a node of height h has level h - 1 at most
            hipLaunchKernelGGL(k_merge_keys, dim3(g), dim3(256), 0, 0, M, lv);
            hipLaunchKernelGGL(k_merge_insert, dim3(g), dim3(256), 0, 0, M, lv);
            hipLaunchKernelGGL(k_merge_rep, dim3(g), dim3(256), 0, 0, M, lv);
        }
        hipLaunchKernelGGL(k_merge_kept, dim3(g), dim3(256), 0, 0, M, d_fin);
        if ((st = scan_u64(ctx, E, d_fin, total, &d_rep->kept)) != CQX_OK) return st;
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipMemcpy(&kept_total, &d_rep->kept, 8, hipMemcpyDeviceToHost));
    }
    // ---- the levels above the regions: schedule, capacity ----
    DRegionKey* h_tkeys;
    uint32_t *h_lvl_off, *h_cbeg, *h_cend;
    uint64_t* h_tab_off;
    uint64_t ntop = 0;
    const uint32_t levels = uint32_t(32 - hs);
    for (uint32_t l = 0; l <= levels; l++) ntop += plan.level_keys[l].size();
    Stage above;
    if ((st = above.reserve(E->staged[1], Stage::room((levels + 2) * 4) + Stage::room((levels + 2) * 8) +
                                              Stage::room(ntop * sizeof(DRegionKey)) + 2 * Stage::room(ntop * 4) +
                                              Stage::room(size_t(nr) * 4))) != CQX_OK)
        return st;
    const uint32_t* const d_lvl_off = above.put(levels + 2, &h_lvl_off);
    const uint64_t* const d_tab_off = above.put(levels + 2, &h_tab_off);
    const DRegionKey* const d_tkeys = above.put(ntop, &h_tkeys);
    const uint32_t* const d_cbeg = above.put(ntop, &h_cbeg);
    const uint32_t* const d_cend = above.put(ntop, &h_cend);
    const uint32_t* const d_morton = above.put(plan.morton_regions);
    uint32_t at = 0;
    h_tab_off[0] = 0;
    for (uint32_t l = 0; l <= levels; l++) {
        h_lvl_off[l] = at;
        const auto& lk = plan.level_keys[l];
        for (size_t i = 0; i < lk.size(); i++, at++) {
            h_tkeys[at] = { lk[i].x, lk[i].y, lk[i].z };
            h_cbeg[at] = l == 0 ? 0 : h_lvl_off[l - 1] + plan.level_children[l][i];
            h_cend[at] = l == 0 ? 0 : h_lvl_off[l - 1] + plan.level_children[l][i + 1];
        }
        h_tab_off[l + 1] = h_tab_off[l] + (l == 0 ? 0 : pow2_at_least(std::max<uint64_t>(2, 2 * lk.size())));
    }
    h_lvl_off[levels + 1] = at;
    const uint64_t top_slots = h_tab_off[levels + 1];
    if ((st = above.send()) != CQX_OK) return st;
    st = ensure_store(ctx, vol, base + kept_total + ntop);
    if (st != CQX_OK) return st;
    st = ensure_index(ctx, vol, base + kept_total + ntop);
    if (st != CQX_OK) return st;
    if (total) {
        hipLaunchKernelGGL(k_merge_write, dim3(grid_for(std::max<uint64_t>(total, nr), ctx, 256)), dim3(256), 0, 0, M,
                           d_fin, vol->nodes, d_results);
        hipLaunchKernelGGL(k_index_insert, dim3(grid_for(std::max<uint64_t>(kept_total, 1), ctx, 256)), dim3(256), 0, 0,
                           vol->nodes, base, base + kept_total, E->index, E->index_cap - 1);
        HIP_TRY(hipGetLastError());
    }
    E->indexed = base + kept_total;
    ms[2] = ms_since(t_phase);
    t_phase = clock::now();

    // ---- the levels above the regions, and the new root's SubDAGs ----
    uint32_t *d_res, *d_cand, *d_ckey, *d_ttable, *d_old;
    uint64_t* d_cslot;
    if ((st = buf(E, kBufRes, ntop, &d_res)) != CQX_OK || (st = buf(E, kBufCand, 2 * ntop, &d_cand)) != CQX_OK ||
        (st = buf(E, kBufCkey, ntop * 8, &d_ckey)) != CQX_OK || (st = buf(E, kBufTopTable, top_slots, &d_ttable)) != CQX_OK ||
        (st = buf(E, kBufCslot, ntop, &d_cslot)) != CQX_OK || (st = buf(E, kBufOld, ntop, &d_old)) != CQX_OK)
        return st;
    hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(top_slots, ctx, 256)), dim3(256), 0, 0, d_ttable, top_slots, kEmptySlot);
    TopArgs T{ vol->nodes, E->index, E->index_cap - 1, vol->root, hs, levels, d_lvl_off, d_tkeys, d_cbeg, d_cend,
               d_morton, d_results, d_res, d_cand, d_ckey, d_cand + ntop, d_cslot, d_ttable, d_tab_off,
               uint32_t(base + kept_total), d_rep, d_old };
    uint32_t first_small = 1;
    while (h_lvl_off[first_small + 1] - h_lvl_off[first_small] > 64) first_small++;
    if (first_small > 1) {
        hipLaunchKernelGGL(k_top_begin, dim3(1), dim3(kTopBlock), 0, 0, T);
        for (uint32_t l = first_small - 1; l >= 2; l--) {
            const uint32_t lb = h_lvl_off[l], le = h_lvl_off[l + 1];
            hipLaunchKernelGGL(k_top_old, dim3((le - lb + 255) / 256), dim3(256), 0, 0, T, l, lb, le);
        }
        for (uint32_t l = 1; l < first_small; l++) {
            const uint32_t lb = h_lvl_off[l], le = h_lvl_off[l + 1];
            const dim3 waves((le - lb + 63) / 64);
            hipLaunchKernelGGL(k_top_build, waves, dim3(64), 0, 0, T, l, lb, le);
            hipLaunchKernelGGL(k_top_unique, waves, dim3(64), 0, 0, T, l, lb, le);
            hipLaunchKernelGGL(k_top_append, dim3(1), dim3(kTopBlock), 0, 0, T, l, lb, le);
            hipLaunchKernelGGL(k_top_write, waves, dim3(64), 0, 0, T, l, lb, le);
            hipLaunchKernelGGL(k_top_index, waves, dim3(64), 0, 0, T, l, lb, le);
        }
    }
    hipLaunchKernelGGL(k_top_small, dim3(1), dim3(kTopBlock), 0, 0, T, first_small > 1 ? 1u : 0u);
    hipLaunchKernelGGL(k_find_subdags, dim3(1), dim3(64), 0, 0, vol->nodes, kEmptySlot, vol->sub, d_rep);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpy(&rep, d_rep, sizeof(rep), hipMemcpyDeviceToHost));
    const uint64_t kOffset32Nodes = uint64_t(1) << 27; // the child-offset width the traversal uses
    if (ctx->pt_plan && (base <= kOffset32Nodes) != (uint64_t(rep.count) <= kOffset32Nodes)) {
        cqx::destroy_pt_plan(ctx->pt_plan); // its captured graph holds the old offset width
        ctx->pt_plan = nullptr;
    }
    vol->node_count = rep.count;
    E->indexed = rep.count;
    st = set_root(ctx, vol, rep.root, base, rep);
    if (st != CQX_OK) return st;
    ms[3] = ms_since(t_phase);
    cqx::log_debug("device edits: %llu spheres over %u regions of side 2^%d (%d runs); %llu listed, %llu appended, "
                   "%llu above; plan %.2f ms, regions %.2f ms, merge %.2f ms, levels above %.2f ms",
                   (unsigned long long)n, nr, hs, attempts, (unsigned long long)total, (unsigned long long)kept_total,
                   (unsigned long long)(rep.count - base - kept_total), ms[0], ms[1], ms[2], ms[3]);
    E->roots.resize(E->current + 1);
    E->roots[E->current] = vol->root;
    return CQX_OK;
}

cqx_status cqx_volume_checkpoint(cqx_ctx* ctx, cqx_dvolume* vol)
{
    cqx_status st = check_args(ctx, vol);
    if (st != CQX_OK) return st;
    cqx::DeviceEdits* E = vol->edits;
    E->roots.resize(E->current + 1);
    E->roots[E->current] = vol->root;
    E->roots.push_back(vol->root);
    E->current++;
    return CQX_OK;
}

cqx_status cqx_volume_undo(cqx_ctx* ctx, cqx_dvolume* vol)
{
    cqx_status st = check_args(ctx, vol);
    if (st != CQX_OK) return st;
    cqx::DeviceEdits* E = vol->edits;
    E->roots[E->current] = vol->root;
    if (E->current > 0) E->current--;
    return switch_root(ctx, vol, E->roots[E->current]);
}

cqx_status cqx_volume_redo(cqx_ctx* ctx, cqx_dvolume* vol)
{
    cqx_status st = check_args(ctx, vol);
    if (st != CQX_OK) return st;
    cqx::DeviceEdits* E = vol->edits;
    E->roots[E->current] = vol->root;
    if (E->current + 1 < E->roots.size()) E->current++;
    return switch_root(ctx, vol, E->roots[E->current]);
}

cqx_status cqx_volume_download(cqx_ctx* ctx, const cqx_dvolume* vol, uint64_t first, uint64_t count, uint32_t* nodes)
{
    if (!ctx || !vol || (count && !nodes)) return fail(CQX_ERR_INVALID_ARG, "null argument");
    if (first > vol->node_count || count > vol->node_count - first)
        return fail(CQX_ERR_INVALID_ARG, "nodes [%llu, %llu) outside the store of %llu", (unsigned long long)first,
                    (unsigned long long)(first + count), (unsigned long long)vol->node_count);
    HIP_TRY(hipSetDevice(ctx->device));
    if (count) HIP_TRY(hipMemcpy(nodes, vol->nodes + first * 8, size_t(count) * 32, hipMemcpyDeviceToHost));
    return CQX_OK;
}

} // extern "C"
