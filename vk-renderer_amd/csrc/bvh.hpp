// bvh.hpp - host-side BVH builder for the gfx950 traversal kernels.
//
// The reference has no acceleration structure: trace_ray scans every
// primitive linearly (Assets/Tracer.comp:374-431).  This BVH replaces that
// scan; the kernels recover the scan's exact order-dependent acceptance rule
// from the hits it reports (see trace_kernels.hip).
//
// Layout (all records 16-byte aligned for 128-bit loads):
//   Node (48 B): the bounds of BOTH children, as centre and half-extent per
//   axis, plus their refs, so one node fetch tests two boxes.  Centres are
//   floats, half-extents 16-bit floats rounded up (the kernels' mixed
//   multiply-add reads them as they are), so that [c - e, c + e] contains the
//   float box; no half-extent is below 2^-14.  m is the float 1.0 in the nodes
//   of the sphere subtree and 0 elsewhere; the traversal multiplies its
//   per-ray widening by it.  Three 128-bit loads instead of the four that
//   32-bit half-extents need: with several emitters the L1 takes close to an
//   access a cycle (each lane's load counts).  Two loads a node (16-bit centres
//   on the scene's grid) gained nothing more: their decoding costs ten VALU
//   instructions a step (100k-triangle soup 72.8 / 72.6 ms, heightfield +4%).
//   With a centre/extent box the slab test is t = (c - o) / d -+ e / |d|, and
//   a per-ray widening w of the box is one more term: (e + w) / |d|.
//   Triangles and spheres live in separate subtrees: when both exist, node 0
//   is a root whose child 0 is the triangle subtree and child 1 the sphere
//   subtree (an always-entered box), and the nodes from index sph_node0 on
//   belong to the sphere subtree.  The traversal widens the boxes of the
//   sphere subtree per ray (the reference's sphere test is imprecise far from
//   the sphere, see traverse.hpp).
//   ref: bit31 = leaf; for a leaf bit30 = sphere leaf, bits 27..29 = count-1,
//   bits 0..26 = first record; for an inner node 3 * the node index (its
//   offset in units of 16 bytes).
//   Triangle record (48 B): (v0, key) (e1, mat_index) (e2, 0) where
//   e1 = fl(v1 - v0), e2 = fl(v2 - v0) are exactly the edges the reference
//   computes (Tracer.comp:342-343) and key is the triangle's scan index.
//   Sphere record (16 B + 4 B key): (centre, r) and the sphere's scan index.
#pragma once

#include <cstddef>
#include <cstdint>
#include <cstring>
#include <vector>

namespace vkr {

constexpr uint32_t kRefLeaf = 0x80000000u;
constexpr uint32_t kRefSphere = 0x40000000u;
constexpr uint32_t kRefCountShift = 27;
constexpr uint32_t kRefFirstMask = (1u << 27) - 1u;
constexpr uint32_t kMaxLeaf = 8;
// Default leaf size cap: small leaves keep the lanes of a wave's leaf pass
// busy.  Scenes with several emitters are traced by the pooled kernel,
// mostly shadow rays: there single-primitive leaves run fastest (1080p /
// 100k-triangle soup: 113 ms against 122 ms with 2, 135 ms with 3).  With
// one emitter, 2 is best on the 2M-triangle heightfield (9.9 ms against
// 10.3 ms with 1).
constexpr uint32_t kDefaultLeaf = 2;
inline uint32_t default_leaf(uint32_t n_emitters) { return n_emitters >= 2u ? 1u : kDefaultLeaf; }
// Default depth cap: trees of at most 23 levels run the path kernel with a
// 24-entry stack (one entry holds the end marker), which keeps 5 waves of the
// pooled kernel resident per SIMD instead of 4.  The SAH split search respects
// the cap.
constexpr uint32_t kDefaultMaxDepth = 23;

struct alignas(16) BvhNode {
    float c0[3], c1x;         // child 0's centre, child 1's x
    float c1yz[2];
    uint32_t ref[2];
    uint16_t e[6];            // half-extents: child 0 x y z, child 1 x y z
    float m;
};
static_assert(sizeof(BvhNode) == 48, "node is 48 bytes");
inline uint32_t inner_ref(std::size_t index) { return 3u * (uint32_t)index; }

struct alignas(16) TriRecord {
    float v0[3]; uint32_t key;
    float e1[3]; uint32_t mat_index;
    float e2[3]; uint32_t pad;
};
static_assert(sizeof(TriRecord) == 48, "triangle record is 48 bytes");

// The least 16-bit float >= x, for x >= 0 (above 65504: infinity), but at
// least 2^-14, the smallest normal one.
#if defined(__HIP__)
__host__ __device__
#endif
inline uint16_t half_up(float x)
{
    if (!(x > 0x1p-14f)) return 0x0400u;
    if (x > 65504.0f) return 0x7C00u;
    uint32_t u;
    memcpy(&u, &x, sizeof u);
    return (uint16_t)(((u >> 13) - (112u << 10)) + ((u & 0x1FFFu) ? 1u : 0u));
}

struct BuildInput {
    const float* tri_v;       // n_tris * 12 floats: v0(3) pad v1(3) pad v2(3) pad (std430)
    const uint32_t* tri_mat;  // optional, stride 12 u32 (the v0 padding word)
    uint32_t n_tris = 0;
    const float* sph;         // n_spheres * 16 floats (std430 Sphere: P at 12, r at 15)
    uint32_t n_spheres = 0;
    uint32_t max_leaf = kDefaultLeaf;
    uint32_t max_depth = kDefaultMaxDepth;
    float traversal_cost = 0.0f;  // SAH cost of a node visit relative to one primitive test (0 = 3)
};

struct BuildOutput {
    std::vector<BvhNode> nodes;
    std::vector<TriRecord> tris;
    std::vector<float> sph;        // 4 floats per sphere record (centre, r)
    std::vector<uint32_t> sph_key; // scan index per sphere record
    uint32_t leaves = 0;
    uint32_t depth = 0;            // deepest leaf (root children are depth 1)
    uint32_t sph_node0 = 0xFFFFFFFFu;  // first node of the sphere subtree (none: all ones)
    float sph_c[3] = {0.0f, 0.0f, 0.0f};  // sphere centres lie within sph_r of sph_c
    float sph_r = 0.0f;
    float sph_rmin = 0.0f;         // least radius
    bool empty = true;
};

// The node above a device-built triangle subtree and a sphere subtree:
// child 0 the triangle box [lo, hi] (an empty box: never entered) with ref
// tri_ref, child 1 always entered with ref sph_ref.
BvhNode join_root(const float lo[3], const float hi[3], uint32_t tri_ref, uint32_t sph_ref);

// Moves every inner-node ref of nodes by off nodes (leaf refs are unchanged).
void offset_inner_refs(std::vector<BvhNode>& nodes, uint32_t off);

// Builds a binned-SAH BVH.  Leaves hold one primitive kind only and at most
// max_leaf primitives; no leaf is deeper than max_depth (splits fall back to
// balanced median splits near the cap), so a traversal stack of max_depth + 1
// entries (one holds the end marker) never overflows.
BuildOutput build_bvh(const BuildInput& in);

}  // namespace vkr
