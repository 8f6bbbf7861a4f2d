// Four-wide BVH used by the GPU traversal.
//
// It is derived on the host, at context creation, from the binary two-level
// BVH of the payload (the reference node format, noor/cuda/bvh.cuh:28-140):
// each wide node holds the boxes of up to four children, taken unchanged from
// the binary nodes they replace, so one 128-byte fetch tests four boxes and a
// ray needs about half the dependent node fetches of the binary traversal.
// Together with the conservative slab test this returns the same hits as the
// binary traversal (see box4_hit in dev_core.h).
//
// Child references (also the traversal stack entries), 32 bits:
//   bit 31      TLAS level: the world-space ray applies below this entry
//   bits 30-29  kind: 0 inner (wide node index), 1 triangle leaf,
//               2 instance (transform index), 3 area-light node (light index)
//   leaf:       bits 0-25 first triangle (leaf order), bits 26-28 count - 1
//   inner:      bits 0-27 index, bit 28 set in the top level's own nodes
//   others:     bits 0-28 index
//
// Flat meshes: a mesh placed by exactly one instance whose world-to-object
// matrix is the identity is traversed with the world-space ray.  Its nodes and
// leaves carry the TLAS bit, and the top level (`root`) refers to its root
// directly, so a ray neither visits an instance nor changes space; the instance
// of a hit is read from the triangle's record.  The
// identity's product with a ray gives back the same bits except for infinite
// and NaN components and the sign of a zero, which the direction's reciprocal
// turns into an infinity of the other sign and a hit at distance zero can keep:
// rays with a zero or infinite direction component or a -0, infinite or NaN
// origin component start at a second top level (`root_strict`) that enters flat
// meshes through their instance like any other, over the same nodes (a NaN
// direction component hits no triangle either way).  Without the instance visits and
// the ray rebuilds in both directions (about 140 instructions each, paid by the
// whole wave) the megakernel takes 3.4 instead of 4.1 ms for 512x512x4 samples of
// the Cornell box (all meshes flat), and k_extend 20.3 instead of 22.1, k_shadow
// 8.0 instead of 9.0 ms for the 1080p terrain film (the ground is flat, the 1,000
// spheres are not).
#ifndef NOOR_WIDE_BVH_H
#define NOOR_WIDE_BVH_H

#include <stdint.h>

namespace noor {

constexpr uint32_t REF_TLAS = 0x80000000u;
constexpr uint32_t REF_KIND_SHIFT = 29;
constexpr uint32_t REF_INNER = 0u, REF_LEAF = 1u, REF_INST = 2u, REF_LIGHT = 3u;
constexpr uint32_t REF_INDEX_MASK = 0x1FFFFFFFu;
constexpr uint32_t REF_TOP = 0x10000000u;        // of an inner reference
// (ref & REF_LEAVES_FLAT) != 0 for the references of the top level itself, 0
// for those of a flat mesh (whose leaves hold at most REF_FLAT_LEAF_MAX
// triangles, so that bit 28 of theirs is clear)
constexpr uint32_t REF_LEAVES_FLAT = 0x40000000u | REF_TOP;
constexpr uint32_t REF_FLAT_LEAF_MAX = 4u;
constexpr uint32_t REF_NODE_MASK = 0x0FFFFFFFu;  // index of an inner reference
constexpr uint32_t REF_LEAF_START_MASK = 0x03FFFFFFu;
constexpr uint32_t REF_LEAF_COUNT_SHIFT = 26;
constexpr uint32_t REF_LEAF_MAX = 8u;
constexpr uint32_t REF_EMPTY = 0xFFFFFFFFu;

// Host form of a wide node: SoA boxes of the four children (an empty slot has
// lo = +inf, hi = -inf), then their references.  The builder and the checks
// work on this form; the GPU reads the compressed QNode below.
struct alignas(128) WNode {
    float lo[3][4];
    float hi[3][4];
    uint32_t ref[4];
    uint32_t pad[4];
};
static_assert(sizeof(WNode) == 128, "WNode is one 128-byte line");

// Device form, 64 bytes: the four child boxes quantised to 8 bits per plane on
// a grid local to the node (as in Ylitie, Karras & Laine, "Efficient Incoherent
// Ray Traversal on GPUs Through Compressed Wide BVHs", HPG 2017).  On axis a a
// plane decodes to
//     org[a] + (float)q * |scale[a]|            (binary32, no contraction)
// with |scale[a]| a power of two.  The encoder rounds lower planes down and
// upper planes up and checks the decoded values, so every decoded box contains
// its child's exact box; with the conservative slab test the traversal
// therefore returns the same hits as over the exact boxes.  The children fill
// the slots from 0 on; slot 0 is never empty, and the signs of the scales say
// which others are: scale[2] negative for slot 1, scale[1] for slot 2, scale[0]
// for slot 3.  Slot c is byte c of each q word.
struct alignas(64) QNode {
    float org[3];
    float scale[3];
    uint32_t qlo[3];
    uint32_t qhi[3];
    uint32_t ref[4];
};
static_assert(sizeof(QNode) == 64, "QNode is 64 bytes");

}  // namespace noor

#include <string>
#include <vector>

#include "noor_hip.h"

namespace noor {

struct WideBvh {
    std::vector<WNode> nodes;         // exact boxes (host)
    std::vector<QNode> qnodes;        // the same nodes, compressed (uploaded)
    std::vector<uint32_t> inst_root;  // per transform: reference of its BLAS root
    std::vector<uint32_t> tri_inst;   // per triangle of a flat mesh: its instance (empty without flat meshes)
    uint32_t root = REF_EMPTY;
    uint32_t root_strict = REF_EMPTY;  // the top level for rays whose components the identity would change
    uint32_t stack_need = 0;          // most stack entries any traversal can hold
};

// Builds the wide BVH of a validated payload.  Returns an empty string on
// success, else the reason the payload cannot be represented.
std::string build_wide_bvh(const noor_payload_view* P, WideBvh& out);

// Structural check of a built wide BVH against the payload (see
// noor_wide_bvh_check).  Returns an empty string when it holds.
std::string check_wide_bvh(const noor_payload_view* P, const WideBvh& W);

}  // namespace noor

#endif
