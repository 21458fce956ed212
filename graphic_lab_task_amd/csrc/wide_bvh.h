// Six-wide BVH with quantised boxes: the layout that trace_wide.hip walks, and the rule that packs
// one node (used by the host builder and by the device refit of the instance level).
//
// Nodes of one base and three power-of-two steps with 8-bit planes, children consecutive, are those of H. Ylitie, T.
// Karras and S. Laine, "Efficient Incoherent Ray Traversal on GPUs Through Compressed Wide BVHs", HPG 2017 (eight
// wide there; six make one line segment here, and the leaves carry the exact boxes the sequential walk tests).
//
// The tree is collapsed from the binary one (device-layout pairs, TLAS nodes) at commit and lives in
// one array of 64-byte blocks, so that a node, a triangle or half an instance is one aligned line
// segment of four 16-byte loads. The children of a node are consecutive: inner children take one
// block, triangle leaves one block per triangle, SDF leaves one, instance leaves two.
#pragma once
#include "lrt_math.h"
#include "lrt_types.h"

namespace lrt {

constexpr uint32_t WIDE_CHILDREN = 6;
constexpr uint32_t WIDE_MAX_BLOCKS = 1u << 26;   // child block index field
constexpr uint32_t WIDE_MAX_LEAF_BLOCKS = 4;     // 2-bit field, blocks - 1
// Levels of a root-to-leaf path, both trees together: the walk keeps at most one stack entry a level.
constexpr uint32_t WIDE_MAX_LEVELS = 40;

struct WideBlock {
  uint32_t w[16];
};

// One inner node. Plane k of axis a lies at base[a] + q * 2^(exponent[a] - 127), lower planes rounded
// down and upper planes up, so a child's packed box contains its box.
struct alignas(16) WideNode {
  float    base[3];
  uint32_t exponents;   // 3 x 8 bits, biased as in a float
  // per axis three words: lo[0..3] | lo[4] lo[5] hi[4] hi[5] | hi[0..3] (one byte each)
  uint32_t planes[9];
  uint32_t children;    // first child block (26 bits), then one leaf bit per child
  uint32_t sizes;       // per child 2 bits: blocks - 1; bits 12-14: number of children
  uint32_t pad;
};
static_assert(sizeof(WideNode) == 64, "one block");

// One triangle of a leaf: its corners, its index in leaf order, and the box of the binary leaf it
// belongs to (which the sequential walk tests before the triangle).
struct alignas(16) WideTri {
  float3   a;
  uint32_t prim;
  float3   b;
  float    box_lx;
  float3   c;
  float    box_hx;
  float    box_ly, box_hy, box_lz, box_hz;
};
static_assert(sizeof(WideTri) == 64, "one block");

// SDF leaves carry their rank among the binary tree's leaves from left to right, and whether two sides that
// no plane separates lie above them: only among the leaves below one such pair can the sequential walk's
// order differ from the order of box entries along a ray. A frame-octree leaf has both in its FrameLeaf's
// `tex` (the bit WIDE_OVERLAP), a brick names the topmost such pair (WIDE_NO_OVERLAP: none).
constexpr uint32_t WIDE_OVERLAP = 0x80000000u;
constexpr uint32_t WIDE_NO_OVERLAP = 0xFFFFFFFFu;

// One brick of a sparse brick set: its binary leaf's box, its index in the set, its rank, its node record
// and the pair.
struct alignas(16) WideBrick {
  float3     boxMin;
  float3     boxMax;
  uint32_t   prim;
  uint32_t   rank;
  SdfSBSNode node;
  uint32_t   overlap;
  uint32_t   pad[3];
};
static_assert(sizeof(WideBrick) == 64, "one block");

// One instance: columns of the inverse transform (rows 0-2), its box in world space, the root of its
// geometry and the ids a hit reports.
struct alignas(16) WideInstance {
  float    inv[12];
  float3   boxMin;
  uint32_t root;      // WideRef of the geometry's root
  float3   boxMax;
  uint32_t inst_id;
  uint32_t geom_id;
  uint32_t rank;      // place in the sequential walk's order of instances
  uint32_t pad[10];
};
static_assert(sizeof(WideInstance) == 128, "two blocks");

LRT_HD WideInstance wide_instance(const InstanceData& in, uint32_t id, uint32_t root, uint32_t rank) {
  WideInstance w{};
  for (int c = 0; c < 4; ++c)
    for (int r = 0; r < 3; ++r) w.inv[3 * c + r] = in.transformInv.m[4 * c + r];
  w.boxMin = xyz(in.boxMin);
  w.boxMax = xyz(in.boxMax);
  w.root = root;
  w.inst_id = id;
  w.geom_id = in.geomId;
  w.rank = rank;
  return w;
}

// A place the walk can be at: block (26 bits) | (blocks - 1) << 26 | leaf bit 31.
LRT_HD uint32_t wide_ref(uint32_t block, uint32_t blocks, bool leaf) {
  return block | ((blocks - 1u) << 26) | (leaf ? 0x80000000u : 0u);
}

// The child in `slot` of a node (its children and sizes words).
LRT_HD uint32_t wide_child(uint32_t children, uint32_t sizes, uint32_t slot) {
  const uint32_t below = sizes & ((1u << (2 * slot)) - 1u);
  const uint32_t off = slot + uint32_t(__builtin_popcount(below & 0x555u)) + 2u * uint32_t(__builtin_popcount(below & 0xAAAu));
  const uint32_t leaf = ((children >> (26 + slot)) & 1u) << 31;
  return ((children & (WIDE_MAX_BLOCKS - 1u)) + off) | (((sizes >> (2 * slot)) & 3u) << 26) | leaf;
}

struct WideBox {
  float3 mn, mx;
};

// Packs the planes of n child boxes; returns false when a box is not finite or too large to pack.
LRT_HD bool wide_pack_planes(const WideBox* box, uint32_t n, WideNode& out) {
  uint8_t lo[3][6], hi[3][6];
  out.exponents = 0;
  for (int a = 0; a < 3; ++a) {
    float mn[6], mx[6];
    float base = 0.0f, top = 0.0f;
    for (uint32_t k = 0; k < 6; ++k) {
      if (k >= n) { lo[a][k] = 255; hi[a][k] = 0; continue; }
      mn[k] = a == 0 ? box[k].mn.x : (a == 1 ? box[k].mn.y : box[k].mn.z);
      mx[k] = a == 0 ? box[k].mx.x : (a == 1 ? box[k].mx.y : box[k].mx.z);
      if (!(mn[k] <= mx[k]) || !(mn[k] >= -1e30f) || !(mx[k] <= 1e30f)) return false;
      base = k == 0 || mn[k] < base ? mn[k] : base;
      top = k == 0 || mx[k] > top ? mx[k] : top;
    }
    // smallest power of two whose 255 steps span the boxes (at least 2^-100); the search begins eight to nine
    // powers below the span, where 255 steps are too few
    const double span = double(top) - double(base);
    uint64_t bits;
    __builtin_memcpy(&bits, &span, sizeof(bits));
    const int below = int(bits >> 52 & 0x7FF) - 1023 - 9;
    int e = below < -100 ? 27 : below + 127;
    bits = uint64_t(e - 127 + 1023) << 52;
    double step;   // 2^(e - 127)
    __builtin_memcpy(&step, &bits, sizeof(step));
    while (255.0 * step < span) { step *= 2.0; ++e; }
    for (;;) {
      bool fits = true;
      for (uint32_t k = 0; k < n; ++k) {
        int l = int((double(mn[k]) - double(base)) / step);
        while (l > 0 && double(base) + l * step > double(mn[k])) --l;
        int h = int((double(mx[k]) - double(base)) / step);
        while (double(base) + h * step < double(mx[k])) ++h;
        if (h > 255) { fits = false; break; }
        lo[a][k] = uint8_t(l);
        hi[a][k] = uint8_t(h);
      }
      if (fits) break;
      step *= 2.0;
      ++e;
    }
    out.base[a] = base;
    out.exponents |= uint32_t(e) << (8 * a);
    uint32_t* w = out.planes + 3 * a;
    w[0] = lo[a][0] | (uint32_t(lo[a][1]) << 8) | (uint32_t(lo[a][2]) << 16) | (uint32_t(lo[a][3]) << 24);
    w[1] = lo[a][4] | (uint32_t(lo[a][5]) << 8) | (uint32_t(hi[a][4]) << 16) | (uint32_t(hi[a][5]) << 24);
    w[2] = hi[a][0] | (uint32_t(hi[a][1]) << 8) | (uint32_t(hi[a][2]) << 16) | (uint32_t(hi[a][3]) << 24);
  }
  return true;
}

}  // namespace lrt
