// Host collapse of the binary trees into the six-wide layout of wide_bvh.h, at every commit of new geometry:
// subtrees are collapsed in parallel and each is copied to its place once. Commits with and without the tree, on 16
// cores: 327,680 triangles 13.6 and 7.3 ms (33.7 when subtrees were appended one by one, moved again and kept),
// 20,480 triangles 1.0 and 0.47, 1,280 triangles 0.44 and 0.30.
#include <algorithm>
#include <cstring>
#include <new>

#include "scene.h"
#include "wide_bvh.h"

namespace lrt {
namespace {

using Blocks = std::vector<WideBlock>;

// A child of a wide node while it is gathered: its exact box and what it is in the binary tree.
struct Child {
  float3 mn, mx;
  uint32_t word;     // what Tree::children opens, or a leaf word
  uint32_t source;   // index of its binary node (instance level)
  uint32_t depth;    // binary depth
  float area;        // of an inner child; negative for a leaf, which is never opened
};

// A wide node still to be packed and where it goes.
struct Item {
  uint32_t word, block, level, depth;
  float3 mn, mx;
};

float half_area(float3 mn, float3 mx) {
  const float3 d = mx - mn;
  return d.x * d.y + d.y * d.z + d.z * d.x;
}

bool contains(float3 mn, float3 mx, const BVHNode& c) {
  return c.boxMin.x >= mn.x && c.boxMin.y >= mn.y && c.boxMin.z >= mn.z && c.boxMax.x <= mx.x && c.boxMax.y <= mx.y &&
         c.boxMax.z <= mx.z;
}

// A collapsed tree: its top, and subtrees whose own blocks follow it one subtree after the other. Child indices
// count from the top's first block in the top and from a subtree's own first block in the subtree.
struct Subtree {
  Blocks blocks;
  std::vector<uint32_t> nodes;   // places of the nodes among the blocks (the first is the root, which has none)
  WideNode root;
  uint32_t at = 0;               // the root's place in the top
};
struct Collapsed {
  Blocks top;
  std::vector<uint32_t> top_nodes;
  std::vector<Subtree> subs;
  size_t size() const {
    size_t n = top.size();
    for (const Subtree& s : subs) n += s.blocks.size();
    return n;
  }
};

// Copies a part's blocks to their place and makes the child indices of its nodes count from block 0 of the tree.
void place(const Blocks& from, const std::vector<uint32_t>& nodes, size_t skip, WideBlock* tree, uint32_t base) {
  std::copy(from.begin(), from.end(), tree + base);
  for (size_t k = skip; k < nodes.size(); ++k) {
    WideNode n;
    std::memcpy(&n, tree + base + nodes[k], sizeof(n));
    n.children += base;
    std::memcpy(tree + base + nodes[k], &n, sizeof(n));
  }
}

// One tree's collapse. Tree opens an inner word into its two binary children; Leaf gives the blocks of a
// leaf word and writes them.
template <class Tree, class Leaf>
struct Collapse {
  const Tree& tree;
  const Leaf& leaf;

  // Gathers up to six children of the binary node it.word: the inner child of largest surface area
  // is replaced by its own two children until six are held or none is left.
  bool gather(const Item& it, Child* ch, uint32_t* count) const {
    uint32_t n = 0;
    auto open = [&](uint32_t word, float3 mn, float3 mx, uint32_t depth, uint32_t slot) -> bool {
      BVHNode two[2];
      uint32_t source[2];
      tree.children(word, two, source);
      bool in_slot = slot < n;
      for (int k = 0; k < 2; ++k) {
        if (two[k].leftOffset == LEAF_NORMAL) continue;   // the empty sibling of a one-leaf tree
        if (!contains(mn, mx, two[k])) return false;
        const bool is_leaf = (two[k].leftOffset & LEAF_BIT) != 0;
        const uint32_t to = in_slot ? slot : n++;
        in_slot = false;
        ch[to] = Child{two[k].boxMin, two[k].boxMax, two[k].leftOffset, source[k], depth + 1,
                       is_leaf ? -1.0f : half_area(two[k].boxMin, two[k].boxMax)};
      }
      return true;
    };
    if (!open(it.word, it.mn, it.mx, it.depth, WIDE_CHILDREN)) return false;
    while (n < WIDE_CHILDREN) {
      int best = -1;
      for (uint32_t k = 0; k < n; ++k)
        if (ch[k].area >= 0.0f && (best < 0 || ch[k].area > ch[best].area)) best = int(k);
      if (best < 0) break;
      const Child c = ch[best];
      if (!open(c.word, c.mn, c.mx, c.depth, uint32_t(best))) return false;
    }
    *count = n;
    return n > 0;
  }

  // Packs one item's node and appends its children's blocks to `out`; `todo` takes the inner children.
  // The caller writes `node` to its place.
  bool expand(const Item& it, Blocks& out, WideNode* node, std::vector<Item>& todo, uint32_t* max_level,
              std::vector<uint32_t>* sources) const {
    Child ch[WIDE_CHILDREN];
    uint32_t n = 0;
    if (!gather(it, ch, &n)) return false;
    WideBox box[WIDE_CHILDREN];
    uint32_t size[WIDE_CHILDREN], total = 0, leaf_bits = 0;
    *node = WideNode{};
    for (uint32_t k = 0; k < n; ++k) {
      box[k] = WideBox{ch[k].mn, ch[k].mx};
      size[k] = 1;
      if (ch[k].word & LEAF_BIT) {
        size[k] = leaf.blocks(ch[k].word);
        leaf_bits |= 1u << k;
      }
      if (size[k] < 1 || size[k] > WIDE_MAX_LEAF_BLOCKS) return false;
      // the sequential walk drops pushes past its stack; so deep a tree keeps that walk
      if (ch[k].depth >= uint32_t(STACK_SIZE)) return false;
      node->sizes |= (size[k] - 1) << (2 * k);
      total += size[k];
    }
    if (!wide_pack_planes(box, n, *node)) return false;
    const size_t first = out.size();
    if (first + total >= WIDE_MAX_BLOCKS) return false;
    node->children = uint32_t(first) | (leaf_bits << 26);
    node->sizes |= n << 12;
    out.resize(first + total);
    if (sources) {
      sources->resize(out.size() * WIDE_CHILDREN, 0xFFFFFFFFu);
      for (uint32_t k = 0; k < n; ++k) (*sources)[size_t(it.block) * WIDE_CHILDREN + k] = ch[k].source;
    }
    uint32_t b = uint32_t(first);
    for (uint32_t k = 0; k < n; ++k) {
      if (leaf_bits >> k & 1u) {
        if (!leaf.write(ch[k].word, ch[k].mn, ch[k].mx, &out[b])) return false;
      } else {
        todo.push_back(Item{ch[k].word, b, it.level + 1, ch[k].depth, ch[k].mn, ch[k].mx});
        *max_level = std::max(*max_level, it.level + 1);
      }
      b += size[k];
    }
    return true;
  }

  // The tree: its root is block 0 of `out.top`. The top is built breadth first until there are enough subtrees
  // for the cores, then each subtree depth first into blocks of its own, so that a subtree's blocks stay together.
  bool run(Collapsed& out, uint32_t* max_level, std::vector<uint32_t>* sources) const {
    const float inf = 3e38f;
    std::vector<Item> todo{Item{0u, 0u, 1u, 0u, make3(-inf, -inf, -inf), make3(inf, inf, inf)}};
    out.top.assign(1, WideBlock{});
    if (sources) sources->assign(WIDE_CHILDREN, 0xFFFFFFFFu);
    *max_level = 1;
    size_t at = 0;
    while (at < todo.size() && (sources || todo.size() - at < 256)) {
      const Item it = todo[at++];
      WideNode node;
      if (!expand(it, out.top, &node, todo, max_level, sources)) return false;
      std::memcpy(&out.top[it.block], &node, sizeof(node));
      out.top_nodes.push_back(it.block);
    }
    const int n_sub = int(todo.size() - at);
    out.subs.resize(size_t(n_sub));
    std::vector<uint32_t> levels(size_t(n_sub), 0u);
    bool ok = true;
#pragma omp parallel for schedule(dynamic, 1)
    for (int k = 0; k < n_sub; ++k) {
      Subtree& s = out.subs[size_t(k)];
      bool good = true;
      try {   // (nothing may leave the loop's threads)
        std::vector<Item> stack{todo[at + size_t(k)]};
        s.at = stack[0].block;
        while (good && !stack.empty()) {
          const Item it = stack.back();
          stack.pop_back();
          WideNode node;
          const bool first = s.nodes.empty();
          good = expand(it, s.blocks, &node, stack, &levels[size_t(k)], nullptr);
          if (!good) break;
          if (first) s.root = node;
          else std::memcpy(&s.blocks[it.block], &node, sizeof(node));
          s.nodes.push_back(it.block);
        }
      } catch (const std::bad_alloc&) {
        good = false;
      }
      if (!good)
#pragma omp atomic write
        ok = false;
    }
    if (!ok) return false;
    for (uint32_t l : levels) *max_level = std::max(*max_level, l);
    return out.size() < WIDE_MAX_BLOCKS;
  }
};

struct PairTree {
  const BVHNodePair* pairs;
  void children(uint32_t word, BVHNode* two, uint32_t* source) const {
    two[0] = pairs[word].left;
    two[1] = pairs[word].right;
    source[0] = source[1] = 0;
  }
};

struct TlasTree {
  const BVHNode* nodes;
  void children(uint32_t word, BVHNode* two, uint32_t* source) const {
    for (uint32_t k = 0; k < 2; ++k) {
      two[k] = nodes[word + k];
      source[k] = word + k;
    }
  }
};

struct TriLeaf {
  const float4* soup;   // of the geometry
  uint32_t blocks(uint32_t word) const { return extract_count(word); }
  bool write(uint32_t word, float3 mn, float3 mx, WideBlock* out) const {
    for (uint32_t j = 0; j < extract_count(word); ++j) {
      const uint32_t prim = extract_start(word) + j;
      const float4* q = soup + size_t(prim) * 3;
      const WideTri t{xyz(q[0]), prim, xyz(q[1]), mn.x, xyz(q[2]), mx.x, mn.y, mx.y, mn.z, mx.z};
      std::memcpy(out + j, &t, sizeof(t));
    }
    return true;
  }
};

// Where the sequential walk has an SDF leaf: its rank from the left, and the topmost pair above it whose two
// sides overlap.
struct LeafOrder {
  uint32_t rank = 0, above = WIDE_NO_OVERLAP;
};

bool same_box(float3 amn, float3 amx, float3 bmn, float3 bmx) {
  return amn.x == bmn.x && amn.y == bmn.y && amn.z == bmn.z && amx.x == bmx.x && amx.y == bmx.y && amx.z == bmx.z;
}

struct FrameLeafWriter {
  const FrameLeaf* leaves;   // of the geometry
  const LeafOrder* order;
  uint32_t blocks(uint32_t) const { return 1; }
  bool write(uint32_t word, float3 mn, float3 mx, WideBlock* out) const {
    FrameLeaf f = leaves[extract_start(word)];
    const LeafOrder& at = order[extract_start(word)];
    f.tex = at.rank | (at.above != WIDE_NO_OVERLAP ? WIDE_OVERLAP : 0u);   // untextured leaves have no use for it
    std::memcpy(out, &f, sizeof(f));
    // the leaf routine tests the record's box, the binary walk the node's: they must be the same
    return same_box(f.boxMin, f.boxMax, mn, mx);
  }
};

struct BrickLeaf {
  const SdfSBSNode* nodes;   // of the geometry
  size_t count;
  const LeafOrder* order;
  uint32_t blocks(uint32_t) const { return 1; }
  bool write(uint32_t word, float3 mn, float3 mx, WideBlock* out) const {
    const uint32_t prim = extract_start(word);
    if (prim >= count) return false;   // the dummy box beside a single brick
    const WideBrick b{mn, mx, prim, order[prim].rank, nodes[prim], order[prim].above, {}};
    std::memcpy(out, &b, sizeof(b));
    return true;
  }
};

struct InstanceLeaf {
  const InstanceData* instances;
  const uint32_t* roots;   // per geometry
  const uint32_t* ranks;   // per instance
  uint32_t blocks(uint32_t) const { return 2; }
  bool write(uint32_t word, float3, float3, WideBlock* out) const {
    const uint32_t i = extract_start(word);
    const WideInstance w = wide_instance(instances[i], i, roots[instances[i].geomId], ranks[i]);
    std::memcpy(out, &w, sizeof(w));
    return true;
  }
};

}  // namespace

namespace {

// Marks a BLAS's device pairs with what the order of its leaves needs (the BLAS walks do not read escape
// indices): right.escapeIndex the rank of the right side's first leaf, counted from the left (a mesh
// counts triangles: the rank is the index of the leaf's first one), and left.escapeIndex 1 where no plane
// separates the two sides. `order` takes a box leaf's rank and the topmost such pair above it. False where
// a mesh's triangle indices do not grow from left to right.
bool apart(const BVHNode& l, const BVHNode& r) {
  return l.leftOffset == LEAF_NORMAL || r.leftOffset == LEAF_NORMAL || l.boxMax.x <= r.boxMin.x || r.boxMax.x <= l.boxMin.x ||
         l.boxMax.y <= r.boxMin.y || r.boxMax.y <= l.boxMin.y || l.boxMax.z <= r.boxMin.z || r.boxMax.z <= l.boxMin.z;
}

bool mark_mesh_order(BVHNodePair* pairs, uint32_t n) {
  // per pair the first triangle below it and the one after the last: an empty side has neither
  std::vector<uint2> span(n);
  auto of = [&](const BVHNode& c, uint32_t empty) {
    if (c.leftOffset == LEAF_NORMAL) return uint2{empty, empty};
    if (c.leftOffset & LEAF_BIT) return uint2{extract_start(c.leftOffset), extract_start(c.leftOffset) + extract_count(c.leftOffset)};
    return span[c.leftOffset];
  };
  // children are stored after their parent
  for (uint32_t p = n; p-- > 0;) {
    BVHNode &l = pairs[p].left, &r = pairs[p].right;
    for (const BVHNode* c : {&l, &r})
      if (!(c->leftOffset & LEAF_BIT) && (c->leftOffset <= p || c->leftOffset >= n)) return false;
    const uint2 right = of(r, l.leftOffset == LEAF_NORMAL ? 0u : of(l, 0u).y);
    const uint2 left = of(l, right.x);
    if (left.y != right.x) return false;
    span[p] = uint2{left.x, right.y};
    r.escapeIndex = right.x;
    l.escapeIndex = apart(l, r) ? 0u : 1u;
  }
  return n == 0 || span[0].x == 0;
}

bool mark_leaf_order(BVHNodePair* pairs, uint32_t n, std::vector<LeafOrder>& order) {
  std::vector<uint32_t> count(n, 0u), first(n, 0u), above(n, WIDE_NO_OVERLAP);
  auto leaves = [&](const BVHNode& c) -> uint32_t {
    if (c.leftOffset == LEAF_NORMAL) return 0u;   // the empty sibling of a one-leaf tree
    return c.leftOffset & LEAF_BIT ? 1u : count[c.leftOffset];
  };
  // children are stored after their parent
  for (uint32_t p = n; p-- > 0;) {
    for (const BVHNode* c : {&pairs[p].left, &pairs[p].right})
      if (!(c->leftOffset & LEAF_BIT) && (c->leftOffset <= p || c->leftOffset >= n)) return false;
    count[p] = leaves(pairs[p].left) + leaves(pairs[p].right);
  }
  order.assign(n == 0 ? 0u : count[0], LeafOrder{});
  for (uint32_t p = 0; p < n; ++p) {
    BVHNode &l = pairs[p].left, &r = pairs[p].right;
    const bool separate = apart(l, r);
    const uint32_t overlap = above[p] != WIDE_NO_OVERLAP || separate ? above[p] : p;
    uint32_t at = first[p];
    for (BVHNode* c : {&l, &r}) {
      if (c->leftOffset == LEAF_NORMAL) continue;
      if (!(c->leftOffset & LEAF_BIT)) {
        first[c->leftOffset] = at;
        above[c->leftOffset] = overlap;
      } else {
        if (extract_start(c->leftOffset) >= order.size()) return false;
        order[extract_start(c->leftOffset)] = LeafOrder{at, overlap};
      }
      at += leaves(*c);
    }
    r.escapeIndex = first[p] + leaves(l);
    l.escapeIndex = separate ? 0u : 1u;
  }
  return true;
}

}  // namespace

// The instance level: its nodes and instance blocks fill the first 3 blocks per instance, wideTop
// (fewer nodes than instances, two blocks an instance), so that a new instance tree of the same
// instances fits again. Returns false when it cannot be packed.
bool Scene::build_wide_instances(uint32_t* levels) {
  const size_t room = 3 * instances.size();
  // the sequential walk takes left children first
  std::vector<uint32_t> ranks(instances.size(), 0u);
  if (instances.size() > 1) {
    std::vector<uint32_t> stack{1u, 0u};
    uint32_t rank = 0;
    while (!stack.empty()) {
      const uint32_t lo = tlas[stack.back()].leftOffset;
      stack.pop_back();
      if (lo & LEAF_BIT) {
        ranks[extract_start(lo)] = rank++;
      } else {
        stack.push_back(lo + 1);
        stack.push_back(lo);
      }
    }
  }
  const InstanceLeaf leaf{instances.data(), wideRoots.data(), ranks.data()};
  Collapsed tree;
  std::vector<WideBlock>& top = tree.top;
  wideSources.clear();
  *levels = 0;
  if (instances.size() == 1) {
    top.resize(2);
    leaf.write(pack_offset_and_size(0, 1), float3{}, float3{}, top.data());
    wideRoot = wide_ref(0, 2, true);
  } else {
    const TlasTree binary{tlas.data()};
    if (!Collapse<TlasTree, InstanceLeaf>{binary, leaf}.run(tree, levels, &wideSources)) return false;
    wideRoot = wide_ref(0, 1, false);
  }
  if (top.size() > room) return false;
  wideTop = std::move(top);
  wideTop.resize(room);
  return true;
}

// Builds wideBuild from the device layout (devNodes, triSoup, frameLeaves, sbsNodes) and the TLAS, or leaves
// no tree where the wide walk does not apply: it takes scenes of triangle meshes only, and scenes of one
// instance of a frame octree, sparse voxel set or sparse brick set. Nor is there one where memory is short.
void Scene::build_wide() {
  bool ok = false;
  try {
    ok = build_wide_tree();
  } catch (const std::bad_alloc&) {
  }
  if (ok) return;
  wideBuild.reset();
  wideCount = 0;
  wideTop.clear();
  wideSources.clear();
}

bool Scene::build_wide_tree() {
  wideRoots.assign(geomData.size(), 0u);
  const uint32_t kinds = leaf_kinds();
  const bool sdf = (kinds == LK_FRAME || kinds == LK_SBS) && instances.size() == 1;
  if ((kinds != LK_TRI && !sdf) || instances.empty()) return false;
  std::vector<uint8_t> used(geomData.size(), 0);
  for (const InstanceData& i : instances) used[i.geomId] = 1;
  std::vector<Collapsed> geom(geomData.size());
  wideBlasLevels = 0;
  size_t total = 3 * instances.size();
  for (size_t g = 0; g < geomData.size(); ++g) {
    if (!used[g]) continue;
    const size_t first = geomData[g].bvhOffset, end = g + 1 < geomData.size() ? geomData[g + 1].bvhOffset : devNodes.size();
    if (first >= end) return false;   // an empty mesh
    std::vector<LeafOrder> order;
    if (kinds == LK_TRI ? !mark_mesh_order(devNodes.data() + first, uint32_t(end - first))
                        : !mark_leaf_order(devNodes.data() + first, uint32_t(end - first), order))
      return false;
    const PairTree tree{devNodes.data() + first};
    uint32_t levels = 0;
    bool ok;
    if (kinds == LK_FRAME) {
      const FrameLeafWriter leaf{frameLeaves.data() + geomData[g].offset.y, order.data()};
      ok = Collapse<PairTree, FrameLeafWriter>{tree, leaf}.run(geom[g], &levels, nullptr);
    } else if (kinds == LK_SBS) {
      const uint32_t set = geomData[g].offset.x;
      const size_t last = set + 1 < sbsRoots.size() ? sbsRoots[set + 1] : sbsNodes.size();
      const BrickLeaf leaf{sbsNodes.data() + sbsRoots[set], last - sbsRoots[set], order.data()};
      ok = Collapse<PairTree, BrickLeaf>{tree, leaf}.run(geom[g], &levels, nullptr);
    } else {
      const TriLeaf leaf{triSoup.data() + geomData[g].offset.x};
      ok = Collapse<PairTree, TriLeaf>{tree, leaf}.run(geom[g], &levels, nullptr);
    }
    if (!ok) return false;
    wideRoots[g] = wide_ref(uint32_t(total), 1, false);
    total += geom[g].size();
    if (total >= WIDE_MAX_BLOCKS) return false;
    wideBlasLevels = std::max(wideBlasLevels, levels);
  }
  uint32_t levels = 0;
  if (!build_wide_instances(&levels) || levels + wideBlasLevels > WIDE_MAX_LEVELS) return false;
  wideLevels = levels + wideBlasLevels;
  wideBuild.reset(new WideBlock[total]);   // not cleared: every block is written below
  wideCount = total;
  WideBlock* tree = wideBuild.get();
  std::copy(wideTop.begin(), wideTop.end(), tree);
  for (size_t g = 0; g < geom.size(); ++g) {
    const Collapsed& c = geom[g];
    if (c.top.empty()) continue;
    const uint32_t base = wideRoots[g] & (WIDE_MAX_BLOCKS - 1);
    place(c.top, c.top_nodes, 0, tree, base);
    const int n_sub = int(c.subs.size());
    std::vector<uint32_t> at(c.subs.size() + 1, base + uint32_t(c.top.size()));
    for (int k = 0; k < n_sub; ++k) at[size_t(k) + 1] = at[size_t(k)] + uint32_t(c.subs[size_t(k)].blocks.size());
#pragma omp parallel for schedule(dynamic, 1)
    for (int k = 0; k < n_sub; ++k) {
      const Subtree& s = c.subs[size_t(k)];
      place(s.blocks, s.nodes, 1, tree, at[size_t(k)]);
      WideNode root = s.root;
      root.children += at[size_t(k)];
      std::memcpy(tree + base + s.at, &root, sizeof(root));
    }
  }
  return true;
}

}  // namespace lrt
