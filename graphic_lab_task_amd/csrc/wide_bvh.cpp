// Host collapse of the binary trees into the six-wide layout of wide_bvh.h.
#include <algorithm>
#include <cstring>

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

  // The tree of `root` (its node becomes block 0 of `out`): the top breadth first until there are
  // enough subtrees for the cores, then each subtree depth first into blocks of its own, appended in
  // order, so that a subtree's blocks stay together.
  bool run(Blocks& out, uint32_t* max_level, std::vector<uint32_t>* sources) const {
    const float inf = 3e38f;
    std::vector<Item> todo{Item{0u, 0u, 1u, 0u, make3(-inf, -inf, -inf), make3(inf, inf, inf)}};
    out.assign(1, WideBlock{});
    if (sources) sources->assign(WIDE_CHILDREN, 0xFFFFFFFFu);
    *max_level = 1;
    size_t at = 0;
    while (at < todo.size() && (sources || todo.size() - at < 256)) {
      const Item it = todo[at++];
      WideNode node;
      if (!expand(it, out, &node, todo, max_level, sources)) return false;
      std::memcpy(&out[it.block], &node, sizeof(node));
    }
    const int n_sub = int(todo.size() - at);
    struct Sub {
      Blocks blocks;
      WideNode root;
      uint32_t levels = 0;
      bool ok = true;
    };
    std::vector<Sub> subs(size_t(n_sub) > 0 ? size_t(n_sub) : 0);
#pragma omp parallel for schedule(dynamic, 1)
    for (int k = 0; k < n_sub; ++k) {
      Sub& s = subs[size_t(k)];
      std::vector<Item> stack{todo[at + size_t(k)]};
      bool first = true;
      while (s.ok && !stack.empty()) {
        const Item it = stack.back();
        stack.pop_back();
        WideNode node;
        s.ok = expand(it, s.blocks, &node, stack, &s.levels, nullptr);
        if (first) s.root = node;
        else if (s.ok) std::memcpy(&s.blocks[it.block], &node, sizeof(node));
        first = false;
      }
    }
    for (int k = 0; k < n_sub; ++k) {
      Sub& s = subs[size_t(k)];
      if (!s.ok || out.size() + s.blocks.size() >= WIDE_MAX_BLOCKS) return false;
      const uint32_t base = uint32_t(out.size());
      s.root.children += base;
      std::memcpy(&out[todo[at + size_t(k)].block], &s.root, sizeof(s.root));
      *max_level = std::max(*max_level, s.levels);
      shift(s.blocks, s.root, base);
      out.insert(out.end(), s.blocks.begin(), s.blocks.end());
      s.blocks = Blocks();
    }
    return true;
  }

  // Adds `base` to the child indices of every node below `root`, whose own index is already moved.
  static void shift(Blocks& blocks, const WideNode& root, uint32_t base) {
    std::vector<WideNode> stack{root};
    while (!stack.empty()) {
      const WideNode n = stack.back();
      stack.pop_back();
      uint32_t b = (n.children & (WIDE_MAX_BLOCKS - 1)) - base;
      for (uint32_t k = 0; k < (n.sizes >> 12); ++k) {
        if (!(n.children >> (26 + k) & 1u)) {
          WideNode c;
          std::memcpy(&c, &blocks[b], sizeof(c));
          c.children += base;
          std::memcpy(&blocks[b], &c, sizeof(c));
          stack.push_back(c);
        }
        b += (n.sizes >> (2 * k) & 3u) + 1;
      }
    }
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
bool mark_order(BVHNodePair* pairs, uint32_t n, bool mesh, std::vector<LeafOrder>& order) {
  std::vector<uint32_t> count(n, 0u), first(n, 0u), above(n, WIDE_NO_OVERLAP);
  auto leaves = [&](const BVHNode& c) -> uint32_t {
    if (c.leftOffset == LEAF_NORMAL) return 0u;   // the empty sibling of a one-leaf tree
    if (c.leftOffset & LEAF_BIT) return mesh ? extract_count(c.leftOffset) : 1u;
    return count[c.leftOffset];
  };
  // children are stored after their parent
  for (uint32_t p = n; p-- > 0;) {
    for (const BVHNode* c : {&pairs[p].left, &pairs[p].right})
      if (!(c->leftOffset & LEAF_BIT) && (c->leftOffset <= p || c->leftOffset >= n)) return false;
    count[p] = leaves(pairs[p].left) + leaves(pairs[p].right);
  }
  order.assign(mesh || n == 0 ? 0u : count[0], LeafOrder{});
  for (uint32_t p = 0; p < n; ++p) {
    BVHNode &l = pairs[p].left, &r = pairs[p].right;
    const bool apart = l.leftOffset == LEAF_NORMAL || r.leftOffset == LEAF_NORMAL || l.boxMax.x <= r.boxMin.x ||
                       r.boxMax.x <= l.boxMin.x || l.boxMax.y <= r.boxMin.y || r.boxMax.y <= l.boxMin.y ||
                       l.boxMax.z <= r.boxMin.z || r.boxMax.z <= l.boxMin.z;
    const uint32_t overlap = above[p] != WIDE_NO_OVERLAP || apart ? above[p] : p;
    uint32_t at = first[p];
    for (BVHNode* c : {&l, &r}) {
      if (c->leftOffset == LEAF_NORMAL) continue;
      if (!(c->leftOffset & LEAF_BIT)) {
        first[c->leftOffset] = at;
        above[c->leftOffset] = overlap;
      } else if (mesh) {
        if (extract_start(c->leftOffset) != at) return false;
      } else {
        if (extract_start(c->leftOffset) >= order.size()) return false;
        order[extract_start(c->leftOffset)] = LeafOrder{at, overlap};
      }
      at += leaves(*c);
    }
    r.escapeIndex = first[p] + leaves(l);
    l.escapeIndex = apart ? 0u : 1u;
  }
  return true;
}

}  // namespace

// The instance level: its nodes and instance blocks fill the first 3 blocks per instance of wideBlocks
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
  std::vector<WideBlock> top;
  wideSources.clear();
  *levels = 0;
  if (instances.size() == 1) {
    top.resize(2);
    leaf.write(pack_offset_and_size(0, 1), float3{}, float3{}, top.data());
    wideRoot = wide_ref(0, 2, true);
  } else {
    const TlasTree tree{tlas.data()};
    if (!Collapse<TlasTree, InstanceLeaf>{tree, leaf}.run(top, levels, &wideSources)) return false;
    wideRoot = wide_ref(0, 1, false);
  }
  if (top.size() > room) return false;
  std::copy(top.begin(), top.end(), wideBlocks.begin());
  return true;
}

// Builds wideBlocks from the device layout (devNodes, triSoup, frameLeaves, sbsNodes) and the TLAS, or
// leaves it empty where the wide walk does not apply: it takes scenes of triangle meshes only, and scenes
// of one instance of a frame octree, sparse voxel set or sparse brick set.
void Scene::build_wide() {
  wideBlocks.clear();
  wideSources.clear();
  wideRoots.assign(geomData.size(), 0u);
  const uint32_t kinds = leaf_kinds();
  const bool sdf = (kinds == LK_FRAME || kinds == LK_SBS) && instances.size() == 1;
  if ((kinds != LK_TRI && !sdf) || instances.empty()) return;
  std::vector<uint8_t> used(geomData.size(), 0);
  for (const InstanceData& i : instances) used[i.geomId] = 1;
  std::vector<Blocks> geom(geomData.size());
  wideBlasLevels = 0;
  size_t total = 3 * instances.size();
  for (size_t g = 0; g < geomData.size(); ++g) {
    if (!used[g]) continue;
    const size_t first = geomData[g].bvhOffset, end = g + 1 < geomData.size() ? geomData[g + 1].bvhOffset : devNodes.size();
    if (first >= end) return;   // an empty mesh
    std::vector<LeafOrder> order;
    if (!mark_order(devNodes.data() + first, uint32_t(end - first), kinds == LK_TRI, order)) return;
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
    wideRoots[g] = wide_ref(uint32_t(total), 1, false);
    total += geom[g].size();
    if (!ok || total >= WIDE_MAX_BLOCKS) return;
    wideBlasLevels = std::max(wideBlasLevels, levels);
  }
  wideBlocks.resize(total);
  uint32_t levels = 0;
  if (!build_wide_instances(&levels) || levels + wideBlasLevels > WIDE_MAX_LEVELS) {
    wideBlocks.clear();
    return;
  }
  wideLevels = levels + wideBlasLevels;
#pragma omp parallel for schedule(dynamic, 1)
  for (int g = 0; g < int(geom.size()); ++g) {
    Blocks& b = geom[size_t(g)];
    if (b.empty()) continue;
    const uint32_t base = wideRoots[size_t(g)];
    WideNode root;
    std::memcpy(&root, &b[0], sizeof(root));
    root.children += base;
    std::memcpy(&b[0], &root, sizeof(root));
    Collapse<PairTree, TriLeaf>::shift(b, root, base);
    std::copy(b.begin(), b.end(), wideBlocks.begin() + base);
  }
}

}  // namespace lrt
