// The walk of one wave through the six-wide tree (wide_bvh.h), shared by the trace kernels
// (trace_wide.hip) and the differentiable brick-set kernels (diff_kernels.hip).
#pragma once
#include "traverse.h"
#include "wide_bvh.h"

namespace lrt {

enum WideLeafKind { WIDE_TRI, WIDE_FRAME, WIDE_BRICK };

constexpr int WIDE_BLOCK = 64;
constexpr int WIDE_LDS_STACK = 12;   // entries in LDS; the deeper ones spill
// Idle lanes from which on parts of rays are handed over (327,680 triangles, 512 x 512: 8 193 us, 16 186, 32 186)
constexpr uint32_t WIDE_SHARE = 16;
constexpr uint32_t WIDE_DONE = 0xFFFFFFFFu;
constexpr uint32_t WIDE_LEAF = 0x80000000u;
constexpr uint32_t WIDE_INDEX = WIDE_MAX_BLOCKS - 1;

typedef __attribute__((address_space(3))) uint32_t wide_lds;

// One stack entry: a node's children word and, in the second word, its sizes (12 bits) and the slots
// still to visit, nearest first (3 bits each, 7 ends the list).
template <int BLOCK>
struct WideStack {
  wide_lds* col;     // entry i at col[2 i BLOCK], col[(2 i + 1) BLOCK]
  uint32_t* spill;   // entry i >= WIDE_LDS_STACK at spill[2 (i - WIDE_LDS_STACK)]
  __device__ __forceinline__ void put(int i, uint32_t a, uint32_t b) {
    if (i < WIDE_LDS_STACK) {
      col[2 * i * BLOCK] = a;
      col[(2 * i + 1) * BLOCK] = b;
    } else {
      spill[2 * (i - WIDE_LDS_STACK)] = a;
      spill[2 * (i - WIDE_LDS_STACK) + 1] = b;
    }
  }
  __device__ __forceinline__ void put_order(int i, uint32_t b) {
    if (i < WIDE_LDS_STACK) col[(2 * i + 1) * BLOCK] = b;
    else spill[2 * (i - WIDE_LDS_STACK) + 1] = b;
  }
  __device__ __forceinline__ uint2 get(int i) const {
    uint2 e;
    if (i < WIDE_LDS_STACK) {
      e.x = col[2 * i * BLOCK];
      e.y = col[(2 * i + 1) * BLOCK];
    } else {
      e.x = spill[2 * (i - WIDE_LDS_STACK)];
      e.y = spill[2 * (i - WIDE_LDS_STACK) + 1];
    }
    return e;
  }
};

__device__ __forceinline__ float byte_of(uint32_t w, int k) { return float((w >> (8 * k)) & 0xFFu); }

__device__ __forceinline__ void order2(uint32_t& a, uint32_t& b) {
  const uint32_t lo = a < b ? a : b;
  b = a < b ? b : a;
  a = lo;
}

// Limit for box entries once a hit at t is known: a little past t (2^-14 of it, and `slop` for the
// rounding of instance boxes and transforms), so that a leaf whose entry rounds past its own triangle's t
// is still seen.
__device__ __forceinline__ float wide_limit(float t, float slop) { return __builtin_fmaf(t, 6.1035156e-5f, t) + slop; }

// BVHRT's matmul4x3 / matmul3x3 (w = 1 / 0) with the columns of a WideInstance.
__device__ __forceinline__ float3 wide_transform(const float* m, float3 v, float w) {
  return make3(v.x * m[0] + v.y * m[3] + v.z * m[6] + w * m[9], v.x * m[1] + v.y * m[4] + v.z * m[7] + w * m[10],
               v.x * m[2] + v.y * m[5] + v.z * m[8] + w * m[11]);
}

// Hit children of the node at q, as sort keys: entry distance with the slot in its low 3 bits, sorted,
// all ones for a miss. A plane's distance is q * (step * inv) + (base - o) * inv; the part with base is
// widened by 2^-21 of itself and the exit by 2^-20, more than the roundings by which this and the exact
// test (2 each, 2^-24) can differ. NaN products drop out of min and max, which lets the child through.
__device__ __forceinline__ void wide_test(const uint4& a, const uint4& b, const uint4& c, const uint4& e, float3 o,
                                          float3 inv, float tnear, float limit, uint32_t key[6]) {
  float tn[6], tf[6];
  const uint32_t planes[9] = {b.x, b.y, b.z, b.w, c.x, c.y, c.z, c.w, e.x};
  const float base[3] = {__uint_as_float(a.x), __uint_as_float(a.y), __uint_as_float(a.z)};
  const float org[3] = {o.x, o.y, o.z}, rcp[3] = {inv.x, inv.y, inv.z};
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    const float step = __uint_as_float(((a.w >> (8 * x)) & 0xFFu) << 23) * rcp[x];
    const float at = (base[x] - org[x]) * rcp[x];
    const float err = fabsf(at) * 4.7683716e-7f;
    const float an = at - err, af = at + err;
    const bool neg = rcp[x] < 0.0f;
    const uint32_t p0 = planes[3 * x], p1 = planes[3 * x + 1], p2 = planes[3 * x + 2];
    const uint32_t n0 = neg ? p2 : p0, f0 = neg ? p0 : p2;
    const uint32_t m = neg ? __builtin_amdgcn_alignbit(p1, p1, 16) : p1;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      const float qn = k < 4 ? byte_of(n0, k) : byte_of(m, k - 4);
      const float qf = k < 4 ? byte_of(f0, k) : byte_of(m, k - 2);
      const float n = __builtin_fmaf(qn, step, an), f = __builtin_fmaf(qf, step, af);
      tn[k] = x == 0 ? fmaxf(n, tnear) : fmaxf(tn[k], n);
      tf[k] = x == 0 ? f : fminf(tf[k], f);
    }
  }
  const uint32_t count = e.z >> 12;
#pragma unroll
  for (uint32_t k = 0; k < 6; ++k) {
    const float exit = fminf(__builtin_fmaf(fabsf(tf[k]), 9.536743e-7f, tf[k]), limit);
    key[k] = tn[k] <= exit && k < count ? (__float_as_uint(tn[k]) & ~7u) | k : 0xFFFFFFFFu;
  }
  order2(key[0], key[5]); order2(key[1], key[3]); order2(key[2], key[4]);
  order2(key[1], key[2]); order2(key[3], key[4]);
  order2(key[0], key[3]); order2(key[2], key[5]);
  order2(key[0], key[1]); order2(key[2], key[3]); order2(key[4], key[5]);
  order2(key[1], key[2]); order2(key[3], key[4]);
}

// The ray of an instance block, in the instance's space.
__device__ __forceinline__ void wide_local_ray(const WideInstance* w, float3 p, float3 q, float3& o, float3& d) {
  float m[12];
#pragma unroll
  for (int k = 0; k < 12; ++k) m[k] = w->inv[k];
  o = wide_transform(m, p, 1.0f);
  d = wide_transform(m, q, 0.0f);
}

// Whether the sequential walk of the instance at block `inst` reaches the leaf of rank a before that of
// rank b (both on the ray and below the pair `at`): the nearer-child rule at the pair where they part. A mesh's ranks are
// triangle indices, and within a leaf they are in order. The device pairs hold the first rank of their
// right side in right.escapeIndex. Rare: it reads what it needs.
__device__ __forceinline__ bool wide_before(const SceneView& s, float4 pos, float4 dir, uint32_t inst, uint32_t at,
                                            uint32_t a, uint32_t b) {
  const WideInstance* w = reinterpret_cast<const WideInstance*>(s.wide + inst);
  float3 o, d;
  wide_local_ray(w, xyz(pos), xyz(dir), o, d);
  const float3 inv = safe_inverse(d);
  const uint32_t lo = a < b ? a : b, hi = a < b ? b : a;
  const BVHNodePair* nodes = s.nodes + s.geoms[w->geom_id].bvhOffset;
  for (int k = 0; k < STACK_SIZE; ++k) {   // such trees are no deeper
    const BVHNodePair* pair = nodes + at;
    const uint32_t split = pair->right.escapeIndex;
    uint32_t child;
    if (hi < split) child = pair->left.leftOffset;
    else if (lo >= split) child = pair->right.leftOffset;
    else {
      const float l = ray_box2_fast(o, inv, pair->left.boxMin, pair->left.boxMax).x;
      const float r = ray_box2_fast(o, inv, pair->right.boxMin, pair->right.boxMax).x;
      return (a == lo) == (l <= r);
    }
    if (child & LEAF_BIT) break;
    at = child;
  }
  return a == lo;
}

// How far along the ray a leaf can begin that the sequential walk reaches before the leaf of rank a, which
// begins at `entry`. A plane between the sides of a binary node puts all that is visited earlier before
// `entry`; where the sides overlap (left.escapeIndex 1) and the other one is visited first, its exit.
__device__ __forceinline__ float wide_reach(const SceneView& s, float4 pos, float4 dir, uint32_t inst, uint32_t at,
                                            uint32_t a, float entry) {
  const WideInstance* w = reinterpret_cast<const WideInstance*>(s.wide + inst);
  float3 o, d;
  wide_local_ray(w, xyz(pos), xyz(dir), o, d);
  const float3 inv = safe_inverse(d);
  const BVHNodePair* nodes = s.nodes + s.geoms[w->geom_id].bvhOffset;
  float reach = entry;
  for (int k = 0; k < STACK_SIZE; ++k) {
    const BVHNodePair* pair = nodes + at;
    const bool left = a < pair->right.escapeIndex;
    if (pair->left.escapeIndex != 0u) {
      const float2 l = ray_box2_fast(o, inv, pair->left.boxMin, pair->left.boxMax);
      const float2 r = ray_box2_fast(o, inv, pair->right.boxMin, pair->right.boxMax);
      const float2 other = left ? r : l;
      if (other.x <= other.y && left != (l.x <= r.x)) reach = fmaxf(reach, other.y);
    }
    const uint32_t child = left ? pair->left.leftOffset : pair->right.leftOffset;
    if (child & LEAF_BIT) break;
    at = child;
  }
  return reach;
}

// Walks rays with all lanes of a wave (a one-wave block) until `fetch` has no more. A lane whose ray has
// ended takes a new one (once a quarter of the wave is idle); when the rays run out, an idle lane takes
// the oldest stack entry of a busy one, that is the largest part of its ray still to walk, and walks it
// for that ray: the last rays of a batch, and all rays of a small one, are walked by many lanes each. The
// parts' results are merged by the lane that holds the ray. Inner nodes are stepped until half of the
// wave's working lanes stand at a leaf.
// ANY: only whether a ray hits. BARE (bricks): t, the ids and the hit voxel's index only.
//   fetch(idle, n_idle, rank, i, exhausted): per lane, whether it takes a ray and which (rank: the lane's
//     place among the n_idle idle ones); called by all lanes, sets exhausted (wave-uniform) at the end
//   done(i, hit, voxel, again): per ended ray; again: the sequential walk must answer it. A triangle
//     hit's instId is its instance's block, an SDF hit's says which leaf (sdf_order).
// lds: 2 * WIDE_LDS_STACK * 64 words; keep: 6 * 64 words, for scenes of several instances only.
template <WideLeafKind LEAF, bool ANY, bool BARE, class Fetch, class Done>
__device__ __forceinline__ void wide_walk(const SceneView& s, const float4* __restrict__ pos,
                                          const float4* __restrict__ dir, wide_lds* lds, wide_lds* keep,
                                          uint32_t* spill, bool single, Fetch&& fetch, Done&& done) {
  constexpr int BLOCK = WIDE_BLOCK;
  constexpr bool TRI = LEAF == WIDE_TRI;
  const uint32_t lane = threadIdx.x;
  WideStack<BLOCK> st;
  st.col = lds + lane;
  st.spill = spill;
  wide_lds* kp = keep + lane;
  const uint4* __restrict__ blocks = reinterpret_cast<const uint4*>(s.wide);
  // the geometry of an SDF scene's only instance
  const uint32_t sdf_geom = TRI ? 0u : reinterpret_cast<const WideInstance*>(s.wide)->geom_id;
  const GeomRef sdf = TRI ? GeomRef{} : geom_ref(s, sdf_geom);
  const SdfSBSHeader header = LEAF == WIDE_BRICK ? s.sbs_headers[sdf.offset.x] : SdfSBSHeader{};
  const uint32_t v_size = header.brick_size + 2 * header.brick_pad + 1;
  const uint32_t mask_base = LEAF == WIDE_BRICK && s.sbs_mask ? s.sbs_mask_base[sdf.offset.x] : 0u;
  const uint32_t mask_stride = 1u + (header.brick_size * header.brick_size * header.brick_size + 31u) / 32u;

  uint32_t i = 0, cur = WIDE_DONE;
  float3 o = make3(0, 0, 0), d = make3(0, 0, 0), inv = make3(0, 0, 0);
  float tnear = 0.0f, tfar = 0.0f, limit = 0.0f, slop = 0.0f;
  CRT_Hit hit = miss_hit(0.0f);
  uint32_t voxel = 0;
  float entry = 0.0f;          // of the current instance (triangles), of the hit leaf (SDF)
  uint32_t inst_block = 0;     // block of the current instance
  int bottom = 0, floor_ = 0, top = 0;   // stack entries [bottom, top); those below floor_ are the instance level's
  bool unsure = false;         // the sequential walk could differ from this hit
  bool again = false;          // the sequential walk must answer this ray
  bool busy = false, inside = false;
  // a brick being marched: where the march is and ends, the brick's corner and size, the voxels stepped,
  // the brick's first data and mask words
  bool marching = false, at_surface = false;   // at_surface: waiting for the solve
  float march_t = 0.0f, march_end = 0.0f, brick_sz = 0.0f;
  float3 brick_min = make3(0, 0, 0);
  uint32_t steps = 0, data_offset = 0, mask_offset = 0;
  uint32_t holder = lane;      // lane that holds the ray
  uint32_t parts = 0;          // other lanes walking for this lane's ray
  bool first = true, exhausted = false;

  // Next place of the walk: the nearest unvisited child of the top entry, across the instance level.
  auto pop = [&]() {
    if (inside && top <= floor_) {
      inside = false;
      if (!single && top > bottom) {
        o = make3(__uint_as_float(kp[0]), __uint_as_float(kp[BLOCK]), __uint_as_float(kp[2 * BLOCK]));
        d = make3(__uint_as_float(kp[3 * BLOCK]), __uint_as_float(kp[4 * BLOCK]), __uint_as_float(kp[5 * BLOCK]));
        inv = safe_inverse(d);
      }
    }
    if (top <= bottom) {
      cur = WIDE_DONE;
      return;
    }
    const uint2 e = st.get(top - 1);
    const uint32_t slot = (e.y >> 12) & 7u;
    const uint32_t rest = (e.y >> 15) | (7u << 15);
    cur = wide_child(e.x, e.y, slot);
    if ((rest & 7u) == 7u) --top;
    else st.put_order(top - 1, (e.y & 0xFFFu) | (rest << 12));
  };
  auto stop = [&]() {
    cur = WIDE_DONE;
    bottom = top = floor_ = 0;
    inside = false;
  };

  // Whether the sequential walk meets a triangle before the hit triangle at the same distance ...
  auto tri_before = [&](uint32_t inst, uint32_t prim) -> bool {
    if (inst != hit.instId)
      return reinterpret_cast<const WideInstance*>(s.wide + inst)->rank <
             reinterpret_cast<const WideInstance*>(s.wide + hit.instId)->rank;
    return wide_before(s, pos[i], dir[i], inst, 0u, prim, hit.primId);
  };
  // ... and a hitting SDF leaf (with this box entry) before the hit's. A frame-octree leaf is given by its
  // `tex`, a brick by its block, here and in hit.instId.
  auto sdf_order = [&](uint32_t leaf) -> uint2 {   // rank, topmost overlapping pair
    if (LEAF == WIDE_FRAME) return uint2{leaf & ~WIDE_OVERLAP, (leaf & WIDE_OVERLAP) != 0u ? 0u : WIDE_NO_OVERLAP};
    const WideBrick* w = reinterpret_cast<const WideBrick*>(s.wide + leaf);
    return uint2{w->rank, w->overlap};
  };
  auto sdf_before = [&](float e, uint32_t leaf) -> bool {
    const uint2 a = sdf_order(leaf), b = sdf_order(hit.instId);
    const bool under = a.y != WIDE_NO_OVERLAP && a.y == b.y;
    if (!under && e != entry) return e < entry;
    return wide_before(s, pos[i], dir[i], 0u, under ? a.y : 0u, a.x, b.x);
  };
  // Boxes past the new hit no longer matter.
  auto narrow = [&]() {
    float reach = hit.t;
    if (!TRI) {
      reach = entry;
      if (!ANY) {
        const uint2 at = sdf_order(hit.instId);
        if (at.y != WIDE_NO_OVERLAP) reach = wide_reach(s, pos[i], dir[i], 0u, at.y, at.x, entry);
      }
      reach = fmaxf(reach, tnear);
    }
    limit = fminf(limit, wide_limit(reach, TRI ? slop : 0.0f));
  };

  for (;;) {
    const uint64_t ended = __ballot(busy && cur == WIDE_DONE);
    if (ended) {
      // ---- parts that ended: into the lanes that hold their rays ----
      uint64_t merge = __ballot(busy && cur == WIDE_DONE && holder != lane);
      if (holder != lane && cur == WIDE_DONE) busy = false;
      while (merge) {
        const int from = int(__ffsll((unsigned long long)merge)) - 1;
        merge &= merge - 1;
        const uint32_t to = __builtin_amdgcn_readlane(holder, from);
        auto lane_f = [&](float v) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), from)); };
        CRT_Hit h = miss_hit(0.0f);
        h.t = lane_f(hit.t);
        h.primId = __builtin_amdgcn_readlane(hit.primId, from);
        h.instId = __builtin_amdgcn_readlane(hit.instId, from);
        if (!TRI) h.geomId = __builtin_amdgcn_readlane(hit.geomId, from);
        if (!BARE) {
#pragma unroll
          for (int k = LEAF == WIDE_FRAME ? 2 : 0; k < (TRI ? 2 : 4); ++k) h.coords[k] = lane_f(hit.coords[k]);
          if (LEAF == WIDE_FRAME) h.coords[0] = 0.0f;
        }
        const uint32_t v = BARE ? __builtin_amdgcn_readlane(voxel, from) : 0u;
        const float e = TRI ? 0.0f : lane_f(entry);
        const uint32_t bits = __builtin_amdgcn_readlane((unsure ? 1u : 0u) | (again ? 2u : 0u), from);
        if (lane == to) {
          --parts;
          if (bits & 2u) again = true;
          if (h.primId != 0xFFFFFFFFu) {
            const bool doubt = (bits & 1u) != 0u;
            bool take = hit.primId == 0xFFFFFFFFu;
            if (take) {
              unsure = doubt;
            } else if (!ANY && TRI) {
              take = h.t < hit.t;
              if (take) {
                unsure = doubt;
              } else if (h.t == hit.t) {
                take = tri_before(h.instId, h.primId);
                unsure = unsure || doubt;
              }
            } else if (!ANY) {
              take = sdf_before(e, h.instId);
            }
            if (take) {
              hit = h;
              voxel = v;
              if (!TRI) entry = e;
              narrow();
            }
          }
          if (ANY && hit.primId != 0xFFFFFFFFu) {
            limit = -1.0f;   // ends the other parts
            marching = at_surface = false;
            stop();
          }
        }
      }
      // ---- rays that ended ----
      if (busy && cur == WIDE_DONE && parts == 0u) {
        busy = false;
        done(i, hit, voxel, again || unsure);
      }
    }
    const uint64_t idle = __ballot(!busy);
    const uint32_t n_idle = uint32_t(__popcll(idle));
    const uint32_t rank = uint32_t(__popcll(idle & ((1ull << lane) - 1ull)));
    if (!exhausted && (n_idle >= 16u || first)) {
      // ---- new rays ----
      first = false;
      const bool mine = fetch(!busy, n_idle, rank, i, exhausted);
      if (mine) {
        const float4 p = pos[i];
        float4 q = dir[i];
        if (ANY) q.w *= -1.0f;   // RayQuery_AnyHit flips the sign of w (BVH2Common.cpp:3394-3399)
        const bool first_hit = q.w <= 0.0f;
        if (first_hit) q.w *= -1.0f;
        o = xyz(p);
        d = xyz(q);
        tnear = p.w;
        tfar = q.w;
        busy = true;
        holder = lane;
        stop();
        hit = miss_hit(tfar);
        slop = 0.0f;
        if (TRI) {
          const float dmax = fmaxf(fmaxf(fabsf(d.x), fabsf(d.y)), fabsf(d.z));
          slop = 9.536743e-7f * (fabsf(o.x) + fabsf(o.y) + fabsf(o.z)) / dmax;
        }
        limit = wide_limit(tfar, slop);
        entry = 0.0f;
        unsure = false;
        again = !box_test_fast(o, d) || !(tnear >= 0.0f) || !(tfar >= 0.0f) || (TRI && !ANY && first_hit);
        if (!again) {
          inv = safe_inverse(d);
          cur = s.wide_root;
          if (!single) {
            kp[0] = __float_as_uint(o.x);
            kp[BLOCK] = __float_as_uint(o.y);
            kp[2 * BLOCK] = __float_as_uint(o.z);
            kp[3 * BLOCK] = __float_as_uint(d.x);
            kp[4 * BLOCK] = __float_as_uint(d.y);
            kp[5 * BLOCK] = __float_as_uint(d.z);
          }
        }
      }
      continue;   // rays that end at once are taken off before the walk
    }
    if (exhausted) {
      if (n_idle == uint32_t(BLOCK)) break;
      // ---- parts of rays for idle lanes ----
      const bool gives = busy && top > bottom;
      const uint64_t giving = __ballot(gives);
      if (n_idle >= WIDE_SHARE && giving) {
        const uint32_t give_rank = uint32_t(__popcll(giving & ((1ull << lane) - 1ull)));
        const uint32_t pairs = min(n_idle, uint32_t(__popcll(giving)));
        const bool takes = !busy && rank < pairs;
        // lane r learns the r-th taker
        const uint32_t taker = uint32_t(__builtin_amdgcn_ds_permute(int(takes ? rank : 63u) * 4, int(lane)));
        const uint32_t to_lane = __shfl(taker, int(give_rank), 64);
        // the giver leaves its oldest entry, the ray in that entry's space and what goes with it in the
        // taker's (empty) stack
        if (gives && give_rank < pairs) {
          wide_lds* to = (wide_lds*)(lds) + to_lane;
          const uint2 e = st.get(bottom);
          const bool local = inside && bottom >= floor_;
          ++bottom;
          to[0] = e.x;
          to[BLOCK] = e.y;
          to[2 * BLOCK] = local ? 1u : 0u;
          if (local || !inside) {
            to[3 * BLOCK] = __float_as_uint(o.x);
            to[4 * BLOCK] = __float_as_uint(o.y);
            to[5 * BLOCK] = __float_as_uint(o.z);
            to[6 * BLOCK] = __float_as_uint(d.x);
            to[7 * BLOCK] = __float_as_uint(d.y);
            to[8 * BLOCK] = __float_as_uint(d.z);
          } else {
            for (int k = 0; k < 6; ++k) to[(3 + k) * BLOCK] = kp[k * BLOCK];
          }
          to[9 * BLOCK] = __float_as_uint(tnear);
          to[10 * BLOCK] = __float_as_uint(tfar);
          to[11 * BLOCK] = __float_as_uint(limit);
          to[12 * BLOCK] = __float_as_uint(entry);
          to[13 * BLOCK] = inst_block;
          to[14 * BLOCK] = i;
          to[15 * BLOCK] = holder;
          to[16 * BLOCK] = __float_as_uint(slop);
        }
        __syncthreads();
        if (takes) {
          const wide_lds* c = st.col;
          inside = c[2 * BLOCK] != 0u;
          o = make3(__uint_as_float(c[3 * BLOCK]), __uint_as_float(c[4 * BLOCK]), __uint_as_float(c[5 * BLOCK]));
          d = make3(__uint_as_float(c[6 * BLOCK]), __uint_as_float(c[7 * BLOCK]), __uint_as_float(c[8 * BLOCK]));
          tnear = __uint_as_float(c[9 * BLOCK]);
          tfar = __uint_as_float(c[10 * BLOCK]);
          limit = __uint_as_float(c[11 * BLOCK]);
          entry = __uint_as_float(c[12 * BLOCK]);
          inst_block = c[13 * BLOCK];
          i = c[14 * BLOCK];
          holder = c[15 * BLOCK];
          slop = __uint_as_float(c[16 * BLOCK]);
          if (!single && !inside) {   // the world ray
            for (int k = 0; k < 6; ++k) kp[k * BLOCK] = c[(3 + k) * BLOCK];
          }
          busy = true;
          inv = safe_inverse(d);
          hit = miss_hit(tfar);
          unsure = again = false;
          bottom = floor_ = 0;
          top = 1;
        }
        // one more part for each holder
        uint64_t taken = __ballot(takes);
        while (taken) {
          const int t = int(__ffsll((unsigned long long)taken)) - 1;
          taken &= taken - 1;
          if (lane == __builtin_amdgcn_readlane(holder, t)) ++parts;
        }
        if (takes) pop();
      }
      // what the holder knows by now narrows its parts
      limit = fminf(limit, __shfl(limit, holder, 64));
      if (ANY && busy && limit < 0.0f) {
        marching = at_surface = false;
        stop();
      }
    }
    // ---- inner nodes ----
    for (;;) {
      const bool inner = (cur & WIDE_LEAF) == 0;
      if (inner) {
        const uint4* q = blocks + size_t(cur & WIDE_INDEX) * 4;
        const uint4 a = q[0], b = q[1], c = q[2], e = q[3];
        uint32_t key[6];
        wide_test(a, b, c, e, o, inv, tnear, limit, key);
        if (key[0] == 0xFFFFFFFFu) {
          pop();
        } else {
          const uint32_t rest = (key[1] & 7u) | ((key[2] & 7u) << 3) | ((key[3] & 7u) << 6) | ((key[4] & 7u) << 9) |
                                ((key[5] & 7u) << 12) | (7u << 15);
          if ((rest & 7u) != 7u) {
            st.put(top, e.y, (e.z & 0xFFFu) | (rest << 12));
            ++top;
          }
          cur = wide_child(e.y, e.z, key[0] & 7u);
        }
      }
      const uint32_t walking = uint32_t(__popcll(__ballot((cur & WIDE_LEAF) == 0)));
      const uint32_t working = uint32_t(__popcll(__ballot(cur != WIDE_DONE)));
      if (walking * (LEAF == WIDE_BRICK ? 4 : 2) <= working || working <= 48u) break;
    }
    // ---- leaves ----
    if ((cur & WIDE_LEAF) != 0 && cur != WIDE_DONE && !marching) {
      const uint4* q = blocks + size_t(cur & WIDE_INDEX) * 4;
      bool entered = false;
      if (!inside) {
        // an instance: its exact box, then the ray in its space
        const WideInstance* w = reinterpret_cast<const WideInstance*>(q);
        const float2 bh = ray_box2_fast(o, inv, w->boxMin, w->boxMax);
        if (bh.x <= bh.y && bh.y > tnear && bh.x < (ANY || !TRI ? tfar : limit)) {
          float3 lo, ld;
          wide_local_ray(w, o, d, lo, ld);
          inst_block = cur & WIDE_INDEX;
          if (TRI) entry = bh.x;
          entered = true;
          if (box_test_fast(lo, ld)) {
            cur = w->root;
            o = lo;
            d = ld;
            inv = safe_inverse(d);
            floor_ = top;
            inside = true;
          } else {   // the sequential walk answers
            again = true;
            stop();
          }
        }
      } else if (LEAF == WIDE_FRAME) {
        const float4* r = reinterpret_cast<const float4*>(q);
        const float4 r0 = r[0], r1 = r[1];
        const float2 tm = ray_box2_fast(o, inv, make3(r0.x, r0.y, r0.z), make3(r0.w, r1.x, r1.y));
        if (tm.x <= tm.y && tm.y >= tnear && tm.x <= fminf(tfar, limit)) {
          CRT_Hit h = miss_hit(tfar);
          const FrameLeaf* leaf = reinterpret_cast<const FrameLeaf*>(q);
          const uint32_t leaf_rank = leaf->tex;
          frame_leaf_intersect(s, sdf.type, leaf, o, d, fmax_ref(tnear, 0.01f), 0u, sdf_geom, h);
          if (h.t < tfar && (hit.primId == 0xFFFFFFFFu || (!ANY && sdf_before(tm.x, leaf_rank)))) {
            hit = h;
            hit.instId = leaf_rank;
            entry = tm.x;
            narrow();
          }
        }
      } else if (LEAF == WIDE_BRICK) {
        const WideBrick* leaf = reinterpret_cast<const WideBrick*>(q);
        const float2 tm = ray_box2_fast(o, inv, leaf->boxMin, leaf->boxMax);
        if (tm.x <= tm.y && tm.y >= tnear && tm.x <= fminf(tfar, limit)) {
          // the start of sbs_brick_intersect
          const SdfSBSNode node = leaf->node;
          brick_sz = float(node.pos_z_lod_size & 0x0000FFFF);
          const float sz_inv = 2.0f / brick_sz;
          brick_min = make3(-1, -1, -1) + sz_inv * make3(float(node.pos_xy >> 16), float(node.pos_xy & 0x0000FFFF),
                                                         float(node.pos_z_lod_size >> 16));
          const float2 nf = ray_box2(o, inv, brick_min, brick_min + sz_inv * make3(1, 1, 1));
          march_t = nf.x;
          march_end = nf.y;
          steps = 0;
          data_offset = node.data_offset;
          mask_offset = mask_base + leaf->prim * mask_stride;
          marching = s.sbs_mask == nullptr || s.sbs_mask[mask_offset] != 0u;   // a brick without surface cannot hit
          entered = marching;
        }
      } else {
        const uint32_t count = ((cur >> 26) & 3u) + 1u;
        const float tmin = fmax_ref(tnear, 0.01f);
        for (uint32_t j = 0; j < count; ++j, q += 4) {
          const float4* r = reinterpret_cast<const float4*>(q);
          const float4 ra = r[0], rb = r[1], rc = r[2];
          const float3 edge1 = xyz(rb) - xyz(ra);
          const float3 edge2 = xyz(rc) - xyz(ra);
          const float3 pvec = cross3(d, edge2);
          const float3 tvec = o - xyz(ra);
          const float3 qvec = cross3(tvec, edge1);
          const float invDet = 1.0f / dot3(edge1, pvec);
          const float v = dot3(tvec, pvec) * invDet;
          const float u = dot3(qvec, d) * invDet;
          const float t = dot3(edge2, qvec) * invDet;
          if (v >= -1e-6f && u >= -1e-6f && (u + v <= 1.0f + 1e-6f) && t > tmin && t <= hit.t) {
            const float4 rd = r[3];
            const float2 tm = ray_box2_fast(o, inv, make3(rb.w, rd.x, rd.z), make3(rc.w, rd.y, rd.w));
            if (tm.x <= tm.y && tm.y >= tnear && tm.x <= tfar && (t < hit.t || hit.primId != 0xFFFFFFFFu)) {
              const bool early = tm.x > t || entry >= t;   // before its own boxes: it could have been culled
              bool take = t < hit.t;
              if (!ANY && !take) {
                take = tri_before(inst_block, __float_as_uint(ra.w));
                unsure = unsure || early;
              } else {
                unsure = early;
              }
              if (take) {
                hit.t = t;
                hit.primId = __float_as_uint(ra.w);
                hit.instId = inst_block;
                hit.coords[0] = u;
                hit.coords[1] = v;
                narrow();
              }
            }
          }
        }
      }
      if (ANY && hit.primId != 0xFFFFFFFFu) {   // any hit will do
        unsure = false;
        limit = -1.0f;
        stop();
        entered = true;
      }
      if (!entered) pop();
    }
    if (LEAF == WIDE_BRICK) {
      // ---- bricks: sbs_brick_intersect's march, in two stages ----
      const float bs = float(header.brick_size), brick_d = 2.0f / (brick_sz * bs), scale = 0.5f * brick_sz * bs;
      const float hi = bs - 1e-6f;
      const uint32_t max_steps = 4 * header.brick_size + 8;
      float3 vox, vox_min;
      float2 nf;
      auto at_voxel = [&]() {   // the voxel at march_t
        const float3 local = ((o + march_t * d) - brick_min) * scale;
        vox = make3(floorf(clamp_ref(local.x, 1e-6f, hi)), floorf(clamp_ref(local.y, 1e-6f, hi)),
                    floorf(clamp_ref(local.z, 1e-6f, hi)));
        vox_min = brick_min + brick_d * vox;
        nf = ray_box2(o, inv, vox_min, vox_min + brick_d * make3(1, 1, 1));
      };
      auto voxel_index = [&]() {
        return (uint32_t(vox.x) * header.brick_size + uint32_t(vox.y)) * header.brick_size + uint32_t(vox.z);
      };
      if (marching && !at_surface) {   // to the next voxel with surface
        while (march_t < march_end && steps < max_steps) {
          steps++;
          at_voxel();
          at_surface = true;
          if (s.sbs_mask) {
            const uint32_t v = voxel_index();
            at_surface = ((s.sbs_mask[mask_offset + 1u + (v >> 5)] >> (v & 31u)) & 1u) != 0u;
          }
          if (at_surface) break;
          march_t += fmax_ref(0.0f, nf.y - march_t) + 1e-6f;
        }
        if (!at_surface) {
          marching = false;
          pop();
        }
      }
      // Solving the surface takes about a thousand vector instructions however few lanes do it, so lanes at
      // a surface voxel wait until a quarter of the working lanes do (8 x 256 x 256 rays, forward and
      // adjoint: 758 us; at once 896, at half 797, all 1,240: then the wave's solves follow its walks).
      const uint32_t waiting = uint32_t(__popcll(__ballot(at_surface)));
      const uint32_t working = uint32_t(__popcll(__ballot(cur != WIDE_DONE)));
      if (waiting * 4u >= working && at_surface) {
        at_surface = false;
        at_voxel();
        CRT_Hit h = miss_hit(tfar);
        const WideBrick* leaf = reinterpret_cast<const WideBrick*>(blocks + size_t(cur & WIDE_INDEX) * 4);
        float values[8];
        const float vmin = sbs_load_values_at(s, header, data_offset, vox, v_size, 2.0f / brick_sz, values);
        if (fmax_ref(tnear, 0.01f) < nf.x && vmin <= 0.0f) {
          const float3 start_q = ((o + nf.x * d) - vox_min) * scale;
          local_surface_intersection<false, !BARE>(s, sdf.type, d, 0u, sdf_geom, values, leaf->prim, brick_d, 0.0f,
                                                   (nf.y - nf.x) * scale, nf, start_q, h);
        }
        march_t += fmax_ref(0.0f, nf.y - march_t) + 1e-6f;
        const bool found = h.t < tfar;
        if (found) {
          const float2 tm = ray_box2_fast(o, inv, leaf->boxMin, leaf->boxMax);
          const uint32_t leaf_block = cur & WIDE_INDEX;
          if (hit.primId == 0xFFFFFFFFu || (!ANY && sdf_before(tm.x, leaf_block))) {
            if (!BARE) sbs_brick_coords(s, header, data_offset, v_size, brick_min, brick_sz, o, d, h);
            hit = h;
            hit.instId = leaf_block;
            voxel = voxel_index();
            entry = tm.x;
            narrow();
          }
        }
        if (found || !(march_t < march_end && steps < max_steps)) {
          marching = false;
          if (ANY && found) {
            limit = -1.0f;
            stop();
          } else {
            pop();
          }
        }
      }
    }
  }
}

}  // namespace lrt
