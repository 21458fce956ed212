// The wide walk: closest-hit and any-hit rays over the six-wide quantised tree of wide_bvh.h, for scenes
// of triangle meshes and for one ordered frame octree.
//
// The binary walk's time is its chain of dependent 64-byte pair fetches and, on incoherent rays, the
// texture addresser that expands four 16-byte loads per pair and lane; a six-wide node is the same four
// loads and replaces about two and a half pairs. Children are visited nearest first; the ones left for
// later share one 8-byte stack entry per level (child base, sizes, order), so the stack is short enough
// to stay in LDS. What bounds it now: 2^22 rays leaving the surfaces of 4,096 instances keep the vector
// units and the texture addresser busy (2.7 ms; the two-pass binary walk 86 ms, the persistent binary
// walk 5.9 ms on a like scene); camera rays wait for the waves with the most grazing rays, about 2 us a
// step (327,680 triangles, 512 x 512: 177 us against 262; octree of depth 9, 1024 x 1024: 0.45 ms against
// 0.99); 1,000 rays take 33 us against 88.
//
// Results are the sequential walk's (traverse.h). The packed boxes and the widened slab test only let
// more leaves through. What the sequential walk finds is then decided with its own arithmetic:
//  * a triangle counts only if its ray passes the exact box tests of the triangle's binary leaf and of
//    its instance. Every box above contains these, and the slab test grows with its box (subtraction,
//    multiplication, min and max are monotonic), so the sequential walk's tests above pass with them.
//  * the nearest such triangle is the sequential answer whenever it lies behind its own box entries:
//    no earlier hit can then have culled it. If it does not (its t rounds below a box entry), the ray is
//    queued and walked again by the sequential kernel. So are rays the monotonic test does not cover
//    (zero or non-finite components, box_test_fast) and rays that stop at the sequential walk's first
//    hit. Of two triangles at one distance the first in the sequential order counts (wide_before).
//    What is left open: a triangle in front of its own boxes by more than wide_limit's slack that
//    another hit within that distance hides from this walk and not from the sequential one (none seen in
//    80 million rays between overlapping instances).
//  * a frame-octree walk ends at the first leaf that hits. Where a plane separates the two children of
//    every binary node (checked at commit), every ray passes the leaves in the order of their box
//    entries and the sequential walk visits them in that order, so the answer is the hitting leaf with
//    the smallest entry; two hitting leaves of one entry queue the ray.
#include <algorithm>
#include <atomic>

#include "kernels.h"
#include "traverse.h"
#include "wide_bvh.h"

namespace lrt {
namespace {

constexpr int WIDE_BLOCK = 64;
constexpr int WIDE_LDS_STACK = 12;   // entries in LDS; the deeper ones spill
constexpr int WIDE_DEVICES = 64;
// Rays the counter hands out at once. Every fetch is an atomic on one address, about 16 ns each: at 32
// the 1024 x 1024 octree view takes 0.51 ms instead of 0.43, at 128 the last chunks are uneven (0.53).
constexpr uint32_t WIDE_CHUNK = 64;
// Neighbouring rays that start in one wave. Slow rays (silhouettes) are neighbours, and a wave steps
// through the sum of what its lanes wait for: 327,680 triangles, 512 x 512: 258 us in whole waves of
// neighbours, 210 in groups of 16, 186 in groups of 8.
constexpr uint32_t WIDE_GROUP = 8;
// Idle lanes from which on parts of rays are handed over (8: 193 us in that case, 16: 186, 32: 186)
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

// Whether the sequential walk reaches triangle (inst_a, prim_a) before (inst_b, prim_b), two hits of one
// ray at the same distance: by the instances' order in the TLAS, or in one instance by the nearer-child
// rule of the binary node where their leaves part (prim indices grow from left to right; the device
// pairs hold the first index of their right side in right.escapeIndex). Rare: it reads what it needs.
__device__ __forceinline__ bool wide_before(const SceneView& s, const float4* pos, const float4* dir, uint32_t i,
                                            uint32_t inst_a, uint32_t prim_a, uint32_t inst_b, uint32_t prim_b) {
  const WideInstance* a = reinterpret_cast<const WideInstance*>(s.wide + inst_a);
  if (inst_a != inst_b) return a->rank < reinterpret_cast<const WideInstance*>(s.wide + inst_b)->rank;
  const float3 p = xyz(pos[i]), q = xyz(dir[i]);
  const float* m = a->inv;
  const float3 o = wide_transform(m, p, 1.0f), inv = safe_inverse(wide_transform(m, q, 0.0f));
  const uint32_t lo = prim_a < prim_b ? prim_a : prim_b, hi = prim_a < prim_b ? prim_b : prim_a;
  const BVHNodePair* nodes = s.nodes + s.geoms[a->geom_id].bvhOffset;
  uint32_t at = 0;
  for (int k = 0; k < STACK_SIZE; ++k) {   // such trees are no deeper
    const BVHNodePair* pair = nodes + at;
    const uint32_t split = pair->right.escapeIndex;
    uint32_t child;
    if (hi < split) child = pair->left.leftOffset;
    else if (lo >= split) child = pair->right.leftOffset;
    else {
      const float l = ray_box2_fast(o, inv, pair->left.boxMin, pair->left.boxMax).x;
      const float r = ray_box2_fast(o, inv, pair->right.boxMin, pair->right.boxMax).x;
      return (prim_a == lo) == (l <= r);
    }
    if (child & LEAF_BIT) break;
    at = child;
  }
  return prim_a == lo;   // one leaf, in order
}

// Persistent one-wave blocks. A lane whose ray has ended takes a new one (once a quarter of the wave is
// idle); when the rays run out, an idle lane takes the oldest stack entry of a busy one, that is the
// largest part of its ray still to walk, and walks it for that ray: the last rays of a batch, and all
// rays of a small one, are walked by many lanes each. The parts' results are merged by the lane that
// holds the ray. Inner nodes are stepped until half of the wave's working lanes stand at a leaf.
// FRAME: frame-octree leaves, else triangles. ANY: only whether a ray hits. `per_wave` rays of a wave's
// own come first (a power of two up to 64, in groups of at most WIDE_GROUP neighbours from distant parts
// of the batch), then chunks from the counter.
template <bool FRAME, bool ANY>
__global__ __launch_bounds__(WIDE_BLOCK, 5) void k_trace_wide(SceneView s, const float4* __restrict__ pos,
                                                           const float4* __restrict__ dir, CRT_Hit* __restrict__ out,
                                                           uint32_t* __restrict__ any_out, uint32_t n, uint32_t per_wave, uint32_t turns,
                                                           uint32_t* __restrict__ spill, uint32_t spill_stride,
                                                           uint32_t* counter, TailQueue* queue) {
  constexpr int BLOCK = WIDE_BLOCK;
  constexpr uint32_t KINDS = FRAME ? LK_FRAME : LK_TRI;
  __shared__ uint32_t lds[2 * WIDE_LDS_STACK * BLOCK];
  __shared__ uint32_t keep[6 * BLOCK];   // world ray of each lane while it is inside an instance
  static_assert(2 * WIDE_LDS_STACK >= 17, "a taker's stack holds what it is given");
  const uint32_t lane = threadIdx.x;
  WideStack<BLOCK> st;
  st.col = (wide_lds*)(lds) + lane;
  st.spill = spill + size_t(blockIdx.x * BLOCK + lane) * spill_stride;
  wide_lds* kp = (wide_lds*)(keep) + lane;
  const uint4* __restrict__ blocks = reinterpret_cast<const uint4*>(s.wide);
  const bool single = s.n_instances == 1;

  uint32_t i = 0, cur = WIDE_DONE;
  float3 o = make3(0, 0, 0), d = make3(0, 0, 0), inv = make3(0, 0, 0);
  float tnear = 0.0f, tfar = 0.0f, limit = 0.0f, slop = 0.0f;
  CRT_Hit hit = miss_hit(0.0f);
  float entry = 0.0f;          // of the current instance (triangles), of the hit leaf (frame octrees)
  uint32_t inst_block = 0;     // block of the current instance
  int bottom = 0, floor_ = 0, top = 0;   // stack entries [bottom, top); those below floor_ are the instance level's
  bool unsure = false;         // the sequential walk could differ from this hit
  bool again = false;          // the sequential walk must answer this ray
  bool busy = false, inside = false;
  uint32_t holder = lane;      // lane that holds the ray
  uint32_t parts = 0;          // other lanes walking for this lane's ray
  // the counter hands out the rays past the waves' own; an atomic on one address takes about 16 ns, so
  // a wave asks for a chunk at a time
  const uint32_t own = min(n, gridDim.x * per_wave * turns);
  uint32_t next = 0, end = 0, turn = 0;
  bool exhausted = false;

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
        CRT_Hit h = miss_hit(0.0f);
        h.t = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(hit.t), from));
        h.primId = __builtin_amdgcn_readlane(hit.primId, from);
        h.instId = __builtin_amdgcn_readlane(hit.instId, from);
        const uint32_t c0 = __builtin_amdgcn_readlane(__float_as_uint(FRAME ? hit.coords[2] : hit.coords[0]), from);
        const uint32_t c1 = __builtin_amdgcn_readlane(__float_as_uint(FRAME ? hit.coords[3] : hit.coords[1]), from);
        const float e = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(entry), from));
        const uint32_t bits = __builtin_amdgcn_readlane((unsure ? 1u : 0u) | (again ? 2u : 0u), from);
        const uint32_t geom = FRAME ? __builtin_amdgcn_readlane(hit.geomId, from) : 0u;
        if (lane == to) {
          --parts;
          if (bits & 2u) again = true;
          if (h.primId != 0xFFFFFFFFu) {
            const bool doubt = (bits & 1u) != 0u;
            bool take = hit.primId == 0xFFFFFFFFu || (FRAME ? e < entry : h.t < hit.t);
            if (take) {
              unsure = doubt;
            } else if (FRAME) {
              unsure = unsure || e == entry;
            } else if (!ANY && h.t == hit.t) {
              take = wide_before(s, pos, dir, i, h.instId, h.primId, hit.instId, hit.primId);
              unsure = unsure || doubt;
            }
            if (take) {
              hit.t = h.t;
              hit.primId = h.primId;
              hit.instId = h.instId;
              if (FRAME) {
                hit.geomId = geom;
                hit.coords[0] = hit.coords[1] = 0.0f;
                hit.coords[2] = __uint_as_float(c0);
                hit.coords[3] = __uint_as_float(c1);
                entry = e;
                limit = fminf(limit, wide_limit(fmaxf(e, tnear), 0.0f));
              } else {
                hit.coords[0] = __uint_as_float(c0);
                hit.coords[1] = __uint_as_float(c1);
                limit = fminf(limit, wide_limit(h.t, slop));
              }
            }
          }
          if (ANY && hit.primId != 0xFFFFFFFFu) {
            limit = -1.0f;   // ends the other parts
            stop();
          }
        }
      }
      // ---- rays that ended ----
      if (busy && cur == WIDE_DONE && parts == 0u) {
        busy = false;
        if (again || unsure) {
          queue->list[atomicAdd(&queue->count, 1u)] = i;
        } else if (ANY) {
          any_out[i] = hit.primId != 0xFFFFFFFFu ? 1u : 0u;
        } else {
          if (!FRAME && hit.primId != 0xFFFFFFFFu) {
            const WideInstance* w = reinterpret_cast<const WideInstance*>(s.wide + hit.instId);
            hit.instId = w->inst_id;
            hit.geomId = w->geom_id | (TYPE_MESH_TRIANGLE << SH_TYPE);
            hit.coords[2] = 0.0f;
            hit.coords[3] = 0.0f;
          }
          finish_hit<KINDS>(s, hit);
          store_hit(out, i, hit);
        }
      }
    }
    const uint64_t idle = __ballot(!busy);
    const uint32_t n_idle = uint32_t(__popcll(idle));
    const uint32_t rank = uint32_t(__popcll(idle & ((1ull << lane) - 1ull)));
    if (!exhausted && (n_idle >= 16u || turn == 0)) {
      // ---- new rays ----
      bool mine = false;
      if (turn == 0) {
        turn = 1;
        const uint32_t group = min(per_wave, WIDE_GROUP);
        i = (lane / group * gridDim.x + blockIdx.x) * group + lane % group;
        mine = lane < per_wave && i < own;
        if (n <= own && turns == 1) exhausted = true;
      } else {
        if (next == end && turn < turns) {
          next = (turn * gridDim.x + blockIdx.x) * BLOCK;
          end = next + BLOCK;
          ++turn;
        }
        if (next == end) {
          uint32_t got = 0;
          if (lane == 0) got = atomicAdd(counter, WIDE_CHUNK);
          got = __builtin_amdgcn_readfirstlane(got);
          const uint32_t rest = n - own;
          if (got >= rest) {
            exhausted = true;
            // every wave ends on exactly one fetch past the rays; the one that sees the last value of
            // all clears the counter for the next call on this stream
            const uint32_t over = (rest + WIDE_CHUNK - 1) / WIDE_CHUNK * WIDE_CHUNK;
            if (lane == 0 && got == over + WIDE_CHUNK * (gridDim.x - 1)) atomicExch(counter, 0u);
            continue;
          }
          next = own + got;
          end = rest - got < WIDE_CHUNK ? n : next + WIDE_CHUNK;
        }
        const uint32_t count = min(n_idle, end - next);
        if (!busy && rank < count) {
          i = next + rank;
          mine = true;
        }
        next += count;
        if (next == end && turn == turns && n <= own) exhausted = true;
      }
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
        if (!FRAME) {
          const float dmax = fmaxf(fmaxf(fabsf(d.x), fabsf(d.y)), fabsf(d.z));
          slop = 9.536743e-7f * (fabsf(o.x) + fabsf(o.y) + fabsf(o.z)) / dmax;
        }
        limit = wide_limit(tfar, slop);
        entry = 0.0f;
        unsure = false;
        again = !box_test_fast(o, d) || !(tnear >= 0.0f) || !(tfar >= 0.0f) || (!FRAME && !ANY && first_hit);
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
          if (!inside) {   // the world ray
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
      if (ANY && busy && limit < 0.0f) stop();
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
      if (walking * 2 <= working || working <= 48u) break;
    }
    // ---- leaves ----
    if ((cur & WIDE_LEAF) != 0 && cur != WIDE_DONE) {
      const uint4* q = blocks + size_t(cur & WIDE_INDEX) * 4;
      bool entered = false;
      if (!inside) {
        // an instance: its exact box, then the ray in its space
        const WideInstance* w = reinterpret_cast<const WideInstance*>(q);
        const float2 bh = ray_box2_fast(o, inv, w->boxMin, w->boxMax);
        if (bh.x <= bh.y && bh.y > tnear && bh.x < (ANY || FRAME ? tfar : limit)) {
          float m[12];
#pragma unroll
          for (int k = 0; k < 12; ++k) m[k] = w->inv[k];
          const float3 lo = wide_transform(m, o, 1.0f), ld = wide_transform(m, d, 0.0f);
          inst_block = cur & WIDE_INDEX;
          if (!FRAME) entry = bh.x;
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
      } else if (FRAME) {
        const float4* r = reinterpret_cast<const float4*>(q);
        const float4 r0 = r[0], r1 = r[1];
        const float2 tm = ray_box2_fast(o, inv, make3(r0.x, r0.y, r0.z), make3(r0.w, r1.x, r1.y));
        if (tm.x <= tm.y && tm.y >= tnear && tm.x <= tfar && !(hit.primId != 0xFFFFFFFFu && tm.x > entry)) {
          CRT_Hit h = miss_hit(tfar);
          const uint32_t geom = reinterpret_cast<const WideInstance*>(blocks)->geom_id;   // the only instance
          frame_leaf_intersect(s, s.geoms[geom].type, reinterpret_cast<const FrameLeaf*>(q), o, d, fmax_ref(tnear, 0.01f),
                               0u, geom, h);
          if (h.t < tfar) {
            if (hit.primId != 0xFFFFFFFFu && tm.x == entry) {
              unsure = true;
            } else {
              hit = h;
              entry = tm.x;
              limit = fminf(limit, wide_limit(fmaxf(entry, tnear), 0.0f));
              unsure = false;
            }
          }
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
                take = wide_before(s, pos, dir, i, inst_block, __float_as_uint(ra.w), hit.instId, hit.primId);
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
                limit = fminf(limit, wide_limit(t, slop));
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
  }
}

// The rays the wide walk queued, by the sequential walk.
template <bool FRAME>
__global__ __launch_bounds__(WIDE_BLOCK) void k_trace_queued(SceneView s, const float4* __restrict__ pos,
                                                             const float4* __restrict__ dir, CRT_Hit* __restrict__ out,
                                                             uint32_t* __restrict__ any_out, uint32_t* overflow_count,
                                                             uint32_t* __restrict__ spill, TailQueue* queue) {
  constexpr int BLOCK = WIDE_BLOCK, S = 16;
  constexpr uint32_t KINDS = FRAME ? LK_FRAME : LK_TRI;
  __shared__ uint32_t lds[S * BLOCK];
  __shared__ uint32_t keep[6 * BLOCK];
  // Wave w takes entries [64 w, 64 w + 64) and so on in steps of the grid; waves without entries (most,
  // mostly all) leave without touching the queue, the others count themselves out and the last clears it.
  const uint32_t total = __atomic_load_n(&queue->count, __ATOMIC_RELAXED);
  const uint32_t waves = min(gridDim.x, (total + BLOCK - 1) / BLOCK);
  if (blockIdx.x >= waves) return;
  for (uint32_t first = blockIdx.x * BLOCK; first < total; first += gridDim.x * BLOCK) {
    if (first + threadIdx.x < total) {
      const uint32_t i = queue->list[first + threadIdx.x];
      LaneStack<S, BLOCK> st;
      st.col = (lds_u32*)(lds) + threadIdx.x;
      st.spill = spill + size_t(blockIdx.x * BLOCK + threadIdx.x) * (STACK_SIZE - 8);
      uint32_t overflow = 0;
      const float4 p = pos[i];
      float4 d = dir[i];
      if (any_out) d.w *= -1.0f;   // RayQuery_AnyHit flips the sign of w (BVH2Common.cpp:3394-3399)
      RayCounts cnt{};
      bool aborted = false;
      CRT_Hit h;
      if (box_test_fast(xyz(p), xyz(d)))
        h = ray_query_nearest<KINDS, S, BLOCK, false, false, true>(s, p, d, st, overflow, cnt, nullptr, 0u, aborted,
                                                                   nullptr, (lds_u32*)(keep) + threadIdx.x);
      else
        h = ray_query_nearest<KINDS, S, BLOCK, false, false, false>(s, p, d, st, overflow, cnt, nullptr, 0u, aborted,
                                                                    nullptr, (lds_u32*)(keep) + threadIdx.x);
      if (out) store_hit(out, i, h);
      if (any_out) any_out[i] = (h.geomId != 0xFFFFFFFFu) ? 1u : 0u;
      if (overflow && overflow_count) atomicAdd(overflow_count, 1u);
    }
  }
  __syncthreads();
  if (threadIdx.x == 0 && atomicAdd(&queue->next, 1u) == waves - 1) {
    queue->count = 0;
    queue->next = 0;
  }
}

// One thread a block of the instance level that is a node: its planes, and the instances it holds.
__global__ void k_wide_refit(WideBlock* blocks, uint32_t n_blocks, const uint32_t* __restrict__ sources,
                             const BVHNode* __restrict__ tlas, const InstanceData* __restrict__ inst) {
  const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
  if (n_blocks == 0) {   // a single instance and no nodes
    WideInstance* w = reinterpret_cast<WideInstance*>(blocks);
    if (b == 0) *w = wide_instance(inst[0], 0u, w->root, w->rank);
    return;
  }
  if (b >= n_blocks) return;
  uint32_t src[WIDE_CHILDREN], n = 0;
  for (uint32_t k = 0; k < WIDE_CHILDREN; ++k) {
    src[k] = sources[b * WIDE_CHILDREN + k];
    if (src[k] != 0xFFFFFFFFu) n = k + 1;
  }
  if (n == 0) return;   // an instance
  WideNode* node = reinterpret_cast<WideNode*>(blocks + b);
  WideNode planes = *node;
  WideBox box[WIDE_CHILDREN];
  for (uint32_t k = 0; k < n; ++k) box[k] = WideBox{tlas[src[k]].boxMin, tlas[src[k]].boxMax};
  if (!wide_pack_planes(box, n, planes)) {
    // boxes that cannot be packed: infinite steps make every plane distance NaN, which passes
    planes.exponents = 0xFFFFFFu;
    for (uint32_t k = 0; k < 9; ++k) planes.planes[k] = 0u;
  }
  *node = planes;
  for (uint32_t k = 0; k < n; ++k) {
    const uint32_t ref = wide_child(planes.children, planes.sizes, k);
    if (!(ref & WIDE_LEAF)) continue;
    const uint32_t id = tlas[src[k]].leftOffset & START_MASK;
    WideInstance* w = reinterpret_cast<WideInstance*>(blocks + (ref & WIDE_INDEX));
    *w = wide_instance(inst[id], id, w->root, w->rank);
  }
}

// Blocks of a kernel that are resident on the current device at once (asked once per device).
template <class K>
hipError_t resident_blocks(K kernel, std::atomic<uint32_t>* known, uint32_t* blocks) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  uint32_t r = dev < WIDE_DEVICES ? known[dev].load(std::memory_order_relaxed) : 0u;
  if (r == 0) {
    int per_cu = 0, cus = 0;
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(kernel), WIDE_BLOCK, 0);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    r = uint32_t(per_cu > 0 ? per_cu : 1) * uint32_t(cus > 0 ? cus : 1);
    if (dev < WIDE_DEVICES) known[dev].store(r, std::memory_order_relaxed);
  }
  *blocks = r;
  return hipSuccess;
}

template <bool FRAME, bool ANY>
hipError_t launch_wide_t(const SceneView& s, const TraceArgs& a, hipStream_t stream) {
  static std::atomic<uint32_t> known[WIDE_DEVICES], known_queued[WIDE_DEVICES];
  const uint32_t waves = (a.n + WIDE_BLOCK - 1) / WIDE_BLOCK;
  uint32_t resident = 0, resident_queued = 0;
  hipError_t e = resident_blocks(k_trace_wide<FRAME, ANY>, known, &resident);
  if (e == hipSuccess) e = resident_blocks(k_trace_queued<FRAME>, known_queued, &resident_queued);
  if (e != hipSuccess) return e;
  // A wave's own rays: as many waves as fit at once share the batch, down to one ray a wave, whose other
  // lanes then walk parts of it. A tree of more levels than the LDS stack spills by lane of the grid.
  uint32_t most = resident, spill_stride = 0;
  if (s.wide_levels > uint32_t(WIDE_LDS_STACK)) {
    spill_stride = 2 * (s.wide_levels - WIDE_LDS_STACK);   // at most 56 words; the spill has 72 a ray
    most = uint32_t(std::min<uint64_t>(most, a.spill_words / (spill_stride * WIDE_BLOCK)));
  }
  uint32_t per_wave = WIDE_BLOCK;
  while (per_wave > 1 && a.n / (per_wave / 2) < most) per_wave /= 2;
  const uint32_t grid = std::min((a.n + per_wave - 1) / per_wave, most);
  // Whole rounds of own rays while a quarter of the batch is left for the counter, which evens out what
  // the waves were dealt (1024 x 1024 octree view: 0.43 ms, all by the counter 0.49; 4 M bounce rays: 2.88
  // ms, none by the counter 3.5).
  const uint32_t turns = std::max(1u, uint32_t(uint64_t(a.n) * 3 / 4 / (uint64_t(grid) * per_wave)));
  hipLaunchKernelGGL((k_trace_wide<FRAME, ANY>), dim3(grid), dim3(WIDE_BLOCK), 0, stream, s, a.pos, a.dir, a.out,
                     a.any_out, a.n, per_wave, turns, a.spill, spill_stride, a.pcount, a.queue);
  hipLaunchKernelGGL((k_trace_queued<FRAME>), dim3(std::min(waves, resident_queued)), dim3(WIDE_BLOCK), 0, stream, s,
                     a.pos, a.dir, a.out, a.any_out, a.overflow_count, a.spill, a.queue);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_trace_wide(const SceneView& s, const TraceArgs& a, hipStream_t stream) {
  const bool frame = s.leaf_kinds == LK_FRAME;
  if (a.any_out) return frame ? launch_wide_t<true, true>(s, a, stream) : launch_wide_t<false, true>(s, a, stream);
  return frame ? launch_wide_t<true, false>(s, a, stream) : launch_wide_t<false, false>(s, a, stream);
}

hipError_t launch_wide_refit(WideBlock* blocks, uint32_t n_blocks, const uint32_t* sources, const BVHNode* tlas,
                             const InstanceData* inst, hipStream_t stream) {
  const uint32_t n = n_blocks ? n_blocks : 1u;
  hipLaunchKernelGGL(k_wide_refit, dim3((n + 63) / 64), dim3(64), 0, stream, blocks, n_blocks, sources, tlas, inst);
  return hipGetLastError();
}

}  // namespace lrt
