// The wide walk: closest-hit and any-hit rays over the six-wide quantised tree of wide_bvh.h, for scenes
// of triangle meshes and for one frame octree or sparse brick set.
//
// The binary walk's time is its chain of dependent 64-byte pair fetches and, on incoherent rays, the
// texture addresser that expands four 16-byte loads per pair and lane; a six-wide node is the same four
// loads and replaces about two and a half pairs. Children are visited nearest first; the ones left for
// later share one 8-byte stack entry per level (child base, sizes, order), so the stack is short enough
// to stay in LDS. What bounds it now: 2^22 rays leaving the surfaces of 4,096 instances keep the vector
// units and the texture addresser busy (2.7 ms; the two-pass binary walk 86 ms, the persistent binary
// walk 5.9 ms on a like scene); camera rays wait for the waves with the most grazing rays, about 2 us a
// step (327,680 triangles, 512 x 512: 177 us against 262; octree of depth 9, 1024 x 1024: 0.45 ms against
// 0.99); 1,000 rays take 33 us against 88. A brick set of 256^3 voxels, 800 x 600: 0.53 ms against 2.76
// (most rays graze bricks and were left to the second pass); there it is the surface solves, about a
// thousand vector instructions each (on average 17 of 64 lanes are active, the vector units busy a third of the
// time; the instanced rays keep them busy all the time at 22 lanes).
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
//    What is left open: a triangle in front of its own boxes by more than wide_limit's slack that another
//    hit hides from this walk and not from the sequential one. That takes a ray in the triangle's plane to
//    within rounding, whose computed distance is noise. Of 400,000 rays made to lie in the planes of 300 to
//    30,000 overlapping triangles 9 to 76 records differ, tilted by 1e-7 7 to 39, by 1e-5 none or one (the
//    two-pass binary walk: 205 to 316, 117 to 182, 1 to 5); none of 80 million rays between overlapping
//    instances, nor of 600,000 into chains of triangles down to 1e-31 across.
//  * an SDF walk ends at the first leaf that hits. Where a plane separates the two children of a binary
//    node, every ray passes the leaves of one side before the other's and the sequential walk visits them
//    in that order, so the answer is the hitting leaf with the smallest box entry. Two leaves of one
//    entry, or below one node whose sides overlap (coarse bricks beside fine ones: a fifth of the leaves
//    of such a set), are compared by the sequential walk's rule at the node where they part
//    (wide_before), and the walk goes on past the hit's entry as far as such a leaf can begin
//    (wide_reach).
#include "wave_rays.h"
#include "wide_walk.h"

namespace lrt {
namespace {

// Leaf kinds of the sequential walk that answers a kernel's queued rays.
constexpr uint32_t wide_kinds(WideLeafKind leaf) { return leaf == WIDE_TRI ? LK_TRI : (leaf == WIDE_FRAME ? LK_FRAME : LK_SBS); }

template <WideLeafKind LEAF, bool ANY>
__global__ __launch_bounds__(WIDE_BLOCK, LEAF == WIDE_BRICK ? 4 : 5) void k_trace_wide(
    SceneView s, const float4* __restrict__ pos, const float4* __restrict__ dir, CRT_Hit* __restrict__ out,
    uint32_t* __restrict__ any_out, uint32_t n, uint32_t per_wave, uint32_t turns, uint32_t* __restrict__ spill,
    uint32_t spill_stride, uint32_t* counter, TailQueue* queue) {
  constexpr int BLOCK = WIDE_BLOCK;
  __shared__ uint32_t lds[2 * WIDE_LDS_STACK * BLOCK];
  __shared__ uint32_t keep[LEAF == WIDE_TRI ? 6 * BLOCK : 1];   // world ray of each lane while it is inside an instance
  const uint32_t lane = threadIdx.x;
  WaveRays fetch{n, per_wave, turns, counter};
  auto done = [&](uint32_t i, CRT_Hit& hit, uint32_t, bool again) {
    if (again) {
      queue->list[atomicAdd(&queue->count, 1u)] = i;
    } else if (ANY) {
      any_out[i] = hit.primId != 0xFFFFFFFFu ? 1u : 0u;
    } else {
      if (hit.primId != 0xFFFFFFFFu) {
        if (LEAF == WIDE_TRI) {
          const WideInstance* w = reinterpret_cast<const WideInstance*>(s.wide + hit.instId);
          hit.instId = w->inst_id;
          hit.geomId = w->geom_id | (TYPE_MESH_TRIANGLE << SH_TYPE);
          hit.coords[2] = 0.0f;
          hit.coords[3] = 0.0f;
        } else {
          hit.instId = 0u;
        }
      }
      finish_hit<wide_kinds(LEAF)>(s, hit);
      store_hit(out, i, hit);
    }
  };
  wide_walk<LEAF, ANY, ANY && LEAF == WIDE_BRICK>(s, pos, dir, (wide_lds*)(lds), (wide_lds*)(keep),
                                                  spill + size_t(blockIdx.x * BLOCK + lane) * spill_stride,
                                                  LEAF != WIDE_TRI || s.n_instances == 1, fetch, done);
}

// The rays the wide walk queued, by the sequential walk.
template <WideLeafKind LEAF>
__global__ __launch_bounds__(WIDE_BLOCK) void k_trace_queued(SceneView s, const float4* __restrict__ pos,
                                                             const float4* __restrict__ dir, CRT_Hit* __restrict__ out,
                                                             uint32_t* __restrict__ any_out, uint32_t* overflow_count,
                                                             uint32_t* __restrict__ spill, TailQueue* queue) {
  constexpr int BLOCK = WIDE_BLOCK, S = 16;
  constexpr uint32_t KINDS = wide_kinds(LEAF);
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

template <WideLeafKind LEAF, bool ANY>
hipError_t launch_wide_t(const SceneView& s, const TraceArgs& a, hipStream_t stream) {
  static std::atomic<uint32_t> known[WAVE_DEVICES], known_queued[WAVE_DEVICES];
  const uint32_t waves = (a.n + WIDE_BLOCK - 1) / WIDE_BLOCK;
  uint32_t resident = 0, resident_queued = 0;
  hipError_t e = resident_blocks(k_trace_wide<LEAF, ANY>, known, &resident);
  if (e == hipSuccess) e = resident_blocks(k_trace_queued<LEAF>, known_queued, &resident_queued);
  if (e != hipSuccess) return e;
  // Lanes without a ray walk parts of the others. A tree of more levels than the LDS stack spills by lane of
  // the grid.
  uint32_t most = resident, spill_stride = 0;
  if (s.wide_levels > uint32_t(WIDE_LDS_STACK)) {
    spill_stride = 2 * (s.wide_levels - WIDE_LDS_STACK);   // at most 56 words; the spill has 72 a ray
    most = uint32_t(std::min<uint64_t>(most, a.spill_words / (spill_stride * WIDE_BLOCK)));
  }
  const WaveShares w = wave_shares(a.n, most);
  hipLaunchKernelGGL((k_trace_wide<LEAF, ANY>), dim3(w.grid), dim3(WIDE_BLOCK), 0, stream, s, a.pos, a.dir, a.out,
                     a.any_out, a.n, w.per_wave, w.turns, a.spill, spill_stride, a.pcount, a.queue);
  hipLaunchKernelGGL((k_trace_queued<LEAF>), dim3(std::min(waves, resident_queued)), dim3(WIDE_BLOCK), 0, stream, s,
                     a.pos, a.dir, a.out, a.any_out, a.overflow_count, a.spill, a.queue);
  return hipGetLastError();
}

template <WideLeafKind LEAF>
hipError_t launch_wide_leaf(const SceneView& s, const TraceArgs& a, hipStream_t stream) {
  return a.any_out ? launch_wide_t<LEAF, true>(s, a, stream) : launch_wide_t<LEAF, false>(s, a, stream);
}

}  // namespace

hipError_t launch_trace_wide(const SceneView& s, const TraceArgs& a, hipStream_t stream) {
  switch (s.leaf_kinds) {
    case LK_TRI: return launch_wide_leaf<WIDE_TRI>(s, a, stream);
    case LK_FRAME: return launch_wide_leaf<WIDE_FRAME>(s, a, stream);
    case LK_SBS: return launch_wide_leaf<WIDE_BRICK>(s, a, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_wide_refit(WideBlock* blocks, uint32_t n_blocks, const uint32_t* sources, const BVHNode* tlas,
                             const InstanceData* inst, hipStream_t stream) {
  const uint32_t n = n_blocks ? n_blocks : 1u;
  hipLaunchKernelGGL(k_wide_refit, dim3((n + 63) / 64), dim3(64), 0, stream, blocks, n_blocks, sources, tlas, inst);
  return hipGetLastError();
}

}  // namespace lrt
