// Trace kernels for multi-octrees (leaf kinds LK_MULTI).
#include "trace_launch.h"
#include "wave_rays.h"

namespace lrt {
namespace {

// The default form for scenes of multi-octrees: persistent one-wave blocks whose lanes take a new ray when
// theirs has ended. A walk alternates node steps (about 150 vector instructions) and leaf solves (about a
// thousand), and a wave runs both for whichever lanes need them, so lanes wait at their next leaf until half
// of the walking lanes do and then solve together. A ray's own order of steps is the sequential walk's, so
// its record is, bit for bit.
// What bounds it: the chain of dependent steps of the rays that graze the most leaves. Octree of depth 8,
// 848 x 480 rays: 0.63 ms; whole walks in the one-ray-a-lane kernel 0.78 (3 waves a SIMD; here 4, which is
// what the stack's LDS allows); solved at once 0.75, at a quarter 0.70; the children's offset fetched from
// the node instead of being on the stack 0.69.
__global__ __launch_bounds__(WAVE_LANES, 4) void k_trace_multi(SceneView s, const float4* __restrict__ pos,
                                                              const float4* __restrict__ dir, CRT_Hit* __restrict__ out,
                                                              uint32_t* __restrict__ any_out, uint32_t n, uint32_t per_wave,
                                                              uint32_t turns, uint32_t* counter) {
  constexpr uint32_t END = 0xFFFFFFFEu;
  __shared__ uint32_t lds[2 * OT_LDS * WAVE_LANES];
  __shared__ uint32_t keep[6 * WAVE_LANES];   // the ray in its instance's space
  lds_u32* kp = (lds_u32*)(keep) + threadIdx.x;
  OTStack<WAVE_LANES> stack;
  stack.col = (lds_u32*)(lds) + threadIdx.x;
  WaveRays fetch{n, per_wave, turns, counter};
  const float lod_size = ot_lod_size(s);
  bool busy = false, at_leaf = false, found = false, exhausted = false;
  uint32_t i = 0, node = 0, inst = 0, root = 0, units = 0;   // node: the next one of the TLAS walk
  int top = -1;
  float tnear = 0.0f, best = 0.0f;
  OTRay r{};
  for (;;) {
    const uint64_t idle = __ballot(!busy);
    if (!exhausted && idle) {
      const uint32_t rank = uint32_t(__popcll(idle & ((1ull << threadIdx.x) - 1ull)));
      uint32_t k = 0;
      if (fetch(!busy, uint32_t(__popcll(idle)), rank, k, exhausted)) {
        i = k;
        busy = true;
        found = false;
        node = 0;
        tnear = pos[i].w;
        best = fabs_ref(dir[i].w);
      }
    }
    if (busy && top < 0) {
      // the TLAS walk (BVHRT::RayQuery_NearestHit) to the next instance whose boxes the ray hits
      float4 d = dir[i];
      if (any_out) d.w *= -1.0f;   // RayQuery_AnyHit flips the sign of w (BVH2Common.cpp:3394-3399)
      const float3 wp = xyz(pos[i]), wd = xyz(d);
      if (found && d.w <= 0.0f) node = END;   // the first hit ends the ray
      const float3 winv = safe_inverse(wd);
      while (node < END) {
        const BVHNode cur = load_node(s.tlas + node);
        const float2 bh = ray_box2(wp, winv, cur.boxMin, cur.boxMax);
        const bool is_leaf = (cur.leftOffset & LEAF_BIT) != 0;
        const bool hits = (bh.x <= bh.y) && (bh.y > tnear) && (bh.x < best);
        node = is_leaf || !hits ? cur.escapeIndex : cur.leftOffset;
        if (node == 0) node = END;
        if (!is_leaf || !hits) continue;
        inst = extract_start(cur.leftOffset);
        const InstanceData* in = s.instances + inst;
        float m[16];
        load_mat(in->transformInv, m);
        const float3 p = matmul4x3(m, wp), q = matmul3x3(m, wd), inv = safe_inverse(q);
        // the geometry's only pair: its box, and a small one beside it that leads to the same octree
        const GeomRef g = geom_ref(s, in->geomId);
        const BVHNodePair fat = load_pair(s.nodes + s.geoms[in->geomId].bvhOffset);
        const float2 t0 = ray_box2(p, inv, fat.left.boxMin, fat.left.boxMax);
        const float2 t1 = ray_box2(p, inv, fat.right.boxMin, fat.right.boxMax);
        const bool hit0 = (t0.x <= t0.y) && (t0.y >= tnear) && (t0.x <= best) && fat.left.leftOffset != LEAF_NORMAL;
        const bool hit1 = (t1.x <= t1.y) && (t1.y >= tnear) && (t1.x <= best) && fat.right.leftOffset != LEAF_NORMAL;
        if (!hit0 && !hit1) continue;
        kp[0 * WAVE_LANES] = __float_as_uint(p.x);
        kp[1 * WAVE_LANES] = __float_as_uint(p.y);
        kp[2 * WAVE_LANES] = __float_as_uint(p.z);
        kp[3 * WAVE_LANES] = __float_as_uint(q.x);
        kp[4 * WAVE_LANES] = __float_as_uint(q.y);
        kp[5 * WAVE_LANES] = __float_as_uint(q.z);
        r = ot_ray(p, q);
        top = 0;
        root = g.offset.x;
        stack.set(0, ot_root(s, root));
        break;
      }
      if (top < 0) {   // no more instances
        busy = false;
        if (!found && out) store_hit(out, i, miss_hit(fabs_ref(d.w)));
        if (any_out) any_out[i] = found ? 1u : 0u;
      }
    }
    const uint64_t walking = __ballot(busy && !at_leaf), waiting = __ballot(at_leaf);
    if ((walking | waiting) == 0) {
      if (exhausted) break;
      continue;
    }
    const float t_sdf = fmax_ref(tnear, 0.01f);
    if (__popcll(waiting) * 2 < __popcll(walking | waiting)) {
      if (busy && !at_leaf) at_leaf = ot_step(s, root, r, stack, top, t_sdf, lod_size, units);
    } else if (at_leaf) {
      at_leaf = false;
      const uint32_t geom = s.instances[inst].geomId;
      const float3 p = make3(__uint_as_float(kp[0 * WAVE_LANES]), __uint_as_float(kp[1 * WAVE_LANES]),
                             __uint_as_float(kp[2 * WAVE_LANES]));
      const float3 q = make3(__uint_as_float(kp[3 * WAVE_LANES]), __uint_as_float(kp[4 * WAVE_LANES]),
                             __uint_as_float(kp[5 * WAVE_LANES]));
      CRT_Hit hit = miss_hit(best);
      ot_solve(s, r, stack.get(top), root, p, q, t_sdf, inst, geom, hit, units);
      --top;
      if (hit.t < best) {   // the walk of an instance ends at its first leaf that is hit
        top = -1;
        best = hit.t;
        found = true;
        if (out) store_hit(out, i, hit);
      }
    }
  }
}

hipError_t launch_multi_default(const SceneView& s, const TraceArgs& a, hipStream_t stream) {
  static std::atomic<uint32_t> known[WAVE_DEVICES];
  uint32_t resident = 0;
  const hipError_t e = resident_blocks(k_trace_multi, known, &resident);
  if (e != hipSuccess) return e;
  const WaveShares w = wave_shares(a.n, resident);
  hipLaunchKernelGGL(k_trace_multi, dim3(w.grid), dim3(WAVE_LANES), 0, stream, s, a.pos, a.dir, a.out, a.any_out, a.n,
                     w.per_wave, w.turns, a.pcount);
  return hipGetLastError();
}

}  // namespace

// The one-ray-a-lane kernels answer counted calls and launch shapes that the caller chose.
hipError_t launch_trace_multi(const SceneView& s, const TraceArgs& a, hipStream_t stream) {
  if (takes_wide_form(s, a)) return launch_multi_default(s, a, stream);
  return launch_kinds<LK_MULTI>(s, a, stream);
}

}  // namespace lrt
