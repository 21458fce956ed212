// How the persistent one-wave blocks of a kernel share a batch of rays.
#pragma once
#include <algorithm>
#include <atomic>

#include "kernels.h"

namespace lrt {

constexpr uint32_t WAVE_LANES = 64;
// Rays a counter hands out at once. Every fetch is an atomic, about 16 ns each on one address: with one
// counter, at 32 the 1024 x 1024 octree view takes 0.51 ms instead of 0.43, at 128 the last chunks are
// uneven (0.53).
constexpr uint32_t WAVE_CHUNK = 64;
// Neighbouring rays that start in one wave. Slow rays (silhouettes) are neighbours, and a wave steps
// through the sum of what its lanes wait for: 327,680 triangles, 512 x 512: 258 us in whole waves of
// neighbours, 210 in groups of 16, 186 in groups of 8.
constexpr uint32_t WAVE_GROUP = 8;

// A wave's rays: `per_wave` of its own come first (a power of two up to 64, in groups of at most WAVE_GROUP
// neighbours from distant parts of the batch), `turns` rounds of them (the later ones of 64, so that more than
// one takes per_wave 64), then chunks from a counter. Wave w uses counter w mod WAVE_COUNTERS, which has its
// own part of the rest: with one counter for all, a wave's fetches and its last, failing one queued up for
// 16 ns each (1100 x 900 rays into 500 triangles: 189 us, now 134; the octree view below 432, now 401).
struct WaveRays {
  uint32_t n, per_wave, turns;
  uint32_t* counter;                 // the wave's, 0 between calls
  uint32_t first = 0, rest = 0;      // its part of the batch
  uint32_t waves = 0;                // that share it
  uint32_t next = 0, end = 0, turn = 0;

  __device__ __forceinline__ WaveRays(uint32_t n_, uint32_t per_wave_, uint32_t turns_, uint32_t* counter_)
      : n(n_), per_wave(per_wave_), turns(turns_) {
    const uint32_t own = min(n, gridDim.x * per_wave * turns), left = n - own;
    const uint32_t counters = min(WAVE_COUNTERS, gridDim.x), c = blockIdx.x % counters;
    const uint32_t part = (left / counters + WAVE_CHUNK) / WAVE_CHUNK * WAVE_CHUNK;   // >= left / counters, whole chunks
    first = min(left, c * part);
    rest = min(left - first, part);
    first += own;
    waves = (gridDim.x - c + counters - 1) / counters;
    counter = counter_ + WAVE_COUNTER_AT + c * WAVE_COUNTER_WORDS;
  }

  // Called by all lanes of the wave. Whether the lane (idle, `rank` of the n_idle idle ones) gets a ray, in
  // i; sets `exhausted` (wave-uniform) when no more come.
  __device__ __forceinline__ bool operator()(bool idle, uint32_t n_idle, uint32_t rank, uint32_t& i, bool& exhausted) {
    const uint32_t lane = threadIdx.x, own = min(n, gridDim.x * per_wave * turns);
    if (turn == 0) {
      turn = 1;
      const uint32_t group = min(per_wave, WAVE_GROUP);
      if (n <= own && turns == 1) exhausted = true;
      i = (lane / group * gridDim.x + blockIdx.x) * group + lane % group;
      return lane < per_wave && i < own;
    }
    if (next == end && turn < turns) {
      next = (turn * gridDim.x + blockIdx.x) * WAVE_LANES;
      end = next + WAVE_LANES;
      ++turn;
    }
    if (next == end) {
      if (rest == 0) {
        exhausted = true;
        return false;
      }
      uint32_t got = 0;
      if (lane == 0) got = atomicAdd(counter, WAVE_CHUNK);
      got = __builtin_amdgcn_readfirstlane(got);
      if (got >= rest) {
        exhausted = true;
        // every wave of the counter ends on exactly one fetch past its rays; the one that sees the last
        // value of all clears it for the next call on this stream
        const uint32_t over = (rest + WAVE_CHUNK - 1) / WAVE_CHUNK * WAVE_CHUNK;
        if (lane == 0 && got == over + WAVE_CHUNK * (waves - 1)) atomicExch(counter, 0u);
        return false;
      }
      next = first + got;
      end = first + (rest - got < WAVE_CHUNK ? rest : got + WAVE_CHUNK);
    }
    const uint32_t count = min(n_idle, end - next);
    const bool mine = idle && rank < count;
    if (mine) i = next + rank;
    next += count;
    if (next == end && turn == turns && n <= own) exhausted = true;
    return mine;
  }
};

// The launch: as many waves as are resident at once (at most `most`) share the batch, down to one ray a wave.
struct WaveShares {
  uint32_t grid, per_wave, turns;
};

inline WaveShares wave_shares(uint32_t n, uint32_t most) {
  WaveShares w{0u, WAVE_LANES, 1u};
  while (w.per_wave > 1 && n / (w.per_wave / 2) < most) w.per_wave /= 2;
  w.grid = std::min((n + w.per_wave - 1) / w.per_wave, most);
  // Whole rounds of own rays while a quarter of the batch is left for the counter, which evens out what
  // the waves were dealt (1024 x 1024 octree view: 0.43 ms, all by the counter 0.49; 4 M bounce rays: 2.88
  // ms, none by the counter 3.5).
  if (w.per_wave == WAVE_LANES)
    w.turns = std::max(1u, uint32_t(uint64_t(n) * 3 / 4 / (uint64_t(w.grid) * w.per_wave)));
  return w;
}

// Blocks of a kernel of one-wave blocks that are resident on the current device at once (asked once per
// device; known: per kernel).
constexpr int WAVE_DEVICES = 64;
template <class K>
hipError_t resident_blocks(K kernel, std::atomic<uint32_t>* known, uint32_t* blocks) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  uint32_t r = dev < WAVE_DEVICES ? known[dev].load(std::memory_order_relaxed) : 0u;
  if (r == 0) {
    int per_cu = 0, cus = 0;
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(kernel), WAVE_LANES, 0);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    r = uint32_t(per_cu > 0 ? per_cu : 1) * uint32_t(cus > 0 ? cus : 1);
    if (dev < WAVE_DEVICES) known[dev].store(r, std::memory_order_relaxed);
  }
  *blocks = r;
  return hipSuccess;
}

}  // namespace lrt
