#include "tune.h"

#include <algorithm>
#include <utility>
#include <vector>

namespace lrt {

namespace {

hipError_t time_one(const std::function<hipError_t(const TuneConfig&)>& launch, hipStream_t stream,
                    const TuneConfig& c, int reps, hipEvent_t e0, hipEvent_t e1, float* ms) {
  hipError_t e = launch(c);   // warm-up
  if (e != hipSuccess) return e;
  float best = 1e30f;
  for (int r = 0; r < reps; ++r) {
    if ((e = hipEventRecord(e0, stream)) != hipSuccess) return e;
    if ((e = launch(c)) != hipSuccess) return e;
    if ((e = hipEventRecord(e1, stream)) != hipSuccess) return e;
    if ((e = hipEventSynchronize(e1)) != hipSuccess) return e;
    float t = 0.0f;
    if ((e = hipEventElapsedTime(&t, e0, e1)) != hipSuccess) return e;
    if (t < best) best = t;
  }
  *ms = best;
  return hipSuccess;
}

bool same_config(const TuneConfig& a, const TuneConfig& b) {
  return a.block == b.block && a.lds_stack == b.lds_stack && a.xcd_remap == b.xcd_remap && a.budget == b.budget &&
         a.tail_waves == b.tail_waves && a.postpone == b.postpone && a.ray_groups == b.ray_groups &&
         a.persistent == b.persistent && a.wide == b.wide;
}

}  // namespace

hipError_t autotune(const std::function<hipError_t(const TuneConfig&)>& launch, hipStream_t stream,
                    const TuneConfig& start, bool tune_postpone, bool tune_wide, int reps, TuneResult* out) {
  hipEvent_t e0 = nullptr, e1 = nullptr;
  hipError_t e = hipEventCreate(&e0);
  if (e == hipSuccess) e = hipEventCreate(&e1);
  TuneResult r{start, 1e30f, 0};
  std::vector<std::pair<float, TuneConfig>> shapes;   // stage-1 results
  std::vector<std::pair<float, TuneConfig>> timed;    // every candidate
  auto consider = [&](const TuneConfig& c, bool stage1) -> hipError_t {
    float ms = 0.0f;
    hipError_t err = time_one(launch, stream, c, reps, e0, e1, &ms);
    if (err != hipSuccess) return err;
    r.tried++;
    timed.emplace_back(ms, c);
    if (stage1) shapes.emplace_back(ms, c);
    if (ms < r.best_ms) {
      r.best_ms = ms;
      r.best = c;
    }
    return hipSuccess;
  };
  const int n_postpone = tune_postpone ? 2 : 1;
  if (tune_wide && e == hipSuccess) {
    TuneConfig c = start;
    c.wide = 1;
    e = consider(c, false);
  }
  for (int pp = 0; pp < n_postpone && e == hipSuccess; ++pp) {
    for (uint32_t groups : {0u, 8u, 32u}) {
      for (int block : {64, 128, 256}) {
        for (int lds : {8, 16, 32}) {
          TuneConfig c = start;
          c.block = block;
          c.lds_stack = lds;
          c.budget = 0;
          c.ray_groups = groups;
          c.persistent = 0;
          c.wide = 0;
          if (tune_postpone) c.postpone = pp;
          if ((e = consider(c, true)) != hipSuccess) break;
          if (groups == 0) {   // the persistent kernel takes rays in order: no interleaving
            c.persistent = 1;
            if ((e = consider(c, false)) != hipSuccess) break;
          }
        }
        if (e != hipSuccess) break;
      }
      if (e != hipSuccess) break;
    }
  }
  // Stage 2 on the three fastest stage-1 shapes: the single-pass ranking of shapes is only a
  // guide once the slowest rays move to the second pass. Both leaf orders are tried again, as
  // the two-pass scheme changes which rays a postponed walk holds up.
  using Timed = std::pair<float, TuneConfig>;
  std::sort(shapes.begin(), shapes.end(), [](const Timed& a, const Timed& b) { return a.first < b.first; });
  std::vector<TuneConfig> tops;
  for (const auto& sh : shapes) {
    bool seen = false;
    for (const TuneConfig& t : tops)
      seen = seen || (t.block == sh.second.block && t.lds_stack == sh.second.lds_stack &&
                      t.ray_groups == sh.second.ray_groups);
    if (!seen) tops.push_back(sh.second);
    if (tops.size() == 3) break;
  }
  for (const TuneConfig& shape : tops) {
    for (int pp = 0; pp < n_postpone && e == hipSuccess; ++pp) {
      for (uint32_t budget : {32u, 48u, 64u, 80u, 96u, 112u, 128u, 192u}) {
        for (uint32_t waves : {1024u, 2048u}) {
          TuneConfig c = shape;
          c.budget = budget;
          c.tail_waves = waves;
          if (tune_postpone) c.postpone = pp;
          if ((e = consider(c, false)) != hipSuccess) break;
        }
        if (e != hipSuccess) break;
      }
    }
    if (e != hipSuccess) break;
  }
  // Stage 3: the fastest distinct candidates were each timed once, one after another, so clock
  // ramps and noise between their turns can decide the ranking. They are timed again in turns,
  // round after round (the first candidate rotating), and the lowest median wins.
  if (e == hipSuccess && !timed.empty()) {
    std::stable_sort(timed.begin(), timed.end(), [](const Timed& a, const Timed& b) { return a.first < b.first; });
    std::vector<TuneConfig> finalists;
    for (const auto& t : timed) {
      bool seen = false;
      for (const TuneConfig& f : finalists) seen = seen || same_config(f, t.second);
      if (!seen) finalists.push_back(t.second);
      if (finalists.size() == 4) break;
    }
    constexpr int kRounds = 7;
    std::vector<std::vector<float>> runs(finalists.size());
    for (int round = 0; round < kRounds && e == hipSuccess; ++round) {
      for (size_t k = 0; k < finalists.size() && e == hipSuccess; ++k) {
        const size_t i = (k + size_t(round)) % finalists.size();
        float ms = 0.0f;
        e = time_one(launch, stream, finalists[i], reps, e0, e1, &ms);
        runs[i].push_back(ms);
      }
    }
    if (e == hipSuccess) {
      float best = 1e30f;
      for (size_t i = 0; i < finalists.size(); ++i) {
        std::vector<float> v = runs[i];
        std::nth_element(v.begin(), v.begin() + v.size() / 2, v.end());
        if (v[v.size() / 2] < best) {
          best = v[v.size() / 2];
          r.best = finalists[i];
        }
      }
      r.best_ms = best;
    }
  }
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  if (e == hipSuccess) *out = r;
  return e;
}

}  // namespace lrt
