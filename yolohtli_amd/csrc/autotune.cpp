// autotune.cpp -- picks the plain-stepper kernel (tile shape x substep depth)
// by timing candidates on the plan's own state with HIP events.  Results are
// cached per (nx, ny, model, masked) for the life of the process.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "plan.h"

namespace {

using Key = std::tuple<int, int, int, int, int>;
std::mutex g_mu;
struct Choice {
  yh_kernel_cfg cfg;  // the fastest configuration
  float ms;
  bool split;  // YH_KERNEL_AUTO's launches are faster still, and ms their time
};
std::map<Key, Choice> g_cache;

std::vector<yh_kernel_cfg> candidates(const yh_plan* pl) {
  std::vector<yh_kernel_cfg> c;
  c.push_back({YH_KERNEL_DIRECT, 1, 0, 0, 1});
  const int kmax = std::min(pl->p.nx, pl->p.ny) - 1;
  // small grids (512^2 has 169 tiles of 64 x 64 on 256 CUs) favour
  // 4-wave regions and deeper fusion; large ones the 8- and 16-wave shapes
  const int Ks[] = {1, 2, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 16};
  const int shapes[][3] = {{4, 4, 1}, {8, 4, 1}, {16, 4, 1}, {4, 8, 1}, {8, 8, 1},
                           {4, 16, 1}, {5, 16, 1}, {8, 16, 1}, {16, 8, 1}, {7, 16, 1},
                           {4, 8, 2}, {8, 8, 2}, {4, 16, 2}};
  for (int K : Ks) {
    if (K > kmax) continue;
    for (auto& s : shapes) {
      const int rows = s[0], waves = s[1], cols = s[2];
      if (2 * K >= 64 * cols || 2 * K >= rows * waves) continue;
      if (!yh::tiled_supported(rows, waves, cols)) continue;
      if (pl->apd_on && !yh::tiled_apd_supported(rows, waves, cols)) continue;
      c.push_back({YH_KERNEL_TILED, K, rows, waves, cols});
    }
  }
  return c;
}

}  // namespace

using namespace yh;

extern "C" int yh_autotune(yh_plan* pl, int steps, void* stream, yh_kernel_cfg* best,
                           float* best_ms) {
  if (!pl || steps < 1) return YH_EINVAL;
  if (pl->p.solidSwitch && !pl->mask_set) return YH_ESTATE;
  if (plan_general(pl)) {  // one kernel shape: nothing to choose
    if (best) *best = pl->cfg;
    if (best_ms) *best_ms = -1.0f;
    return YH_OK;
  }
  hipStream_t s = (hipStream_t)stream;
  // Candidates are timed over whole calls of `steps` steps (at most 2000; a
  // longer call's remainder weighs nothing), repeated to at least 400 steps:
  // a call's remainder launch, or its merge into the last K-step launch,
  // counts, so the choice fits the call size the plan will be driven with
  // (20-step calls favour a K whose remainder merges over one a little
  // faster per step).
  const int call = std::min(steps, 2000);
  const int calls = std::max(1, (400 + call - 1) / call);
  const Key key{pl->p.nx, pl->p.ny, pl->p.model, pl->p.solidSwitch, call};
  {
    std::lock_guard<std::mutex> g(g_mu);
    auto it = g_cache.find(key);
    if (it != g_cache.end()) {
      pl->cfg = it->second.cfg;
      pl->split = it->second.split;
      if (best) *best = it->second.cfg;
      if (best_ms) *best_ms = it->second.ms;
      return YH_OK;
    }
  }
  // Save the state, run the candidates, restore.  Everything that can fail
  // is acquired before the plan is touched.
  const size_t bytes = pl->n * sizeof(float);
  float* save[3] = {nullptr, nullptr, nullptr};
  hipEvent_t e0 = nullptr, e1 = nullptr;
  hipError_t he = hipEventCreate(&e0);
  if (he == hipSuccess) he = hipEventCreate(&e1);
  for (int a = 0; a < pl->nv && he == hipSuccess; ++a) {
    he = hipMalloc(&save[a], bytes);
    if (he == hipSuccess)
      he = hipMemcpyAsync(save[a], pl->buf[pl->cur][a], bytes, hipMemcpyDeviceToDevice, s);
  }
  if (he != hipSuccess) {
    for (float* q : save)
      if (q) (void)hipFree(q);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    return hip_fail(he, "yh_autotune");
  }
  const int64_t count0 = pl->count;
  const bool prev0 = pl->have_prev;
  const yh_kernel_cfg cfg0 = pl->cfg;
  // The candidates run calls as the plan will, keeping u of the step before
  // the last when the plan does (the tip test's input), so their timing
  // counts that output, and the kernels the chosen configuration launches
  // (the previous-u and merged-remainder variants) are loaded and their
  // occupancy known before the caller's first call.
  const bool apd0 = pl->apd_on;  // the timed steps must not touch the APD state
  const bool split0 = pl->split;
  std::vector<yh_kernel_cfg> cands = candidates(pl);
  cands.push_back({YH_KERNEL_AUTO, 1, 0, 0, 1});
  pl->apd_on = false;
  pl->split = false;
  yh_kernel_cfg bestc = cfg0;
  float bestt = 1e30f, autot = 1e30f;
  int rc = YH_OK;
  for (const yh_kernel_cfg& c : cands) {
    pl->cfg = c;
    rc = plan_advance(pl, call, s);  // warm-up call (code object loads)
    if (rc) break;
    if (hipEventRecord(e0, s) != hipSuccess) { rc = YH_EHIP; break; }
    for (int i = 0; i < calls && !rc; ++i) rc = plan_advance(pl, call, s);
    if (rc) break;
    if (hipEventRecord(e1, s) != hipSuccess || hipEventSynchronize(e1) != hipSuccess) {
      rc = YH_EHIP;
      break;
    }
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    const float per_step = ms / ((float)calls * call);
    if (c.variant == YH_KERNEL_AUTO) {
      autot = per_step;
    } else if (per_step < bestt) {
      bestt = per_step;
      bestc = c;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  for (int a = 0; a < pl->nv; ++a) {
    (void)hipMemcpyAsync(pl->buf[pl->cur][a], save[a], bytes, hipMemcpyDeviceToDevice, s);
  }
  (void)hipStreamSynchronize(s);
  for (int a = 0; a < pl->nv; ++a) (void)hipFree(save[a]);
  pl->count = count0;
  pl->apd_on = apd0;
  (void)prev0;
  pl->have_prev = false;  // buf[cur^1] and prev_u hold a candidate's output
  pl->past_prev_u = false;
  if (rc) {
    pl->cfg = cfg0;
    pl->split = split0;
    return rc;
  }
  pl->cfg = bestc;
  // (of tiled configurations alone, whose results AUTO's equal bit for bit)
  pl->split = bestc.variant == YH_KERNEL_TILED && autot < bestt;
  const float ms = pl->split ? autot : bestt;
  {
    std::lock_guard<std::mutex> g(g_mu);
    g_cache[key] = {bestc, ms, pl->split};
  }
  if (best) *best = bestc;
  if (best_ms) *best_ms = ms;
  return YH_OK;
}
