// batch.hip -- many tissues of uneven size and parameters in one launch.
//
// All tissues share one model and one mask mode; sizes, D and the ionic time
// constants vary per tissue.  The state of every tissue lives in one
// concatenated SoA allocation per variable (tissue t at offset off[t],
// 256-byte aligned).  A work list holds one item per (tissue, tile); the
// kernel k_batch walks it with a persistent grid-stride loop in which every
// XCD owns a contiguous range of items, and reads each item's KParams from a
// per-tissue table (uniform per workgroup, so they land in scalar registers).
// One launch advances every tissue by K steps; a whole run of many launches is
// captured once into a hipGraph and replayed.  yh_batch_step_each launches the
// single-tissue kernel once per tissue per chunk instead (the comparison).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <map>
#include <new>
#include <tuple>
#include <vector>

#include "plan.h"
#include "tile.h"

namespace yh {

struct BatchTissue {
  KParams k;
  unsigned long long off;
  int tiles_x;
  int pad;
};

// ISO = 1 when every tissue of the batch has isotropic diffusion (fixed at
// compile time, as in k_tiled), -1 to take each tissue's flag at run time.
template <int MODEL, bool MASKED, int R, int NW, int CW, int ISO>
__global__ __launch_bounds__(64 * NW) void k_batch(const BatchTissue* __restrict__ tissues,
                                                   const int2* __restrict__ items, int nitems,
                                                   CFields in, Fields out,
                                                   const uint8_t* __restrict__ codes, int K) {
  __shared__ TileLds<MODEL, NW, CW> lds;
  const int G = gridDim.x;
  int x = blockIdx.x & 7, local = blockIdx.x >> 3;
  // XCD x handles items [lo, hi) with its workgroups b = x, x+8, x+16, ...;
  // the XCDs with one workgroup more (the first G mod 8) also take the items
  // left over, so with a workgroup per item none runs two (bounds at
  // nitems*x/8 gave some a second item, and the launch twice the time, for
  // most item counts)
  int per_x = (G + 7 - x) >> 3;
  const int q = nitems >> 3, rem = nitems & 7;
  int lo = x * q + (x < rem ? x : rem);
  int hi = lo + q + (x < rem ? 1 : 0);
  if (G < 8) {  // too few workgroups to give every XCD one: plain striding
    local = blockIdx.x;
    per_x = G;
    lo = 0;
    hi = nitems;
  }
  for (int it = lo + local; it < hi; it += per_x) {
    const int2 item = items[it];
    const BatchTissue& T = tissues[item.x];
    const unsigned long long off = T.off;
    CFields ti{{in.f[0] + off, in.f[1] + off, in.f[2] ? in.f[2] + off : nullptr}};
    Fields to{{out.f[0] + off, out.f[1] + off, out.f[2] ? out.f[2] + off : nullptr}};
    const int ty = item.y / T.tiles_x;
    __syncthreads();  // the previous item's last reads of lds are done
    tile_advance<MODEL, MASKED, R, NW, CW, false, false, ISO>(
        T.k, ti, to, MASKED ? codes + off : nullptr, K, item.y - ty * T.tiles_x, ty, lds);
  }
}

template <int MODEL, bool MASKED, int R, int NW, int CW, int ISO>
static hipError_t launch_batch_t(int grid, const BatchTissue* t, const int2* items, int nitems,
                                 CFields in, Fields out, const uint8_t* codes, int K,
                                 hipStream_t s) {
  hipLaunchKernelGGL((k_batch<MODEL, MASKED, R, NW, CW, ISO>), dim3(grid), dim3(64 * NW), 0, s,
                     t, items, nitems, in, out, codes, K);
  return hipGetLastError();
}

template <int MODEL, bool MASKED, int R, int NW, int CW, int ISO>
static int max_resident(int* out) {
  int per_cu = 0;
  hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
      &per_cu, (const void*)k_batch<MODEL, MASKED, R, NW, CW, ISO>, 64 * NW, 0);
  if (e != hipSuccess) return hip_fail(e, "hipOccupancyMaxActiveBlocksPerMultiprocessor");
  int dev = 0, cus = 0;
  YH_HIP(hipGetDevice(&dev));
  YH_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  *out = std::max(1, per_cu) * cus;
  return YH_OK;
}

#define YH_BATCH_DISPATCH(FN, ...)                                                         \
  do {                                                                                     \
    if (model == M2V) {                                                                    \
      if (masked) { YH_BATCH_SHAPES(M2V, true, FN, __VA_ARGS__) }                          \
      else { YH_BATCH_SHAPES(M2V, false, FN, __VA_ARGS__) }                                \
    } else {                                                                               \
      if (masked) { YH_BATCH_SHAPES(MFK, true, FN, __VA_ARGS__) }                          \
      else { YH_BATCH_SHAPES(MFK, false, FN, __VA_ARGS__) }                                \
    }                                                                                      \
  } while (0)

#define YH_BATCH_ONE(M, MK, RR, WW, CC, FN, ...) \
  if (rows == RR && waves == WW && cols == CC) return FN<M, MK, RR, WW, CC, -1>(__VA_ARGS__);

// the default shape also comes with isotropic diffusion fixed at compile time
#define YH_BATCH_ISO(M, MK, RR, WW, CC, FN, ...)                  \
  if (rows == RR && waves == WW && cols == CC)                    \
    return iso ? FN<M, MK, RR, WW, CC, 1>(__VA_ARGS__)            \
               : FN<M, MK, RR, WW, CC, -1>(__VA_ARGS__);

#define YH_BATCH_SHAPES(M, MK, FN, ...)            \
  YH_BATCH_ISO(M, MK, 4, 8, 1, FN, __VA_ARGS__)   \
  YH_BATCH_ISO(M, MK, 8, 8, 1, FN, __VA_ARGS__)   \
  YH_BATCH_ISO(M, MK, 4, 16, 1, FN, __VA_ARGS__)  \
  YH_BATCH_ISO(M, MK, 8, 16, 1, FN, __VA_ARGS__)  \
  YH_BATCH_ONE(M, MK, 16, 8, 1, FN, __VA_ARGS__)  \
  YH_BATCH_ISO(M, MK, 7, 16, 1, FN, __VA_ARGS__)  \
  YH_BATCH_ONE(M, MK, 4, 8, 2, FN, __VA_ARGS__)   \
  YH_BATCH_ONE(M, MK, 8, 8, 2, FN, __VA_ARGS__)   \
  YH_BATCH_ONE(M, MK, 4, 16, 2, FN, __VA_ARGS__)

static bool batch_shape_ok(int rows, int waves, int cols) {
  return (cols == 1 && ((rows == 4 && (waves == 8 || waves == 16)) ||
                        (rows == 8 && (waves == 8 || waves == 16)) || (rows == 16 && waves == 8) ||
                        (rows == 7 && waves == 16))) ||
         (cols == 2 && ((rows == 4 && (waves == 8 || waves == 16)) || (rows == 8 && waves == 8)));
}

static hipError_t launch_batch(int model, bool masked, bool iso, int rows, int waves, int cols,
                               int grid, const BatchTissue* t, const int2* items, int nitems, CFields in,
                               Fields out, const uint8_t* codes, int K, hipStream_t s) {
  if (K < 1) return hipErrorInvalidValue;
  YH_BATCH_DISPATCH(launch_batch_t, grid, t, items, nitems, in, out, codes, K, s);
  return hipErrorInvalidValue;
}

static int batch_resident(int model, bool masked, bool iso, int rows, int waves, int cols,
                          int* out) {
  YH_BATCH_DISPATCH(max_resident, out);
  return YH_EINVAL;
}

}  // namespace yh

struct yh_batch {
  int nt = 0, model = 0, nv = 2;
  bool masked = false;
  bool iso = true;  // every tissue has isotropic diffusion
  std::vector<yh_params> p;
  std::vector<yh_derived> d;
  std::vector<yh::KParams> k;
  std::vector<size_t> off, ncell;
  size_t total = 0;
  float* buf[2][3] = {{nullptr, nullptr, nullptr}, {nullptr, nullptr, nullptr}};
  int cur = 0;
  uint8_t* solid_d = nullptr;
  uint8_t* codes_d = nullptr;
  std::vector<char> mask_set;
  // the configuration the autotuner picks for the 256-tissue workload; K is
  // capped at creation by the smallest tissue (reflected halos are exact for
  // at most min(nx, ny) - 1 substeps)
  yh_kernel_cfg cfg{YH_KERNEL_TILED, 6, 8, 8, 1};
  yh_kernel_cfg first{};  // cfg as created
  int persistent = 0;
  // until a kernel is set or tuned, calls may take other shapes and depths than
  // `first` (the same results) where an estimate of their time is lower; the
  // tuner may find that faster than cfg, the fastest kernel it timed
  bool free = true;
  yh::AutoTable table;
  double first_us[8];  // the same estimate of first's launches of 0 .. 6 steps
  bool use_graph = true;
  int64_t count = 0;
  // work lists: (K, rows, waves, cols) -> (tissue table, items, nitems).  Calls
  // of different sizes take different shapes at the same depth, so each pair
  // has its own list, and a list in use (by captured graphs, too) is never
  // replaced.
  struct WL {
    yh::BatchTissue* tissues = nullptr;
    int2* items = nullptr;
    int nitems = 0;
  };
  std::map<std::tuple<int, int, int, int>, WL> wl;
  // graph cache: (nsteps, cur, K, rows, waves, cols, persistent) -> exec
  std::map<std::tuple<int, int, int, int, int, int, int>, hipGraphExec_t> graphs;
  std::vector<hipGraph_t> graph_objs;
  hipStream_t cap_stream = nullptr;
};

namespace yh {

static void batch_clear_wl(yh_batch* b) {
  for (auto& kv : b->wl) {
    if (kv.second.tissues) (void)hipFree(kv.second.tissues);
    if (kv.second.items) (void)hipFree(kv.second.items);
  }
  b->wl.clear();
}

static void batch_clear_graphs(yh_batch* b) {
  for (auto& kv : b->graphs) (void)hipGraphExecDestroy(kv.second);
  for (auto g : b->graph_objs) (void)hipGraphDestroy(g);
  b->graphs.clear();
  b->graph_objs.clear();
}

static int batch_worklist(yh_batch* b, const yh_kernel_cfg& c, yh_batch::WL** out) {
  const int K = c.substeps;
  const auto key = std::make_tuple(K, c.rows, c.waves, c.cols);
  auto it = b->wl.find(key);
  if (it != b->wl.end()) {
    *out = &it->second;
    return YH_OK;
  }
  const int wout = 64 * c.cols - 2 * K, hout = c.rows * c.waves - 2 * K;
  if (wout <= 0 || hout <= 0) return YH_EINVAL;
  std::vector<BatchTissue> tab(b->nt);
  std::vector<int2> items;
  for (int t = 0; t < b->nt; ++t) {
    tab[t].k = b->k[t];
    tab[t].off = b->off[t];
    tab[t].tiles_x = (b->p[t].nx + wout - 1) / wout;
    tab[t].pad = 0;
    const int tiles_y = (b->p[t].ny + hout - 1) / hout;
    for (int q = 0; q < tab[t].tiles_x * tiles_y; ++q) items.push_back(make_int2(t, q));
  }
  yh_batch::WL w;
  w.nitems = (int)items.size();
  hipError_t e = hipMalloc(&w.tissues, sizeof(BatchTissue) * b->nt);
  if (e == hipSuccess) e = hipMalloc(&w.items, sizeof(int2) * items.size());
  if (e == hipSuccess)
    e = hipMemcpy(w.tissues, tab.data(), sizeof(BatchTissue) * b->nt, hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(w.items, items.data(), sizeof(int2) * items.size(), hipMemcpyHostToDevice);
  if (e != hipSuccess) {  // nothing half-built is kept
    if (w.tissues) (void)hipFree(w.tissues);
    if (w.items) (void)hipFree(w.items);
    return hip_fail(e, "batch work list");
  }
  *out = &b->wl.emplace(key, w).first->second;
  return YH_OK;
}

// Estimated time (us) of a launch, as the plan's tiled_time (plan.cpp) over the
// tiles of all tissues: the constants are fits to 960 timings of each kernel
// family on batches of 2 to 100 tissues of sides 64 to 768.  It compares depths
// of one shape well, and shapes that fill one round of workgroups; in several
// rounds the shapes overlap one workgroup's loads with another's substeps
// differently, which it does not know (24 masked FK tissues of 300 and 500:
// 7 x 16 at K=4 estimated 9% under 8 x 8 at K=6, measured 22% over).  So for
// several rounds the others are taken for a few steps only, mostly loads and
// stores, which it does know (120 tissues of 128, 2V, 3 steps: 17.7 us, 8 x 8
// 19.8): regions of 16 waves up to K=3, 4 x 8 up to K=5.  < 0: not taken.
static double batch_time(const yh_batch* b, int rows, int waves, int K, int cus, int resident) {
  static const double fit[2][2][4] = {
      // substep, row of a wave, issue, load and store
      {{0.175, 0.0134, 0.0111, 0.0067}, {0.205, 0.0, 0.0126, 0.0112}},   // 2V
      {{0.0, 0.0178, 0.0127, 0.0129}, {0.064, 0.0, 0.0150, 0.0187}}};    // FK
  const double* c = fit[b->model == M2V ? 0 : 1][b->masked ? 1 : 0];
  const int wout = 64 - 2 * K, H = rows * waves, hout = H - 2 * K;
  int64_t tiles = 0;
  for (const yh_params& p : b->p)
    tiles += (int64_t)((p.nx + wout - 1) / wout) * ((p.ny + hout - 1) / hout);
  const int64_t per_cu = std::max(1, resident / cus);
  const int64_t L = (tiles + cus - 1) / cus, q = (L + per_cu - 1) / per_cu;
  const int few = rows == 8 && waves == 8 ? 16 : waves == 8 ? 5 : 3;
  if (q > 1 && K > few) return -1.0;
  const double computed = (double)K * H - (double)K * (K + 1);
  return 4.2 + q * K * (c[0] + c[1] * rows) + L * (computed * c[2] + H * c[3]);
}

// Whether a call of n steps takes the table's launches rather than first's: while
// the batch is free, for an estimated gain of 3% (200 steps of 57 other batches
// of 2 to 32 tissues, 0.03 to 8 M cells: never slower, 16% faster in the mean; 2 to
// 40 steps of 38 more: 5% slower at most, 17% faster; a batch of a few small
// tissues twice as fast, since first was picked on 256).
static int batch_auto(yh_batch* b, int n, bool* wins) {
  *wins = false;
  if (!b->free) return YH_OK;
  const int K0 = b->first.substeps;
  if (!b->table.ready) {
    int dev = 0, cus = 0, rc = YH_OK, side = 1 << 30;
    YH_HIP(hipGetDevice(&dev));
    YH_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    auto us = [&](int rows, int waves, int K) {
      int res = 0;
      if (!batch_shape_ok(rows, waves, 1)) return -1.0;
      const int e = batch_resident(b->model, b->masked, b->iso, rows, waves, 1, &res);
      if (e) rc = e;
      return batch_time(b, rows, waves, K, std::max(1, cus), res);
    };
    for (const yh_params& p : b->p) side = std::min({side, p.nx, p.ny});
    b->table.fill(side - 1, us);
    for (int K = 1; K <= K0; ++K) b->first_us[K] = us(b->first.rows, b->first.waves, K);
    b->first_us[0] = 0.0;
    if (rc) {
      b->table.ready = false;
      return rc;
    }
  }
  *wins = b->table.of(n) < 0.97 * ((n / K0) * b->first_us[K0] + b->first_us[n % K0]);
  return YH_OK;
}

// The launch with `remaining` steps to go.
static yh_kernel_cfg batch_next(const yh_batch* b, bool table, int remaining) {
  yh_kernel_cfg c = table ? b->table.next(remaining) : b->free ? b->first : b->cfg;
  c.substeps = std::min(c.substeps, remaining);
  return c;
}

// The work lists of a call of nsteps (they allocate).
static int batch_lists(yh_batch* b, int nsteps, bool table) {
  for (int rem = nsteps; rem > 0;) {
    const yh_kernel_cfg c = batch_next(b, table, rem);
    yh_batch::WL* w = nullptr;
    const int rc = batch_worklist(b, c, &w);
    if (rc) return rc;
    rem -= c.substeps;
  }
  return YH_OK;
}

// Enqueue nsteps.
static int batch_enqueue(yh_batch* b, int nsteps, bool table, hipStream_t s) {
  int remaining = nsteps;
  while (remaining > 0) {
    const yh_kernel_cfg c = batch_next(b, table, remaining);
    yh_batch::WL* w = nullptr;
    int rc = batch_worklist(b, c, &w);
    if (rc) return rc;
    int grid = w->nitems;
    if (b->persistent && !b->free) {
      int res = 0;
      rc = batch_resident(b->model, b->masked, b->iso, c.rows, c.waves, c.cols, &res);
      if (rc) return rc;
      grid = std::min(grid, (res + 7) / 8 * 8);
    }
    const int bi = b->cur;
    CFields in{{b->buf[bi][0], b->buf[bi][1], b->buf[bi][2]}};
    Fields out{{b->buf[bi ^ 1][0], b->buf[bi ^ 1][1], b->buf[bi ^ 1][2]}};
    YH_HIP(launch_batch(b->model, b->masked, b->iso, c.rows, c.waves, c.cols, grid, w->tissues,
                        w->items, w->nitems, in, out, b->masked ? b->codes_d : nullptr,
                        c.substeps, s));
    b->cur ^= 1;
    remaining -= c.substeps;
  }
  return YH_OK;
}

static void batch_free(yh_batch* b) {
  if (!b) return;
  batch_clear_graphs(b);
  batch_clear_wl(b);
  for (int q = 0; q < 2; ++q)
    for (int a = 0; a < 3; ++a)
      if (b->buf[q][a]) (void)hipFree(b->buf[q][a]);
  if (b->solid_d) (void)hipFree(b->solid_d);
  if (b->codes_d) (void)hipFree(b->codes_d);
  if (b->cap_stream) (void)hipStreamDestroy(b->cap_stream);
  delete b;
}

}  // namespace yh

using namespace yh;

extern "C" {

int yh_batch_create(const yh_params* per_tissue, int ntissues, yh_batch** out) {
  if (!per_tissue || ntissues < 1 || !out) return YH_EINVAL;
  *out = nullptr;
  yh_batch* b = new (std::nothrow) yh_batch();
  if (!b) return YH_ENOMEM;
  b->nt = ntissues;
  b->model = per_tissue[0].model;
  b->masked = per_tissue[0].solidSwitch != 0;
  b->nv = nvars_of(b->model);
  size_t off = 0;
  for (int t = 0; t < ntissues; ++t) {
    const yh_params& p = per_tissue[t];
    if (p.model != b->model || (p.solidSwitch != 0) != b->masked || p.reduceSym) {
      batch_free(b);
      return YH_EINVAL;
    }
    if (!standard_branch(p)) {
      batch_free(b);
      return YH_EUNSUPPORTED;
    }
    yh_derived d;
    int rc = yh_params_derive(&p, &d);
    if (rc) {
      batch_free(b);
      return rc;
    }
    KParams k;
    make_kparams(p, d, &k);
    b->p.push_back(p);
    b->d.push_back(d);
    b->k.push_back(k);
    b->iso = b->iso && k.iso;
    b->off.push_back(off);
    const size_t n = (size_t)p.nx * p.ny;
    b->ncell.push_back(n);
    off += (n + 63) / 64 * 64;
  }
  b->total = off;
  b->mask_set.assign(ntissues, 0);
  for (int t = 0; t < ntissues; ++t)
    b->cfg.substeps = std::min(b->cfg.substeps, std::min(b->p[t].nx, b->p[t].ny) - 1);
  b->first = b->cfg;
  hipError_t e = hipSuccess;
  for (int q = 0; q < 2 && e == hipSuccess; ++q)
    for (int a = 0; a < b->nv && e == hipSuccess; ++a) {
      e = hipMalloc(&b->buf[q][a], sizeof(float) * b->total);
      if (e == hipSuccess) e = hipMemset(b->buf[q][a], 0, sizeof(float) * b->total);
    }
  if (e == hipSuccess && b->masked) {
    e = hipMalloc(&b->solid_d, b->total);
    if (e == hipSuccess) e = hipMalloc(&b->codes_d, b->total);
    if (e == hipSuccess) e = hipMemset(b->codes_d, 0x55, b->total);
  }
  if (e != hipSuccess) {
    int rc = hip_fail(e, "yh_batch_create");
    batch_free(b);
    return rc;
  }
  *out = b;
  return YH_OK;
}

void yh_batch_destroy(yh_batch* b) {
  if (b) (void)hipDeviceSynchronize();
  batch_free(b);
}

int yh_batch_size(const yh_batch* b, int* ntissues, int64_t* total_cells) {
  if (!b) return YH_EINVAL;
  if (ntissues) *ntissues = b->nt;
  if (total_cells) {
    int64_t s = 0;
    for (size_t n : b->ncell) s += (int64_t)n;
    *total_cells = s;
  }
  return YH_OK;
}

int yh_batch_set_mask(yh_batch* b, int t, const uint8_t* solid) {
  if (!b || t < 0 || t >= b->nt || !solid) return YH_EINVAL;
  if (!b->masked) return YH_ESTATE;
  const size_t n = b->ncell[t];
  std::vector<uint8_t> m(n);
  for (size_t c = 0; c < n; ++c) m[c] = solid[c] ? 1 : 0;
  YH_HIP(hipDeviceSynchronize());
  YH_HIP(hipMemcpy(b->solid_d + b->off[t], m.data(), n, hipMemcpyHostToDevice));
  YH_HIP(launch_codes(b->solid_d + b->off[t], b->codes_d + b->off[t], b->p[t].nx, b->p[t].ny,
                      nullptr));
  YH_HIP(hipDeviceSynchronize());
  b->mask_set[t] = 1;
  return YH_OK;
}

int yh_batch_set_state(yh_batch* b, int t, const float* u, const float* v, const float* w) {
  if (!b || t < 0 || t >= b->nt || !u || !v || (b->nv == 3 && !w)) return YH_EINVAL;
  const float* src[3] = {u, v, w};
  YH_HIP(hipDeviceSynchronize());
  for (int a = 0; a < b->nv; ++a)
    YH_HIP(hipMemcpy(b->buf[b->cur][a] + b->off[t], src[a], sizeof(float) * b->ncell[t],
                     hipMemcpyHostToDevice));
  return YH_OK;
}

int yh_batch_get_state(yh_batch* b, int t, float* u, float* v, float* w) {
  if (!b || t < 0 || t >= b->nt || !u || !v || (b->nv == 3 && !w)) return YH_EINVAL;
  float* dst[3] = {u, v, w};
  YH_HIP(hipDeviceSynchronize());
  for (int a = 0; a < b->nv; ++a)
    YH_HIP(hipMemcpy(dst[a], b->buf[b->cur][a] + b->off[t], sizeof(float) * b->ncell[t],
                     hipMemcpyDeviceToHost));
  return YH_OK;
}

int yh_batch_set_kernel(yh_batch* b, const yh_kernel_cfg* cfg, int persistent) {
  if (!b || !cfg) return YH_EINVAL;
  if (cfg->variant != YH_KERNEL_TILED || !batch_shape_ok(cfg->rows, cfg->waves, cfg->cols))
    return YH_EINVAL;
  if (cfg->substeps < 1 || cfg->substeps > 16 || 2 * cfg->substeps >= 64 * cfg->cols ||
      2 * cfg->substeps >= cfg->rows * cfg->waves)
    return YH_EINVAL;
  for (int t = 0; t < b->nt; ++t)
    if (cfg->substeps > std::min(b->p[t].nx, b->p[t].ny) - 1) return YH_EINVAL;
  b->cfg = *cfg;
  b->persistent = persistent ? 1 : 0;
  b->free = false;
  return YH_OK;
}

int yh_batch_set_graph(yh_batch* b, int on) {
  if (!b) return YH_EINVAL;
  b->use_graph = on != 0;
  return YH_OK;
}

int yh_batch_step(yh_batch* b, int nsteps, void* stream) {
  if (!b || nsteps < 0) return YH_EINVAL;
  if (nsteps == 0) return YH_OK;
  if (b->masked)
    for (int t = 0; t < b->nt; ++t)
      if (!b->mask_set[t]) return YH_ESTATE;
  hipStream_t s = (hipStream_t)stream;
  bool table = false;
  int rc = batch_auto(b, nsteps, &table);
  if (rc) return rc;
  if (!b->use_graph) {
    rc = batch_enqueue(b, nsteps, table, s);
    if (rc) return rc;
    b->count += nsteps;
    return YH_OK;
  }
  // (a free batch's launches follow from the number of steps)
  const auto key =
      b->free ? std::make_tuple(nsteps, b->cur, 0, 0, 0, 0, 0)
              : std::make_tuple(nsteps, b->cur, b->cfg.substeps, b->cfg.rows, b->cfg.waves,
                                b->cfg.cols, b->persistent);
  auto it = b->graphs.find(key);
  int nlaunch = 0;
  for (int rem = nsteps; rem > 0; rem -= batch_next(b, table, rem).substeps) ++nlaunch;
  if (it == b->graphs.end()) {
    // build the work lists outside the capture
    rc = batch_lists(b, nsteps, table);
    if (rc) return rc;
    int res = 0;
    rc = batch_resident(b->model, b->masked, b->iso, b->cfg.rows, b->cfg.waves, b->cfg.cols,
                            &res);
    if (rc) return rc;
    if (!b->cap_stream) YH_HIP(hipStreamCreateWithFlags(&b->cap_stream, hipStreamNonBlocking));
    const int cur0 = b->cur;
    YH_HIP(hipStreamBeginCapture(b->cap_stream, hipStreamCaptureModeThreadLocal));
    rc = batch_enqueue(b, nsteps, table, b->cap_stream);
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(b->cap_stream, &g);
    b->cur = cur0;  // capture only recorded the launches
    if (rc) {
      if (g) (void)hipGraphDestroy(g);
      return rc;
    }
    YH_HIP(e);
    hipGraphExec_t ex = nullptr;
    YH_HIP(hipGraphInstantiate(&ex, g, nullptr, nullptr, 0));
    b->graph_objs.push_back(g);
    it = b->graphs.emplace(key, ex).first;
  }
  YH_HIP(hipGraphLaunch(it->second, s));
  if (nlaunch & 1) b->cur ^= 1;
  b->count += nsteps;
  return YH_OK;
}

int yh_batch_step_each(yh_batch* b, int nsteps, void* stream) {
  if (!b || nsteps < 0) return YH_EINVAL;
  if (b->masked)
    for (int t = 0; t < b->nt; ++t)
      if (!b->mask_set[t]) return YH_ESTATE;
  hipStream_t s = (hipStream_t)stream;
  const yh_kernel_cfg c = b->cfg;
  int remaining = nsteps;
  while (remaining > 0) {
    const int K = std::min(c.substeps, remaining);
    const int bi = b->cur;
    for (int t = 0; t < b->nt; ++t) {
      const size_t o = b->off[t];
      CFields in{{b->buf[bi][0] + o, b->buf[bi][1] + o, b->nv > 2 ? b->buf[bi][2] + o : nullptr}};
      Fields out{{b->buf[bi ^ 1][0] + o, b->buf[bi ^ 1][1] + o,
                  b->nv > 2 ? b->buf[bi ^ 1][2] + o : nullptr}};
      YH_HIP(launch_tiled(b->model, b->masked, c.rows, c.waves, c.cols, K, b->k[t], in, out,
                          b->masked ? b->codes_d + o : nullptr, s));
    }
    b->cur ^= 1;
    remaining -= K;
  }
  b->count += nsteps;
  return YH_OK;
}

int yh_batch_autotune(yh_batch* b, int steps, void* stream, yh_kernel_cfg* best, float* best_ms) {
  if (!b || steps < 1) return YH_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  // save the state
  std::vector<float*> save(b->nv, nullptr);
  for (int a = 0; a < b->nv; ++a) {
    YH_HIP(hipMalloc(&save[a], sizeof(float) * b->total));
    YH_HIP(hipMemcpyAsync(save[a], b->buf[b->cur][a], sizeof(float) * b->total,
                          hipMemcpyDeviceToDevice, s));
  }
  const yh_kernel_cfg cfg0 = b->cfg;
  const int pers0 = b->persistent;
  const bool graph0 = b->use_graph, free0 = b->free;
  const int64_t count0 = b->count;
  b->use_graph = false;
  hipEvent_t e0, e1;
  YH_HIP(hipEventCreate(&e0));
  YH_HIP(hipEventCreate(&e1));
  int minside = 1 << 30;
  for (int t = 0; t < b->nt; ++t) minside = std::min(minside, std::min(b->p[t].nx, b->p[t].ny));
  const int shapes[][3] = {{4, 8, 1}, {8, 8, 1}, {4, 16, 1}, {8, 16, 1}, {7, 16, 1},
                           {4, 8, 2}, {4, 16, 2}};
  const int Ks[] = {2, 4, 6, 8, 9, 10, 12};
  // The time of a step in whole calls of `steps` (64 steps and more of them), a
  // call's last launch included; the lists are made and the kernels have run
  // before.
  auto time_calls = [&](bool table, float* ms_per_step) {
    const int calls = (63 + steps) / steps;
    int r = batch_lists(b, steps, table);
    if (!r) r = batch_enqueue(b, std::min(steps, 256), table, s);
    if (r) return r;
    if (hipEventRecord(e0, s) != hipSuccess) return (int)YH_EHIP;
    for (int i = 0; i < calls && !r; ++i) r = batch_enqueue(b, steps, table, s);
    if (r) return r;
    if (hipEventRecord(e1, s) != hipSuccess || hipEventSynchronize(e1) != hipSuccess)
      return (int)YH_EHIP;
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    *ms_per_step = ms / ((float)calls * steps);
    return (int)YH_OK;
  };
  yh_kernel_cfg bestc = b->first;
  int bestp = 0;
  bool table = false;
  float bestt = 1e30f, freet = 1e30f;
  b->free = true;
  int rc = batch_auto(b, steps, &table);
  if (!rc) rc = time_calls(table, &freet);
  b->free = false;
  for (int K : Ks) {
    if (rc) break;
    if (K > minside - 1) continue;
    for (auto& sh : shapes) {
      if (rc) break;
      if (2 * K >= 64 * sh[2] || 2 * K >= sh[0] * sh[1]) continue;
      for (int pers = 0; pers < 2 && !rc; ++pers) {
        b->cfg = yh_kernel_cfg{YH_KERNEL_TILED, K, sh[0], sh[1], sh[2]};
        b->persistent = pers;
        float t = 0.f;
        rc = time_calls(false, &t);
        if (!rc && t < bestt) {
          bestt = t;
          bestc = b->cfg;
          bestp = pers;
        }
      }
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  for (int a = 0; a < b->nv; ++a)
    (void)hipMemcpyAsync(b->buf[b->cur][a], save[a], sizeof(float) * b->total,
                         hipMemcpyDeviceToDevice, s);
  // the candidates' lists go, and with them the graphs that point at lists,
  // once no stream runs one any more
  (void)hipDeviceSynchronize();
  batch_clear_graphs(b);
  batch_clear_wl(b);
  for (int a = 0; a < b->nv; ++a) (void)hipFree(save[a]);
  b->use_graph = graph0;
  b->count = count0;
  if (rc) {
    b->cfg = cfg0;
    b->persistent = pers0;
    b->free = free0;
    return rc;
  }
  b->cfg = bestc;
  b->persistent = bestp;
  b->free = freet <= bestt;
  if (best) *best = bestc;
  if (best_ms) *best_ms = std::min(freet, bestt);
  return YH_OK;
}

int yh_batch_get_kernel(const yh_batch* b, yh_kernel_cfg* cfg, int* persistent) {
  if (!b) return YH_EINVAL;
  if (cfg) *cfg = b->cfg;
  if (persistent) *persistent = b->persistent;
  return YH_OK;
}

}  // extern "C"
