// adjoint.hip -- gradient of a sensor-mismatch loss through the FK stepper.
//
// Forward (no reference counterpart; the reference has no gradient path):
//   u' = m*(u + tc*(L_D u - dt*I(u,v,w))),  v' = m*(v - tc*dt*G_v),  w' = ...
//   L_D u = dt/hx^2 sum_{W,E} c*0.5*(D_c + D_n)*(u_n - u) + (same in y)
// with the mask coefficients c in {0,1,2} of reactionDiffusion.cu:162-169,
// the mirror neighbours of coord_i/coord_j (helper_functions.cu:69-79), and
// the Fenton-Karma currents with the Heaviside smoothed to
// 0.5*(1 + tanh(x/w)) so the loss is differentiable.
// Loss = sum over recorded steps n (n % rec == 0) and sensors s of
// (u^n(s) - target)^2.
//
// Reverse: lambda^n = J(X^n)^T lambda^{n+1} + dL/dX^n, gD += (dF/dD)^T
// lambda^{n+1}, gtau += (dF/dtau)^T lambda^{n+1}.  The transpose of the
// mirrored, masked operator is applied in gather form: cell j collects the
// coefficient of every (cell c, direction) whose neighbour is j, including the
// two mirror images at each edge.  The forward keeps every state where they
// fit in 4 GiB; a longer run keeps a checkpoint every `ckpt` steps, and each
// segment is recomputed into a buffer before its reverse sweep.  gD and gtau
// accumulate in FP64 (gtau per workgroup, in a fixed order, so results are
// deterministic).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <vector>

#include "lanes.h"
#include "plan.h"
#include "tile.h"

namespace yh {

struct AdjK {
  int nx, ny;
  float rxt, ryt;  // tc dt / (2 hx^2), tc dt / (2 hy^2)
  float tdt;       // tc dt
  float uc, uv, ucsi, uc1;  // uc1 = 1 + u_c
  float tv1m, tv2m, dtv;    // tau_v1-, tau_v2-, tau_v2- - tau_v1-
  // rounded once on the host from FP64: 2/(w ln 2) and 2k/ln 2 (sigmoid2's
  // exponents), 2/w, 1/tau_d, 1/tau_r, 1/tau_si, 2k/tau_si, 1/tau_0, 1/tau_v+,
  // 1/tau_w-, 1/tau_w+
  float eh, es, tihw, itd, itr, itsi, ksi, it0, itvp, itwm, itwp;
};

// Currents and gate rates of a cell (dv/dt = A, dw/dt = B), their derivatives
// (of -A and -B), and the products that both share with the time constants'.
struct FkEval {
  float I, A, B;
  float Iu, Iv, Iw, Gvu, Gvv, Gwu, Gww;
  float p, vpf, ws, upc, vp, pw;
};

// Correctly rounded 1/t: the hardware reciprocal (within 1 ulp) and one
// Newton step by its exact residual (Markstein, IBM J. Res. Dev. 34(1), 1990;
// equal to the quotient 1.0f/t for every significand), 3 instructions for 11;
// t must be normal and 1/t as well.
__device__ __forceinline__ float recip(float t) {
  const float r = __builtin_amdgcn_rcpf(t);
  return __builtin_fmaf(__builtin_fmaf(-t, r, 1.0f), r, r);
}

// s = sigmoid(e ln 2 x) = 0.5*(1 + tanh(e ln 2 x/2)) and its complement
// sc = 1 - s, both from a = exp2(-e|x|) in (0, 1] with the hardware exp2 and
// reciprocal: the larger is 1/(1 + a), the smaller a/(1 + a), so each keeps a
// relative error of a few ulp (1 - 2/(exp(2y) + 1) loses the smaller one, and
// 1 - tanh^2, to cancellation: 2e-3 relative at tanh's argument 5).
__device__ __forceinline__ void sigmoid2(float x, float e, float* s, float* sc) {
#pragma clang fp contract(off)
  const float a = __builtin_amdgcn_exp2f(-e * __builtin_fabsf(x));
  const float big = __builtin_amdgcn_rcpf(1.0f + a);
  const float small = a * big;
  *s = x >= 0.0f ? big : small;
  *sc = x >= 0.0f ? small : big;
}

// Fenton & Karma 1998 currents and derivatives with the Heaviside smoothed to
// p = 0.5*(1 + tanh((u - u_c)/w)) (q at u_v), p' = (2/w) p (1 - p).  Every fma
// is written out and contraction is off, here and in what is built on it, so
// the kernels that inline them agree bit for bit.  A step is bound by VALU
// issue, so the sums share their products and constants are folded: a reverse
// step takes about 115 instructions in a ring cell and 155 in a tile cell, 165
// and 290 with the formulas as they stand and every operation rounded.  The
// gradients are as far from 64 bits as those (256 x 256, 2000 steps: 6e-6).
__device__ __forceinline__ FkEval fk_eval(const AdjK& k, float u, float v, float w) {
#pragma clang fp contract(off)
  FkEval r;
  float p, pc, q, qc, ss, ssc;
  const float a = u - k.uc;
  sigmoid2(a, k.eh, &p, &pc);
  sigmoid2(u - k.uv, k.eh, &q, &qc);
  sigmoid2(u - k.ucsi, k.es, &ss, &ssc);
  const float f = (1.0f - u) * a, pf = p * f;
  r.p = p;
  r.vp = v * p;
  r.pw = w * p;
  r.vpf = v * pf;
  r.ws = w * ss;
  r.upc = u * pc;
  // J_fi = -v p f/tau_d, J_so = u (1 - p)/tau_0 + p/tau_r, J_si = -w ss/tau_si
  r.I = __builtin_fmaf(-r.ws, k.itsi,
                       __builtin_fmaf(-r.vpf, k.itd, __builtin_fmaf(r.upc, k.it0, p * k.itr)));
  const float itvm = recip(__builtin_fmaf(q, k.tv2m, qc * k.tv1m));
  const float ov = (1.0f - v) * itvm, ow = (1.0f - w) * k.itwm;
  const float open = pc * ov;
  r.A = __builtin_fmaf(-r.vp, k.itvp, open);
  r.B = __builtin_fmaf(-r.pw, k.itwp, pc * ow);
  const float dp = k.tihw * (p * pc), dq = k.tihw * (q * qc);
  const float dpf = __builtin_fmaf(dp, f, p * __builtin_fmaf(-2.0f, u, k.uc1));
  float Iu = __builtin_fmaf(-u, dp, pc) * k.it0;
  Iu = __builtin_fmaf(dp, k.itr, Iu);
  Iu = __builtin_fmaf(-(v * dpf), k.itd, Iu);
  r.Iu = __builtin_fmaf(-(r.ws * ssc), k.ksi, Iu);
  r.Iv = -(pf * k.itd);
  r.Iw = -(ss * k.itsi);
  r.Gvu = __builtin_fmaf(open * itvm, dq * k.dtv, dp * __builtin_fmaf(v, k.itvp, ov));
  r.Gvv = __builtin_fmaf(p, k.itvp, pc * itvm);
  r.Gwu = dp * __builtin_fmaf(w, k.itwp, ow);
  r.Gww = __builtin_fmaf(p, k.itwp, pc * k.itwm);
  return r;
}

struct Coef4 {
  float W, E, N, S;
  bool sc;
};

__device__ __forceinline__ Coef4 coef_of(const uint8_t* codes, int c) {
  Coef4 r{1.f, 1.f, 1.f, 1.f, true};
  if (codes) {
    const uint32_t b = codes[c];
    r.sc = b != kHole;
    const uint32_t q = r.sc ? b : 0u;
    r.W = (float)(q & 3u);
    r.E = (float)((q >> 2) & 3u);
    r.N = (float)((q >> 4) & 3u);
    r.S = (float)((q >> 6) & 3u);
  }
  return r;
}

// Mask coefficients of a stencil code (0xFF: hole).
__device__ __forceinline__ Coef4 coef_from_code(uint32_t b) {
  Coef4 r;
  r.sc = b != kHole;
  const uint32_t q = r.sc ? b : 0u;
  r.W = (float)(q & 3u);
  r.E = (float)((q >> 2) & 3u);
  r.N = (float)((q >> 4) & 3u);
  r.S = (float)((q >> 6) & 3u);
  return r;
}

// ---------------------------------------------------------------- forward
// Weights r (D_c + D_n) of a cell's four links, r = tc dt/(2h^2), and the
// cell's own coefficients times them: constant through the steps.
struct AdjDif {
  float W, E, N, S;
};
__device__ __forceinline__ AdjDif adj_links(const AdjK& k, float Dc, float DW, float DE, float DN,
                                            float DS) {
#pragma clang fp contract(off)
  return AdjDif{k.rxt * (Dc + DW), k.rxt * (Dc + DE), k.ryt * (Dc + DN), k.ryt * (Dc + DS)};
}
__device__ __forceinline__ AdjDif adj_dif(const Coef4& c, const AdjDif& l) {
#pragma clang fp contract(off)
  return AdjDif{c.W * l.W, c.E * l.E, c.N * l.N, c.S * l.S};
}

// One forward step of one cell from its state, its four (mirror) neighbours'
// u and its diffusion weights; shared by both forward kernels, so they agree
// bit for bit.
__device__ __forceinline__ void adj_fwd_cell(const AdjK& k, float u, float v, float w, float uW,
                                             float uE, float uN, float uS, const AdjDif& a,
                                             bool tissue, float& un, float& vn, float& wn) {
#pragma clang fp contract(off)
  float d = a.W * (uW - u);
  d = __builtin_fmaf(a.E, uE - u, d);
  d = __builtin_fmaf(a.N, uN - u, d);
  d = __builtin_fmaf(a.S, uS - u, d);
  const FkEval r = fk_eval(k, u, v, w);
  un = tissue ? u + __builtin_fmaf(-k.tdt, r.I, d) : 0.0f;
  vn = tissue ? __builtin_fmaf(k.tdt, r.A, v) : 0.0f;
  wn = tissue ? __builtin_fmaf(k.tdt, r.B, w) : 0.0f;
}

__global__ __launch_bounds__(256) void k_adj_fwd(const AdjK k, CFields in, Fields out,
                                                 const float* __restrict__ D,
                                                 const uint8_t* __restrict__ codes,
                                                 const int* __restrict__ smap,
                                                 float* __restrict__ trace_row) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  if (i >= k.nx || j >= k.ny) return;
  const int nx = k.nx, ny = k.ny;
  const int c = i + nx * j;
  const int W = mirror(i - 1, nx) + nx * j, E = mirror(i + 1, nx) + nx * j;
  const int N = i + nx * mirror(j + 1, ny), S = i + nx * mirror(j - 1, ny);
  const Coef4 cf = coef_of(codes, c);
  const float* U = in.f[0];
  float un, vn, wn;
  adj_fwd_cell(k, U[c], in.f[1][c], in.f[2][c], U[W], U[E], U[N], U[S],
               adj_dif(cf, adj_links(k, D[c], D[W], D[E], D[N], D[S])), cf.sc, un, vn, wn);
  out.f[0][c] = un;
  out.f[1][c] = vn;
  out.f[2][c] = wn;
  if (trace_row) {
    const int s = smap[c];
    if (s >= 0) trace_row[s] = un;
  }
}

// ------------------------------------------------------------------ tiles
// The tiled kernels run K <= kAdjKmax steps of an output tile of tw x th cells
// (at most kAdjTile squared).  A cell at distance m from the tile (the larger
// of its distances per axis, inside the domain) is needed exact after K - m
// steps, so in step s (from 0) the cells with m <= K - 1 - s are computed.
// One thread holds one cell for the whole launch, its state and coefficients
// in registers; LDS carries only what neighbours read.  Threads are dealt out
// in order of m, the tile first and then ring after ring, so the cells of a
// step are the first threads and every later wave skips it whole: 8 steps of
// a 16 x 16 tile take 73 wave-steps, against 92 with threads on a 32 x 32
// square and 128 with every wave in every step.  Before, a step enumerated its
// cells afresh with an integer division and modulus by run-time widths for
// each, about as many instructions as the step itself.
constexpr int kAdjTile = 16, kAdjKmax = 8, kAdjThreads = 1024;
constexpr int kAdjStride = kAdjTile + 2 * kAdjKmax + 1;  // odd: columns spread over the banks
constexpr int kAdjLds = kAdjStride * (kAdjTile + 2 * kAdjKmax);
static_assert((kAdjTile + 2 * kAdjKmax) * (kAdjTile + 2 * kAdjKmax) <= kAdjThreads,
              "one cell per thread");

struct AdjTile {
  int tiles_x, tw, th;
};

// Thread tid's cell: its coordinates and its ring m (K + 1: none, also where
// the tile or its rings reach past the domain).
struct AdjCell {
  int x, y, m;
};
__device__ __forceinline__ AdjCell adj_cell(int tid, int ox0, int oy0, const AdjTile& t, int K,
                                            int nx, int ny) {
  int m = 0;
  for (int q = 0; q <= K; ++q) m += tid >= (t.tw + 2 * q) * (t.th + 2 * q) ? 1 : 0;
  int dx, dy;
  if (m == 0) {
    dy = tid / t.tw;
    dx = tid - dy * t.tw;
  } else {
    // the ring's south row, north row, west and east column
    const int W = t.tw + 2 * m, H = t.th + 2 * m - 2;
    int p = tid - (W - 2) * H;
    if (p < 2 * W) {
      const bool north = p >= W;
      dx = (north ? p - W : p) - m;
      dy = north ? t.th + m - 1 : -m;
    } else {
      p -= 2 * W;
      const bool east = p >= H;
      dx = east ? t.tw + m - 1 : -m;
      dy = (east ? p - H : p) - m + 1;
    }
  }
  AdjCell c{ox0 + dx, oy0 + dy, m};
  if (c.x < 0 || c.x >= nx || c.y < 0 || c.y >= ny) c.m = K + 1;
  return c;
}

// A cell's place in LDS and its four neighbours' (mirrored at the domain edge,
// helper_functions.cu:69-79).
struct AdjAt {
  int l, W, E, N, S;
};
__device__ __forceinline__ AdjAt adj_at(const AdjCell& c, int ox0, int oy0, int K, int nx,
                                        int ny) {
  const int l = (c.x - ox0 + K) + kAdjStride * (c.y - oy0 + K);
  return AdjAt{l, c.x > 0 ? l - 1 : l + 1, c.x < nx - 1 ? l + 1 : l - 1,
               c.y < ny - 1 ? l + kAdjStride : l - kAdjStride,
               c.y > 0 ? l - kAdjStride : l + kAdjStride};
}

// K forward steps, their states written through to memory (left dirty in the
// XCD's L2 they delay the end of the launch: 10.1 against 9.4 us for 8 steps of
// 256 x 256).  Outputs: with seg, the state after every step into seg
// slots slot0+1 .. slot0+K; otherwise the final state into out.  Sensor traces
// for every step with step % rec == 0.
template <bool MASKED>
__global__ __launch_bounds__(kAdjThreads) void k_adj_fwd_tiled(
    const AdjK k, CFields in, Fields out, const float* __restrict__ D,
    const uint8_t* __restrict__ codes, const int* __restrict__ smap, int K, AdjTile t, int step0,
    int rec, float* __restrict__ traces, int ns, float* __restrict__ seg, size_t n, int slot0) {
  __shared__ float s_u[2][kAdjLds], s_D[kAdjLds];
  const int nx = k.nx, ny = k.ny;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int ty = tile / t.tiles_x, tx = tile - ty * t.tiles_x;
  const int ox0 = tx * t.tw, oy0 = ty * t.th;
  const AdjCell q = adj_cell(threadIdx.x, ox0, oy0, t, K, nx, ny);
  const AdjAt at = adj_at(q, ox0, oy0, K, nx, ny);
  const size_t c = (size_t)q.x + (size_t)nx * q.y;
  float u = 0.0f, v = 0.0f, w = 0.0f, Dc = 0.0f;
  Coef4 cf{1.f, 1.f, 1.f, 1.f, true};
  int sensor = -1;
  if (q.m <= K) {
    u = in.f[0][c];
    v = in.f[1][c];
    w = in.f[2][c];
    Dc = D[c];
    if (MASKED) cf = coef_from_code(codes[c]);
    if (traces && q.m == 0) sensor = smap[c];
    s_u[0][at.l] = u;
    s_D[at.l] = Dc;
  }
  __syncthreads();
  AdjDif a{};
  if (q.m < K)
    a = adj_dif(cf, adj_links(k, Dc, s_D[at.W], s_D[at.E], s_D[at.N], s_D[at.S]));
  // the state after step step0 + s + 1, and the recorded steps to come: `left`
  // steps to the next one, whose row is `row`
  float* slot = seg ? seg + (size_t)(slot0 + 1) * 3 * n : nullptr;
  int left = rec - step0 % rec;
  float* row = traces ? traces + (size_t)(step0 / rec) * ns : nullptr;
  for (int s = 0; s < K; ++s) {
    const float* U = s_u[s & 1];
    if (q.m < K - s) {
      float un, vn, wn;
      adj_fwd_cell(k, u, v, w, U[at.W], U[at.E], U[at.N], U[at.S], a, !MASKED || cf.sc, un, vn,
                   wn);
      u = un;
      v = vn;
      w = wn;
      s_u[(s & 1) ^ 1][at.l] = u;
      if (q.m == 0) {
        if (seg) {
          store_through(slot, (uint32_t)c, u);
          store_through(slot + n, (uint32_t)c, v);
          store_through(slot + 2 * n, (uint32_t)c, w);
        } else if (s == K - 1) {
          store_through(out.f[0], (uint32_t)c, u);
          store_through(out.f[1], (uint32_t)c, v);
          store_through(out.f[2], (uint32_t)c, w);
        }
        if (left == 1 && sensor >= 0) row[sensor] = u;
      }
    }
    if (seg) slot += 3 * n;
    if (--left == 0) {
      left = rec;
      if (traces) row += ns;
    }
    __syncthreads();
  }
}

// The output tile on a device of `cus` compute units, one workgroup a CU at a
// time: the shape whose busiest CU computes the fewest cell-steps, rings
// included (256 x 256: 16 x 16, 256 tiles; 128 x 128: 8 x 8, 256 tiles).
static AdjTile adj_tile(int nx, int ny, int cus) {
  const int shapes[4][2] = {{16, 16}, {16, 8}, {8, 8}, {8, 4}};
  AdjTile best{};
  double least = 1e300;
  for (const auto& sh : shapes) {
    const int tx = (nx + sh[0] - 1) / sh[0], ty = (ny + sh[1] - 1) / sh[1];
    double work = 0.0;
    for (int m = 0; m < kAdjKmax; ++m)  // waves over the four SIMDs of a CU, and a step's latency
      work += 0.5 + std::ceil((sh[0] + 2 * m) * (sh[1] + 2 * m) / 256.0);
    work *= std::ceil((double)tx * ty / std::max(1, cus));
    if (work < least) {
      least = work;
      best = AdjTile{tx, sh[0], sh[1]};
    }
  }
  return best;
}
static int adj_tiles(const AdjTile& t, int ny) { return t.tiles_x * ((ny + t.th - 1) / t.th); }

// Threads of a launch: a cell each of the tile grown by K.
static int adj_threads(const AdjTile& t, int K) {
  return ((t.tw + 2 * K) * (t.th + 2 * K) + 63) / 64 * 64;
}

static hipError_t launch_adj_fwd_tiled(const AdjK& k, const AdjTile& t, CFields in, Fields out,
                                       const float* D, const uint8_t* codes, const int* smap,
                                       int K, int step0, int rec, float* traces, int ns,
                                       float* seg, size_t n, int slot0, hipStream_t s) {
  if (K < 1 || K > kAdjKmax) return hipErrorInvalidValue;
  const dim3 g(adj_tiles(t, k.ny)), b(adj_threads(t, K));
  if (codes)
    hipLaunchKernelGGL(k_adj_fwd_tiled<true>, g, b, 0, s, k, in, out, D, codes, smap, K, t, step0,
                       rec, traces, ns, seg, n, slot0);
  else
    hipLaunchKernelGGL(k_adj_fwd_tiled<false>, g, b, 0, s, k, in, out, D, codes, smap, K, t, step0,
                       rec, traces, ns, seg, n, slot0);
  return hipGetLastError();
}

// ---------------------------------------------------------------- reverse
// The transposed operator at a cell: cw the coefficients with which the updates
// of its west, east, north and south neighbours read it, an edge neighbour's
// mirror image of it included (0 where there is no neighbour), from the
// neighbours' own coefficients; a = cw times the links' weights, and one the
// cell's own row, 1 - the sum of its weights.
struct AdjCol {
  Coef4 cw;
  AdjDif a;
  float one;
};
__device__ __forceinline__ AdjCol adj_col(const AdjDif& l, int x, int y, int nx, int ny,
                                          const Coef4& cf, const Coef4& cW, const Coef4& cE,
                                          const Coef4& cN, const Coef4& cS) {
#pragma clang fp contract(off)
  AdjCol o;
  o.cw.W = (x >= 1 ? cW.E : 0.0f) + (x == 1 ? cW.W : 0.0f);
  o.cw.E = (x + 1 < nx ? cE.W : 0.0f) + (x == nx - 2 ? cE.E : 0.0f);
  o.cw.N = (y + 1 < ny ? cN.S : 0.0f) + (y == ny - 2 ? cN.N : 0.0f);
  o.cw.S = (y >= 1 ? cS.N : 0.0f) + (y == 1 ? cS.S : 0.0f);
  o.a = adj_dif(o.cw, l);
  const AdjDif d = adj_dif(cf, l);
  o.one = 1.0f - ((d.W + d.E) + (d.N + d.S));
  return o;
}

// One reverse step of one cell: lambda of the state the forward step started
// from (r its currents) out of lambda of the step's result, m* the cell's own
// (0 in holes) and L* its neighbours' lambda_u.
__device__ __forceinline__ void adj_rev_cell(const AdjK& k, const FkEval& r, const AdjCol& o,
                                             float mu, float mv, float mw, float LW, float LE,
                                             float LN, float LS, float src, float& lu, float& lv,
                                             float& lw) {
#pragma clang fp contract(off)
  float l = LW * o.a.W;
  l = __builtin_fmaf(LE, o.a.E, l);
  l = __builtin_fmaf(LN, o.a.N, l);
  l = __builtin_fmaf(LS, o.a.S, l);
  const float tmu = k.tdt * mu, tmv = k.tdt * mv, tmw = k.tdt * mw;
  l = __builtin_fmaf(mu, __builtin_fmaf(-k.tdt, r.Iu, o.one), l);
  l = __builtin_fmaf(-tmv, r.Gvu, l);
  lu = __builtin_fmaf(-tmw, r.Gwu, l) + src;
  lv = __builtin_fmaf(-tmu, r.Iv, mv * __builtin_fmaf(-k.tdt, r.Gvv, 1.0f));
  lw = __builtin_fmaf(-tmu, r.Iw, mw * __builtin_fmaf(-k.tdt, r.Gww, 1.0f));
}

// The cell's term of dL/dD in that step: over its links r (c mu - cw L_n)
// (u_n - u), du* the differences, added to the sums of each axis (adj_gD_of()
// weighs them with r).  The factors are exact products' differences rounded once,
// products and sums FP64.
__device__ __forceinline__ void adj_gD(const Coef4& cf, const Coef4& cw, float mu, float LW,
                                       float LE, float LN, float LS, float duW, float duE,
                                       float duN, float duS, double gd[2]) {
#pragma clang fp contract(off)
  const float gW = __builtin_fmaf(-LW, cw.W, mu * cf.W), gE = __builtin_fmaf(-LE, cw.E, mu * cf.E);
  const float gN = __builtin_fmaf(-LN, cw.N, mu * cf.N), gS = __builtin_fmaf(-LS, cw.S, mu * cf.S);
  gd[0] = __builtin_fma((double)gE, (double)duE, __builtin_fma((double)gW, (double)duW, gd[0]));
  gd[1] = __builtin_fma((double)gN, (double)duN, __builtin_fma((double)gS, (double)duS, gd[1]));
}
__device__ __forceinline__ double adj_gD_of(const AdjK& k, const double gd[2]) {
#pragma clang fp contract(off)
  return __builtin_fma((double)k.rxt, gd[0], (double)k.ryt * gd[1]);
}

// Its terms of dL/dtau (tau_d, tau_r, tau_si, tau_0, tau_v+, tau_w+) without
// their constant factors, which adj_tau_factors() puts to the sums.
__device__ __forceinline__ void adj_gtau(const FkEval& r, float mu, float mv, float mw,
                                         double gt[6]) {
#pragma clang fp contract(off)
  gt[0] += (double)(mu * r.vpf);
  gt[1] += (double)(mu * r.p);
  gt[2] += (double)(mu * r.ws);
  gt[3] += (double)(mu * r.upc);
  gt[4] += (double)(mv * r.vp);
  gt[5] += (double)(mw * r.pw);
}
// -tc dt d(1/tau) of the term each sum multiplies: J_fi and J_si enter with a
// minus, J_so's two with a plus, and the gates close with p v/tau_v+, p w/tau_w+.
static void adj_tau_factors(double tdt, const double tau[6], double f[6]) {
  for (int q = 0; q < 6; ++q) f[q] = (q == 0 || q == 2 ? -tdt : tdt) / (tau[q] * tau[q]);
}

// The sums of gt over the first NT threads of a workgroup, those that hold any
// (FP64, fixed order), added to the workgroup's slot, whose value before
// (of threads 0 to 5) is `was` (read early, and the sums by VALU moves: 15.2 ->
// 14.6 us a reverse launch against ds_bpermute trees and a late read).
template <int NT>
__device__ __forceinline__ void adj_gtau_block(const double gt[6], double was, double* slot) {
  __shared__ double red[NT / 64][6];
  const int waves = min(NT, (int)(blockDim.x * blockDim.y)) / 64;
  const int tid = threadIdx.y * blockDim.x + threadIdx.x;
  const int lane = tid & 63, wv = tid >> 6;
  if (wv < waves) {
#pragma unroll
    for (int q = 0; q < 6; ++q) {
      const double v = wave_sum(gt[q]);
      if (lane == 0) red[wv][q] = v;
    }
  }
  __syncthreads();
  if (tid < 6) {
    double s = 0.0;
    for (int w = 0; w < waves; ++w) s += red[w][tid];
    slot[tid] = was + s;
  }
}

__global__ __launch_bounds__(256) void k_adj_rev(const AdjK k, CFields X, CFields lam_in,
                                                 Fields lam_out, const float* __restrict__ D,
                                                 const uint8_t* __restrict__ codes,
                                                 const int* __restrict__ smap,
                                                 const float* __restrict__ src_row,
                                                 double* __restrict__ gD,
                                                 double* __restrict__ gtau_part) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  double gtd[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  if (i < k.nx && j < k.ny) {
    const int c = i + k.nx * j;
    const int W = mirror(i - 1, k.nx) + k.nx * j, E = mirror(i + 1, k.nx) + k.nx * j;
    const int N = i + k.nx * mirror(j + 1, k.ny), S = i + k.nx * mirror(j - 1, k.ny);
    float src = 0.0f;
    if (src_row) {
      const int s = smap[c];
      if (s >= 0) src = src_row[s];
    }
    const Coef4 cf = coef_of(codes, c);
    const AdjCol o = adj_col(adj_links(k, D[c], D[W], D[E], D[N], D[S]), i, j, k.nx, k.ny, cf,
                             coef_of(codes, W), coef_of(codes, E), coef_of(codes, N),
                             coef_of(codes, S));
    const float *U = X.f[0], *L = lam_in.f[0];
    const float u = U[c], LW = L[W], LE = L[E], LN = L[N], LS = L[S];
    const float m = cf.sc ? 1.0f : 0.0f;
    const float mu = m * L[c], mv = m * lam_in.f[1][c], mw = m * lam_in.f[2][c];
    const FkEval r = fk_eval(k, u, X.f[1][c], X.f[2][c]);
    float lu, lv, lw;
    adj_rev_cell(k, r, o, mu, mv, mw, LW, LE, LN, LS, src, lu, lv, lw);
    double gd[2] = {0.0, 0.0};
    adj_gD(cf, o.cw, mu, LW, LE, LN, LS, U[W] - u, U[E] - u, U[N] - u, U[S] - u, gd);
    adj_gtau(r, mu, mv, mw, gtd);
    lam_out.f[0][c] = lu;
    lam_out.f[1][c] = lv;
    lam_out.f[2][c] = lw;
    gD[c] += adj_gD_of(k, gd);
  }
  double* slot = gtau_part + (size_t)(blockIdx.y * gridDim.x + blockIdx.x) * 6;
  const int tid = threadIdx.y * blockDim.x + threadIdx.x;
  adj_gtau_block<256>(gtd, tid < 6 ? slot[tid] : 0.0, slot);
}

// K reverse steps, n_top, n_top-1, ..., of one tile (see the tiles section;
// lambda has the forward's one-cell dependence).  u of each step's state goes through LDS
// (the neighbours of the tile's cells read it for dL/dD), lambda_u through a
// double buffer.  A thread keeps its lambda_v, lambda_w, its row and column of
// the transposed operator (constant through the steps), and, in the tile, its
// dL/dD and dL/dtau sums (FP64).  u, v, w and the sensor source of a step are
// loaded two steps ahead.  A step is bound by VALU issue (see fk_eval): 8 steps
// of a 16 x 16 tile are 21 wave-steps on the busiest SIMD.  Launches of 8 steps
// at 256 x 256: 25.4 us with per-step index arithmetic, 15.5 with a thread a
// cell, 13.0 with fewer instructions a step; the forward's 12.8, 10.1, 8.6.
template <bool MASKED>
__global__ __launch_bounds__(kAdjThreads) void k_adj_rev_tiled(
    const AdjK k, const float* __restrict__ seg, const float* __restrict__ x0, size_t n,
    int slot_top, int n_top, CFields lam_in, Fields lam_out, const float* __restrict__ D,
    const uint8_t* __restrict__ codes, const int* __restrict__ smap,
    const float* __restrict__ src, int rec, int ns, double* __restrict__ gD,
    double* __restrict__ gtau_part, int K, AdjTile t) {
#pragma clang fp contract(off)
  __shared__ float s_U[2][kAdjLds], s_L[2][kAdjLds], s_D[kAdjLds];
  __shared__ uint8_t s_c[MASKED ? kAdjLds : 1];
  const int nx = k.nx, ny = k.ny;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int ty = tile / t.tiles_x, tx = tile - ty * t.tiles_x;
  const int ox0 = tx * t.tw, oy0 = ty * t.th;
  const AdjCell q = adj_cell(threadIdx.x, ox0, oy0, t, K, nx, ny);
  const AdjAt at = adj_at(q, ox0, oy0, K, nx, ny);
  const size_t c = (size_t)q.x + (size_t)nx * q.y;
  const int sensor = src && q.m < K ? smap[c] : -1;
  struct Ahead {
    float u = 0.0f, v = 0.0f, w = 0.0f, src = 0.0f;
  };
  auto fetch = [&](int s) {
    Ahead a;
    if (s < K && q.m <= K - s) {
      const float* X = slot_top - s == 0 ? x0 : seg + (size_t)(slot_top - s) * 3 * n;
      a.u = X[c];
      a.v = X[n + c];
      a.w = X[2 * n + c];
      const int step = n_top - s;
      if (sensor >= 0 && step >= 1 && step % rec == 0)
        a.src = src[(size_t)(step / rec - 1) * ns + sensor];
    }
    return a;
  };
  float Lu = 0.0f, Lv = 0.0f, Lw = 0.0f, Dc = 0.0f;
  Coef4 cf{1.f, 1.f, 1.f, 1.f, true};
  Ahead cur = fetch(0), next = fetch(1);
  if (q.m <= K) {
    Lu = lam_in.f[0][c];
    Lv = lam_in.f[1][c];
    Lw = lam_in.f[2][c];
    Dc = D[c];
    s_L[0][at.l] = Lu;
    s_D[at.l] = Dc;
    s_U[0][at.l] = cur.u;
    if (MASKED) {
      const uint32_t code = codes[c];
      s_c[at.l] = (uint8_t)code;
      cf = coef_from_code(code);
    }
  }
  __syncthreads();
  AdjCol o{};
  const float m = !MASKED || cf.sc ? 1.0f : 0.0f;
  if (q.m < K) {
    Coef4 cW{1.f, 1.f, 1.f, 1.f, true}, cE = cW, cN = cW, cS = cW;
    if (MASKED) {
      cW = coef_from_code(s_c[at.W]);
      cE = coef_from_code(s_c[at.E]);
      cN = coef_from_code(s_c[at.N]);
      cS = coef_from_code(s_c[at.S]);
    }
    o = adj_col(adj_links(k, Dc, s_D[at.W], s_D[at.E], s_D[at.N], s_D[at.S]), q.x, q.y, nx, ny,
                cf, cW, cE, cN, cS);
  }
  // what the sums are added to at the end, read now
  double* gt_slot = gtau_part + (size_t)tile * 6;
  const double gD_was = q.m == 0 ? gD[c] : 0.0;
  const double gt_was = threadIdx.x < 6 ? gt_slot[threadIdx.x] : 0.0;
  double gd[2] = {0.0, 0.0}, gtd[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  for (int s = 0; s < K; ++s) {
    const int b = s & 1;
    const Ahead then = fetch(s + 2);
    if (q.m < K - s) {
      const float* L = s_L[b];
      const float LE = L[at.E], LW = L[at.W], LN = L[at.N], LS = L[at.S];
      const float mu = m * Lu, mv = m * Lv, mw = m * Lw;
      const FkEval r = fk_eval(k, cur.u, cur.v, cur.w);
      adj_rev_cell(k, r, o, mu, mv, mw, LW, LE, LN, LS, cur.src, Lu, Lv, Lw);
      if (q.m == 0) {  // dL/dD and dL/dtau of the tile's cells
        const float* U = s_U[b];
        adj_gD(cf, o.cw, mu, LW, LE, LN, LS, U[at.W] - cur.u, U[at.E] - cur.u,
               U[at.N] - cur.u, U[at.S] - cur.u, gd);
        adj_gtau(r, mu, mv, mw, gtd);
      }
      s_L[b ^ 1][at.l] = Lu;
    }
    if (q.m <= 1) s_U[b ^ 1][at.l] = next.u;
    cur = next;
    next = then;
    __syncthreads();
  }
  if (q.m == 0) {
    store_through(lam_out.f[0], (uint32_t)c, Lu);
    store_through(lam_out.f[1], (uint32_t)c, Lv);
    store_through(lam_out.f[2], (uint32_t)c, Lw);
    gD[c] = gD_was + adj_gD_of(k, gd);
  }
  adj_gtau_block<kAdjTile * kAdjTile>(gtd, gt_was, gt_slot);
}

static hipError_t launch_adj_rev_tiled(const AdjK& k, const AdjTile& t, const float* seg,
                                       const float* x0, size_t n, int slot_top, int n_top,
                                       CFields li, Fields lo, const float* D,
                                       const uint8_t* codes, const int* smap, const float* src,
                                       int rec, int ns, double* gD, double* gtau_part, int K,
                                       hipStream_t s) {
  if (K < 1 || K > kAdjKmax) return hipErrorInvalidValue;
  const dim3 g(adj_tiles(t, k.ny)), b(adj_threads(t, K));
  if (codes)
    hipLaunchKernelGGL(k_adj_rev_tiled<true>, g, b, 0, s, k, seg, x0, n, slot_top, n_top, li, lo,
                       D, codes, smap, src, rec, ns, gD, gtau_part, K, t);
  else
    hipLaunchKernelGGL(k_adj_rev_tiled<false>, g, b, 0, s, k, seg, x0, n, slot_top, n_top, li, lo,
                       D, codes, smap, src, rec, ns, gD, gtau_part, K, t);
  return hipGetLastError();
}

// lambda^N: zero, plus the sensor source of the last recorded step.
__global__ void k_adj_init(Fields lam, size_t n, const int* __restrict__ smap,
                           const float* __restrict__ src_row) {
  for (size_t c = blockIdx.x * (size_t)blockDim.x + threadIdx.x; c < n;
       c += (size_t)gridDim.x * blockDim.x) {
    float s = 0.0f;
    if (src_row) {
      const int q = smap[c];
      if (q >= 0) s = src_row[q];
    }
    lam.f[0][c] = s;
    lam.f[1][c] = 0.0f;
    lam.f[2][c] = 0.0f;
  }
}

// src = 2 (trace - target), the source of the reverse sweep, and the loss sum
// (trace - target)^2 in FP64: per thread, then per wave, then per workgroup in
// a fixed order, one partial a workgroup.
constexpr int kLossBlocks = 64;
__global__ __launch_bounds__(256) void k_adj_loss(const float* __restrict__ traces,
                                                  const float* __restrict__ targets,
                                                  float* __restrict__ src, size_t m,
                                                  double* __restrict__ part) {
  __shared__ double red[4];
  double sum = 0.0;
  for (size_t q = blockIdx.x * (size_t)256 + threadIdx.x; q < m; q += (size_t)kLossBlocks * 256) {
    const double d = (double)traces[q] - (double)targets[q];
    sum += d * d;
    src[q] = (float)(2.0 * d);
  }
  sum = wave_sum(sum);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

__global__ void k_fill_d(double* p, size_t n, double v) {
  for (size_t c = blockIdx.x * (size_t)blockDim.x + threadIdx.x; c < n;
       c += (size_t)gridDim.x * blockDim.x)
    p[c] = v;
}

}  // namespace yh

struct yh_adjoint {
  yh_params p;
  yh_derived d;
  int nsteps = 0, rec = 1, ckpt = 100, ns = 0, nrec = 0, nckpt = 0;
  size_t n = 0;
  std::vector<int> sensors;
  float* X[2][3] = {{nullptr, nullptr, nullptr}, {nullptr, nullptr, nullptr}};
  float* X0[3] = {nullptr, nullptr, nullptr};
  float* ck = nullptr;   // nckpt x 3 x n
  float* seg = nullptr;  // (ckpt + 1) x 3 x n
  float* lam[2][3] = {{nullptr, nullptr, nullptr}, {nullptr, nullptr, nullptr}};
  int* smap = nullptr;
  uint8_t* solid = nullptr;
  uint8_t* codes = nullptr;
  float* traces = nullptr;   // nrec x ns (device)
  float* targets = nullptr;  // nrec x ns (device)
  float* src = nullptr;      // nrec x ns: 2 (trace - target)
  double* gD = nullptr;
  double* gtau_part = nullptr;
  int nblocks = 0;
  double* loss_part = nullptr;  // kLossBlocks
  bool have_targets = false, forward_done = false;
  const float* D = nullptr;
  yh::AdjK k{};
  double tau_f[6] = {};  // adj_tau_factors() of the forward's time constants
  int fwdK = 8;  // steps per launch, forward and reverse: 1 = one-step kernels, else LDS-tiled
  int nparts = 0;  // dL/dtau workgroup slots: the larger of the two reverse grids
  yh::AdjTile tile{};  // output tile of the tiled kernels
  // every state X^0 .. X^nsteps is kept (seg slots 0 .. nsteps), so the reverse
  // sweep recomputes nothing; otherwise checkpoints every ckpt steps
  bool keep = false;
};

namespace yh {

static void adj_free(yh_adjoint* a) {
  if (!a) return;
  for (int b = 0; b < 2; ++b)
    for (int q = 0; q < 3; ++q) {
      if (a->X[b][q]) (void)hipFree(a->X[b][q]);
      if (a->lam[b][q]) (void)hipFree(a->lam[b][q]);
    }
  for (int q = 0; q < 3; ++q)
    if (a->X0[q]) (void)hipFree(a->X0[q]);
  void* ptrs[] = {a->ck, a->seg, a->smap, a->solid, a->codes, a->traces, a->targets, a->src,
                  a->gD, a->gtau_part, a->loss_part};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  delete a;
}

static void adj_k(yh_adjoint* a, const double tau6[6]) {
  AdjK& k = a->k;
  const yh_params& p = a->p;
  k.nx = p.nx;
  k.ny = p.ny;
  const double tdt = p.tc * a->d.dt, ln2 = std::log(2.0);
  k.rxt = (float)(0.5 * tdt / (a->d.hx * a->d.hx));
  k.ryt = (float)(0.5 * tdt / (a->d.hy * a->d.hy));
  k.tdt = (float)tdt;
  const yh_fk_params& f = p.fk;
  k.uc = (float)f.u_c;
  k.uv = (float)f.u_v;
  k.ucsi = (float)f.u_csi;
  k.uc1 = (float)(1.0 + f.u_c);
  // recip() needs a finite sum of the two: one that is infinite, or past the range
  // of a float, switches its recovery off, as 1e30 ms does
  const double tv1m = std::min(f.tau_v1m, 1e30), tv2m = std::min(f.tau_v2m, 1e30);
  k.tv1m = (float)tv1m;
  k.tv2m = (float)tv2m;
  k.dtv = (float)(tv2m - tv1m);
  k.eh = (float)(2.0 / (p.heaviside_width * ln2));
  k.es = (float)(2.0 * f.k / ln2);
  k.tihw = (float)(2.0 / p.heaviside_width);
  k.itd = (float)(1.0 / tau6[0]);
  k.itr = (float)(1.0 / tau6[1]);
  k.itsi = (float)(1.0 / tau6[2]);
  k.ksi = (float)(2.0 * f.k / tau6[2]);
  k.it0 = (float)(1.0 / tau6[3]);
  k.itvp = (float)(1.0 / tau6[4]);
  k.itwp = (float)(1.0 / tau6[5]);
  k.itwm = (float)(1.0 / f.tau_wm);
  adj_tau_factors(tdt, tau6, a->tau_f);
}

// Most device memory a problem takes to keep every state of its forward sweep,
// unless the caller sets another limit.
constexpr int64_t kAdjKeep = (int64_t)4 << 30;

static inline float* slot(float* base, size_t n, int s, int var) {
  return base + ((size_t)s * 3 + var) * n;
}

}  // namespace yh

using namespace yh;

extern "C" {

int yh_adjoint_create(const yh_params* p, int nsteps, int rec_every, int ckpt_every,
                      const int* sensors, int nsensors, yh_adjoint** out) {
  return yh_adjoint_create_keep(p, nsteps, rec_every, ckpt_every, -1, sensors, nsensors, out);
}

int yh_adjoint_create_keep(const yh_params* p, int nsteps, int rec_every, int ckpt_every,
                           int64_t keep_bytes, const int* sensors, int nsensors,
                           yh_adjoint** out) {
  if (!p || !out || nsteps < 1 || rec_every < 1 || ckpt_every < 1 || nsensors < 1 || !sensors)
    return YH_EINVAL;
  if (p->model != YH_MODEL_3V_FK || !(p->heaviside_width > 0) || p->reduceSym)
    return YH_EINVAL;
  if (!standard_branch(*p)) return YH_EUNSUPPORTED;
  *out = nullptr;
  yh_derived d;
  int rc = yh_params_derive(p, &d);
  if (rc) return rc;
  const size_t n = (size_t)p->nx * p->ny;
  for (int s = 0; s < nsensors; ++s)
    if (sensors[s] < 0 || (size_t)sensors[s] >= n) return YH_EINVAL;
  yh_adjoint* a = new (std::nothrow) yh_adjoint();
  if (!a) return YH_ENOMEM;
  a->p = *p;
  a->d = d;
  a->nsteps = nsteps;
  a->rec = rec_every;
  a->ckpt = std::min(ckpt_every, nsteps);
  a->ns = nsensors;
  a->nrec = nsteps / rec_every;
  a->nckpt = (nsteps + a->ckpt - 1) / a->ckpt;
  a->n = n;
  a->sensors.assign(sensors, sensors + nsensors);
  std::vector<int> smap(n, -1);
  for (int s = 0; s < nsensors; ++s) {
    if (smap[sensors[s]] >= 0) {  // duplicate sensor cell
      adj_free(a);
      return YH_EINVAL;
    }
    smap[sensors[s]] = s;
  }
  const double tau6[6] = {p->fk.tau_d, p->fk.tau_r, p->fk.tau_si,
                          p->fk.tau_0, p->fk.tau_vp, p->fk.tau_wp};
  adj_k(a, tau6);
  const dim3 bg((p->nx + 63) / 64, (p->ny + 3) / 4);  // the 64 x 4 one-step blocks
  a->nblocks = bg.x * bg.y;
  int dev = 0, cus = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  a->tile = adj_tile(p->nx, p->ny, cus);
  a->nparts = std::max(a->nblocks, adj_tiles(a->tile, p->ny));
  auto M = [&](void** ptr, size_t bytes) {
    if (e == hipSuccess) e = hipMalloc(ptr, std::max<size_t>(bytes, 4));
  };
  for (int b = 0; b < 2; ++b)
    for (int q = 0; q < 3; ++q) {
      M((void**)&a->X[b][q], n * 4);
      M((void**)&a->lam[b][q], n * 4);
    }
  for (int q = 0; q < 3; ++q) M((void**)&a->X0[q], n * 4);
  // All states where they take at most the limit and a quarter of what is free
  // on the device: recomputing each segment is a second forward sweep (2.4 of
  // 9.0 ms per gradient at 256 x 256 x 2000, whose states are 1.6 GB of 288).
  // If they cannot be had, the checkpoints the caller asked for.
  const size_t all = (size_t)(nsteps + 1) * 3 * n * 4;
  size_t avail = 0, total = 0;
  const size_t limit = (size_t)(keep_bytes < 0 ? kAdjKeep : keep_bytes);
  if (e == hipSuccess && all <= limit && hipMemGetInfo(&avail, &total) == hipSuccess &&
      all <= avail / 4) {
    a->keep = hipMalloc(&a->seg, all) == hipSuccess;
    if (!a->keep) {
      a->seg = nullptr;
      (void)hipGetLastError();
    }
  }
  if (!a->keep) {
    M((void**)&a->ck, (size_t)a->nckpt * 3 * n * 4);
    M((void**)&a->seg, (size_t)(a->ckpt + 1) * 3 * n * 4);
  }
  M((void**)&a->smap, n * 4);
  M((void**)&a->traces, (size_t)a->nrec * a->ns * 4);
  M((void**)&a->targets, (size_t)a->nrec * a->ns * 4);
  M((void**)&a->src, (size_t)a->nrec * a->ns * 4);
  M((void**)&a->gD, n * 8);
  M((void**)&a->loss_part, kLossBlocks * 8);
  M((void**)&a->gtau_part, (size_t)a->nparts * 6 * 8);
  if (e == hipSuccess) e = hipMemcpy(a->smap, smap.data(), n * 4, hipMemcpyHostToDevice);
  for (int q = 0; q < 3 && e == hipSuccess; ++q) e = hipMemset(a->X0[q], 0, n * 4);
  if (e != hipSuccess) {
    rc = hip_fail(e, "yh_adjoint_create");
    adj_free(a);
    return rc;
  }
  *out = a;
  return YH_OK;
}

void yh_adjoint_destroy(yh_adjoint* a) {
  if (a) (void)hipDeviceSynchronize();
  adj_free(a);
}

int yh_adjoint_keeps_states(const yh_adjoint* a) { return a && a->keep ? 1 : 0; }

int yh_adjoint_set_substeps(yh_adjoint* a, int k) {
  if (!a || k < 1 || k > kAdjKmax) return YH_EINVAL;
  a->fwdK = k;
  return YH_OK;
}

int yh_adjoint_set_mask(yh_adjoint* a, const uint8_t* solid) {
  if (!a || !solid) return YH_EINVAL;
  if (!a->p.solidSwitch) return YH_ESTATE;
  if (!a->solid) YH_HIP(hipMalloc(&a->solid, a->n));
  if (!a->codes) YH_HIP(hipMalloc(&a->codes, a->n));
  std::vector<uint8_t> m(a->n);
  for (size_t c = 0; c < a->n; ++c) m[c] = solid[c] ? 1 : 0;
  YH_HIP(hipMemcpy(a->solid, m.data(), a->n, hipMemcpyHostToDevice));
  YH_HIP(launch_codes(a->solid, a->codes, a->p.nx, a->p.ny, nullptr));
  YH_HIP(hipDeviceSynchronize());
  return YH_OK;
}

int yh_adjoint_set_initial(yh_adjoint* a, const float* u, const float* v, const float* w) {
  if (!a || !u || !v || !w) return YH_EINVAL;
  const float* s[3] = {u, v, w};
  for (int q = 0; q < 3; ++q) YH_HIP(hipMemcpy(a->X0[q], s[q], a->n * 4, hipMemcpyHostToDevice));
  a->forward_done = false;
  return YH_OK;
}

int yh_adjoint_set_targets(yh_adjoint* a, const float* targets) {
  if (!a || !targets) return YH_EINVAL;
  const size_t m = (size_t)a->nrec * a->ns;
  YH_HIP(hipMemcpy(a->targets, targets, m * 4, hipMemcpyHostToDevice));
  a->have_targets = true;
  return YH_OK;
}

int yh_adjoint_forward(yh_adjoint* a, const float* d_D, const double tau6[6], void* stream,
                       double* loss, float* traces) {
  if (!a || !d_D || !tau6) return YH_EINVAL;
  for (int q = 0; q < 6; ++q)
    if (!(tau6[q] > 0)) return YH_EINVAL;
  if (a->p.solidSwitch && !a->codes) return YH_ESTATE;
  hipStream_t s = (hipStream_t)stream;
  adj_k(a, tau6);
  a->D = d_D;
  const size_t n = a->n;
  dim3 bb(64, 4), bg((a->p.nx + 63) / 64, (a->p.ny + 3) / 4);
  // X^0 to its slot.  With every state kept, launches write the state after
  // each step into its slot; otherwise a launch that ends on a checkpoint step
  // writes its state into that checkpoint, which the next launch reads.
  float* x0 = a->keep ? a->seg : a->ck;
  for (int q = 0; q < 3; ++q)
    YH_HIP(hipMemcpyAsync(slot(x0, n, 0, q), a->X0[q], n * 4, hipMemcpyDeviceToDevice, s));
  CFields in{{slot(x0, n, 0, 0), slot(x0, n, 0, 1), slot(x0, n, 0, 2)}};
  int nb = 0;  // the work buffer the next launch writes (never the one it reads)
  for (int done = 0; done < a->nsteps;) {
    int K = std::min(a->fwdK, a->nsteps - done);
    if (!a->keep) K = std::min(K, (done / a->ckpt + 1) * a->ckpt - done);  // end on checkpoints
    const int end = done + K;
    const bool to_ck = !a->keep && end % a->ckpt == 0 && end < a->nsteps;
    float* to = a->keep ? slot(a->seg, n, end, 0) : to_ck ? slot(a->ck, n, end / a->ckpt, 0) : nullptr;
    const Fields out = to ? Fields{{to, to + n, to + 2 * n}}
                          : Fields{{a->X[nb][0], a->X[nb][1], a->X[nb][2]}};
    if (a->fwdK == 1) {
      const int step = done + 1;
      float* row = (step % a->rec == 0) ? a->traces + (size_t)(step / a->rec - 1) * a->ns : nullptr;
      hipLaunchKernelGGL(k_adj_fwd, bg, bb, 0, s, a->k, in, out, d_D, a->codes, a->smap, row);
      YH_HIP(hipGetLastError());
    } else {
      YH_HIP(launch_adj_fwd_tiled(a->k, a->tile, in, out, d_D, a->codes, a->smap, K, done, a->rec,
                                  a->traces, a->ns, a->keep ? a->seg : nullptr, n, done, s));
    }
    in = CFields{{out.f[0], out.f[1], out.f[2]}};
    if (!to) nb ^= 1;
    done = end;
  }
  const size_t m = (size_t)a->nrec * a->ns;
  double part[kLossBlocks] = {};
  if (a->have_targets) {
    // on the device: the host's loop over the traces and their way there and
    // back took 0.3 ms at 2000 records of 64 sensors
    hipLaunchKernelGGL(k_adj_loss, dim3(kLossBlocks), dim3(256), 0, s, a->traces, a->targets,
                       a->src, m, a->loss_part);
    YH_HIP(hipGetLastError());
    YH_HIP(hipMemcpyAsync(part, a->loss_part, sizeof part, hipMemcpyDeviceToHost, s));
  }
  if (traces) YH_HIP(hipMemcpyAsync(traces, a->traces, m * 4, hipMemcpyDeviceToHost, s));
  YH_HIP(hipStreamSynchronize(s));
  double L = 0.0;
  for (double q : part) L += q;
  if (loss) *loss = L;
  a->forward_done = true;
  return YH_OK;
}

int yh_adjoint_backward(yh_adjoint* a, void* stream, double* d_gD, double gtau[6]) {
  if (!a || !d_gD || !gtau) return YH_EINVAL;
  if (!a->forward_done || !a->have_targets) return YH_ESTATE;
  hipStream_t s = (hipStream_t)stream;
  const size_t n = a->n;
  const int N = a->nsteps;
  dim3 bb(64, 4), bg((a->p.nx + 63) / 64, (a->p.ny + 3) / 4);
  hipLaunchKernelGGL(k_fill_d, dim3(256), dim3(256), 0, s, a->gD, n, 0.0);
  hipLaunchKernelGGL(k_fill_d, dim3(64), dim3(256), 0, s, a->gtau_part, (size_t)a->nparts * 6, 0.0);
  // lambda^N
  const float* srcN = (N % a->rec == 0) ? a->src + (size_t)(N / a->rec - 1) * a->ns : nullptr;
  int lc = 0;
  Fields l0{{a->lam[0][0], a->lam[0][1], a->lam[0][2]}};
  hipLaunchKernelGGL(k_adj_init, dim3(256), dim3(256), 0, s, l0, n, (const int*)a->smap, srcN);
  YH_HIP(hipGetLastError());
  const int span = a->keep ? N : a->ckpt;
  for (int seg = (N + span - 1) / span - 1; seg >= 0; --seg) {
    const int s0 = seg * span;
    const int s1 = std::min(N, s0 + span);  // reverse steps n = s1-1 .. s0
    // X^{s0}: its slot, or its checkpoint (slot 0 of the segment stands for it)
    float* x0 = slot(a->keep ? a->seg : a->ck, n, seg, 0);
    // with checkpoints, recompute X^{s0+1} .. X^{s1-1} into seg slots 1 .. s1-s0-1
    for (int t = 1; !a->keep && t < s1 - s0;) {
      CFields in = t == 1 ? CFields{{x0, x0 + n, x0 + 2 * n}}
                          : CFields{{slot(a->seg, n, t - 1, 0), slot(a->seg, n, t - 1, 1),
                                     slot(a->seg, n, t - 1, 2)}};
      Fields out{{slot(a->seg, n, t, 0), slot(a->seg, n, t, 1), slot(a->seg, n, t, 2)}};
      const int K = std::min(a->fwdK, s1 - s0 - t);
      if (a->fwdK == 1) {
        hipLaunchKernelGGL(k_adj_fwd, bg, bb, 0, s, a->k, in, out, a->D, a->codes, a->smap,
                           (float*)nullptr);
        YH_HIP(hipGetLastError());
      } else {  // slots t .. t+K-1
        YH_HIP(launch_adj_fwd_tiled(a->k, a->tile, in, out, a->D, a->codes, a->smap, K, s0 + t - 1,
                                    a->rec, nullptr, a->ns, a->seg, n, t - 1, s));
      }
      t += K;
    }
    for (int step = s1 - 1; step >= s0;) {
      const int t = step - s0;
      CFields li{{a->lam[lc][0], a->lam[lc][1], a->lam[lc][2]}};
      Fields lo{{a->lam[lc ^ 1][0], a->lam[lc ^ 1][1], a->lam[lc ^ 1][2]}};
      if (a->fwdK == 1) {
        CFields X = t == 0 ? CFields{{x0, x0 + n, x0 + 2 * n}}
                           : CFields{{slot(a->seg, n, t, 0), slot(a->seg, n, t, 1),
                                      slot(a->seg, n, t, 2)}};
        const float* src = (step >= 1 && step % a->rec == 0)
                               ? a->src + (size_t)(step / a->rec - 1) * a->ns
                               : nullptr;
        hipLaunchKernelGGL(k_adj_rev, bg, bb, 0, s, a->k, X, li, lo, a->D, a->codes, a->smap,
                           src, a->gD, a->gtau_part);
        YH_HIP(hipGetLastError());
        step -= 1;
      } else {  // steps step, step-1, ..., step-K+1 of this segment
        const int K = std::min(a->fwdK, t + 1);
        YH_HIP(launch_adj_rev_tiled(a->k, a->tile, a->seg, x0, n, t, step, li, lo, a->D, a->codes,
                                    a->smap, a->src, a->rec, a->ns, a->gD, a->gtau_part, K, s));
        step -= K;
      }
      lc ^= 1;
    }
  }
  YH_HIP(hipMemcpyAsync(d_gD, a->gD, n * 8, hipMemcpyDeviceToDevice, s));
  std::vector<double> part((size_t)a->nparts * 6);
  YH_HIP(hipMemcpyAsync(part.data(), a->gtau_part, part.size() * 8, hipMemcpyDeviceToHost, s));
  YH_HIP(hipStreamSynchronize(s));
  for (int q = 0; q < 6; ++q) gtau[q] = 0.0;
  for (int b = 0; b < a->nparts; ++b)
    for (int q = 0; q < 6; ++q) gtau[q] += part[(size_t)b * 6 + q];
  for (int q = 0; q < 6; ++q) gtau[q] *= a->tau_f[q];
  return YH_OK;
}

}  // extern "C"
