// general.hip -- the reference kernel's other branches on the device:
// Dirichlet boundaries, the 4th-order compact Laplacian (lap4), the
// anisotropic cross term, RK2 / RK4 and the circular mouse stimulus
// (reactionDiffusion.cu:36-561).  One launch advances several Runge-Kutta
// stages, and where they are few several steps, of a tile held in registers
// and LDS.
//
// The reference writes each stage state into its input while neighbours read
// it (:114-119) and reads lap4's neighbour currents J from the same launch
// (:221-236).  Here a stage reads only the step's input y0 and the previous
// stage's increments d: the stage field is y0 + ki*d_{s-1}, a neighbour's
// current is evaluated from that neighbour's stage state, and the stage field
// of a tile is complete (a barrier, two LDS buffers) before the next stage
// reads it.  Reads outside the domain that the reference makes in the masked
// Dirichlet branch (:364-373 at the domain edge) count as non-tissue.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>

#include "plan.h"
#include "tile.h"

namespace yh {

GParams make_gparams(const yh_params& p, int stim_on, int stim_x, int stim_y) {
  // parameterSetup (saveFiles.cu:144-170) and the startup recomputation after
  // the symmetry-reduction halving (main.cu:148-155)
  const double pi = 3.14159265359;  // globalVariables.cuh:27
  const double hx = p.Lx / (p.nx - 1.0), hy = p.Ly / (p.ny - 1.0);
  const double th = p.degrad * pi / 180.0;
  const double Dxx = p.diff_par * std::cos(th) * std::cos(th) + p.diff_per * std::sin(th) * std::sin(th);
  const double Dyy = p.diff_par * std::sin(th) * std::sin(th) + p.diff_per * std::cos(th) * std::cos(th);
  const double Dxy = (p.diff_par - p.diff_per) * std::sin(th) * std::cos(th);
  const double dt = p.reduceSym ? 0.5 * p.dt : p.dt;
  GParams g;
  g.nx = p.nx;
  g.ny = p.ny;
  g.masked = p.solidSwitch;
  g.neumann = p.neumannBC;
  g.lap4 = p.lap4 ? 1 : 0;
  g.aniso = p.anisotropy ? 1 : 0;
  g.vdiff = (p.model == YH_MODEL_2V_REF && p.gateDiff) ? 1 : 0;
  g.rx = (float)(dt * Dxx / (hx * hx));
  g.ry = (float)(dt * Dyy / (hy * hy));
  g.rxy = (float)(2.0 * Dxy * dt / (4.0 * hx * hy));
  g.rbx = (float)(hx * Dxy / (Dxx * hy));
  g.rby = (float)(hy * Dxy / (Dyy * hx));
  g.q4 = (float)(dt * Dyy / (hy * hy * 12.0) + dt * Dxx / (hx * hx * 12.0));
  g.fx4 = (float)(dt / 12.0);
  g.fy4 = (float)(dt / 12.0);
  g.dt = (float)dt;
  g.tc = (float)p.tc;
  g.rscale = (float)p.rscale;
  g.bval = (float)p.boundaryVal;
  g.mu = (float)p.mu;
  g.alpha = (float)p.alpha;
  g.beta = (float)p.beta;
  g.gamma = (float)p.gamma;
  g.delta = (float)p.delta;
  g.eps = (float)p.eps;
  g.theta = (float)p.theta;
  const yh_fk_params& f = p.fk;
  g.u_c = (float)f.u_c;
  g.u_v = (float)f.u_v;
  g.u_csi = (float)f.u_csi;
  g.kk = (float)f.k;
  // The constants that currents and rates are divided by, as g_quotient takes
  // them: t and r = 1/t.  An infinite one (or past the range of a float) switches
  // its term off, a quotient of 0, which t = r = 0 gives; with the infinity the
  // remainder would be a NaN.  One below the least normal float, whose reciprocal
  // may overflow, counts as that.
  auto divisor = [](float tau, float& t, float& r) {
    t = r = 0.0f;
    if (!(tau <= FLT_MAX)) return;
    t = std::max(tau, FLT_MIN);
    r = (float)(1.0 / (double)t);
  };
  divisor((float)f.tau_d, g.tau_d, g.r_d);
  divisor((float)f.tau_r, g.tau_r, g.r_r);
  divisor(2.0f * (float)f.tau_si, g.tau_2si, g.r_2si);
  divisor((float)f.tau_0, g.tau_0, g.r_0);
  divisor((float)f.tau_vp, g.tau_vp, g.r_vp);
  divisor((float)f.tau_v1m, g.tau_v1m, g.r_v1m);
  divisor((float)f.tau_v2m, g.tau_v2m, g.r_v2m);
  divisor((float)f.tau_wp, g.tau_wp, g.r_wp);
  divisor((float)f.tau_wm, g.tau_wm, g.r_wm);
  g.stim_on = stim_on;
  g.stim_x = stim_x;
  g.stim_y = stim_y;
  return g;
}

// a / t from the reciprocal r of t, itself correctly rounded: the quotient
// estimate a*r and its exact remainder give the correctly rounded quotient
// (Markstein, IBM J. Res. Dev. 34(1), 1990), in 3 instructions where a
// division takes 11; the FK currents have eight.  A quotient that is not finite
// may come out as a NaN.  t and r are normal, or both 0 for a quotient of 0
// (make_gparams).
__device__ __forceinline__ float g_quotient(float a, float t, float r) {
  const float e = a * r;
  return __builtin_fmaf(__builtin_fmaf(-t, e, a), r, e);
}

// Ionic currents (:131-141 for 2V, Fenton & Karma 1998 for FK) at a cell of
// the stage field; st: the mouse stimulus, 24.7 for a cell in its disk, else 0.
template <int MODEL>
__device__ __forceinline__ void g_currents(const GParams& g, float u, float v, float w, float st,
                                           float& Iu, float& Iv, float& Iw) {
  if (MODEL == M2V) {
    Iu = -(g.mu * u * (1.0f - u) * (u - g.alpha) - u * v) - st;
    Iv = -(g.eps * (g.delta * (u - g.gamma) * (g.beta - u) - v - g.theta));
    Iw = 0.0f;
  } else {
    // J_fi = -p v (1-u)(u-u_c)/tau_d, J_so = (1-p) u/tau_0 + p/tau_r,
    // J_si = -w (1 + tanh(k(u-u_csi)))/(2 tau_si), and the gates' rates: p and
    // q are 0 or 1, so each sum of two branches is the quotient of one.
    const bool p = u >= g.u_c, q = u >= g.u_v;
    const float J = g_quotient(p ? -v * (1.0f - u) * (u - g.u_c) : u, p ? g.tau_d : g.tau_0,
                               p ? g.r_d : g.r_0);
    const float J_si = g_quotient(-w * (1.0f + tanhf(g.kk * (u - g.u_csi))), g.tau_2si, g.r_2si);
    const float tvm = q ? g.tau_v2m : g.tau_v1m, rvm = q ? g.r_v2m : g.r_v1m;
    Iu = (p ? J + g.r_r : J) + J_si - st;
    Iv = g_quotient(p ? v : v - 1.0f, p ? g.tau_vp : tvm, p ? g.r_vp : rvm);
    Iw = g_quotient(p ? w : w - 1.0f, p ? g.tau_wp : g.tau_wm, p ? g.r_wp : g.r_wm);
  }
}

// Neighbour rules of a launch (a template constant: each keeps only its own
// registers and LDS arrays).
enum { G_SQUARE = 0, G_LAP4 = 1, G_ANISO = 2, G_LAP4_ANISO = 3, G_MASKED = 4, G_DIRICHLET = 5 };

// A launch advances K steps of `order` stages each, T = K * order stages in
// all.  A workgroup owns a region of 64 columns (one per lane) x `rows` rows;
// row lr belongs to wave lr % 16, so every stage's rows spread evenly over the
// four SIMDs as the region shrinks.  After T stages the inner region, `halo` =
// T * rad cells in from each side, is exact and written out; the ring is
// recomputed by the neighbouring workgroups.  rad is 1 cell per stage, 2 for
// the anisotropic no-flux branch (its edge corrections read two cells along
// the edge).
//
// What bounds it: a stage needs only the stage field and (lap4) the currents
// of the four to eight neighbours, so they live in LDS and every other value
// of a cell (the step's start, the accumulated rhs, the field itself, its
// current, its coefficients) stays in its lane's registers from load to store.
// Neighbours sit at fixed LDS offsets: a cell next to the domain edge also
// writes its value to its mirror image outside (no flux), or the outside holds
// the boundary value (Dirichlet), so no lane computes an index in the loop,
// and a cell's current is evaluated once per stage, not once per neighbour.
// The new state is written through to memory, since what is left dirty in the
// XCDs' L2 delays the end of the launch (RK4 at 1024 x 1024: 11.7 -> 10.9 us a
// step; below 512 x 512 no difference).
// One stage a launch through global memory, as this was before, took 8.7-9.1
// us a stage at 512 x 512 whatever the rule (40 dependent loads a cell).
constexpr int kGenWaves = 16, kGenThreads = 64 * kGenWaves;
constexpr int kGenPer = 3;                     // rows of a wave, at most
constexpr int kGenRows = kGenWaves * kGenPer;  // rows of a region, at most
constexpr int kGenPad = 2;                     // pad cells around the region in LDS
constexpr int kGenStride = 64 + 2 * kGenPad;
constexpr int kGenHalo = 12;
static_assert(kGenHalo <= kGenDeepest, "a step takes a ring cell and more");

struct GenRun {
  int K, order, rad, rows, halo, out_w, out_h, tiles_x, ntiles;
  float ki[5], sw[4];  // :70-95
};

// The values of a cell that neighbours read: u, and v of the 2V model (a
// 64-bit LDS access for the pair).
template <int MODEL>
struct GenPair {
  using type = float;
  static __device__ __forceinline__ float make(float u, float) { return u; }
  static __device__ __forceinline__ float get(float p, int) { return p; }
};
template <>
struct GenPair<M2V> {
  using type = float2;
  static __device__ __forceinline__ float2 make(float u, float v) { return make_float2(u, v); }
  static __device__ __forceinline__ float get(float2 p, int a) { return a ? p.y : p.x; }
};

template <int MODEL, int KIND>
struct GenLds {
  static constexpr bool LAP4 = KIND == G_LAP4 || KIND == G_LAP4_ANISO;
  static constexpr int N = (kGenRows + 2 * kGenPad) * kGenStride;
  typename GenPair<MODEL>::type y[2][N];               // stage field
  typename GenPair<MODEL>::type j[LAP4 ? 2 : 1][LAP4 ? N : 1];  // currents of the stage field
};

// Anisotropic term of variable a on the Neumann square branch (:249-356),
// scaled by s (1 for u, rscale for v).  Y(a, dx, dy) is the stage field at an
// offset from the cell; past an edge it is the mirrored cell (:207-221), whose
// value the corrections b amend.  edges: the workgroup holds cells of the west
// or east edge.
template <class YF>
__device__ __forceinline__ float g_aniso_neumann(const GParams& g, const YF& Y, int a, int i,
                                                 int j, float s, bool edges) {
  const int nx = g.nx, ny = g.ny;
  float b_S = 0.0f, b_N = 0.0f, b_W = 0.0f, b_E = 0.0f;
  float b_SW = 0.0f, b_SE = 0.0f, b_NW = 0.0f, b_NE = 0.0f;
  if (j == 0 || j == ny - 1) {  // the same for the whole wave
    const bool in = i > 0 && i < nx - 1, lo = j == 0;
    const float t = g.rby * (Y(a, 1, 0) - Y(a, -1, 0));
    b_S = lo && in ? t : 0.0f;
    b_N = !lo && in ? -t : 0.0f;
    // in the corner columns the west and east corrections take the side
    // away from this edge
    const float w2 = g.rby * (Y(a, 0, 0) - Y(a, -2, 0)), e2 = g.rby * (Y(a, 2, 0) - Y(a, 0, 0));
    const float w = i > 1 ? w2 : 0.0f, e = i < nx - 2 ? e2 : 0.0f;
    b_SW = lo ? w : 0.0f;
    b_SE = lo ? e : 0.0f;
    b_NW = lo ? 0.0f : -w;
    b_NE = lo ? 0.0f : -e;
  }
  if (edges) {  // some lane may hold a cell of the west or east edge
    const bool W = i == 0, E = i == nx - 1;
    const float t = j > 0 && j < ny - 1 ? g.rbx * (Y(a, 0, 1) - Y(a, 0, -1)) : 0.0f;
    b_W = W ? t : 0.0f;
    b_E = E ? -t : 0.0f;
    if (j > 1) {
      const float s2 = g.rbx * (Y(a, 0, 0) - Y(a, 0, -2));
      b_SW = W ? s2 : b_SW;
      b_SE = E ? -s2 : b_SE;
    }
    if (j < ny - 2) {
      const float n2 = g.rbx * (Y(a, 0, 2) - Y(a, 0, 0));
      b_NW = W ? n2 : b_NW;
      b_NE = E ? -n2 : b_NE;
    }
  }
  float d = ((b_S + b_N) * g.ry + (b_W + b_E) * g.rx) * s;
  d += g.rxy * ((Y(a, -1, -1) + b_SW) + (Y(a, 1, 1) + b_NE) - (Y(a, 1, -1) + b_SE) -
                (Y(a, -1, 1) + b_NW)) * s;
  return d;
}

// What a lane keeps of a cell for the whole launch.
struct GenCell {
  float y0[3], rhs[3], y[3], I[3];
  float stim;
  float cxx, cxy, cxz, cyx, cyy, cyz;  // G_MASKED: coefficients of :156-169
  uint32_t flags;                      // kGenTissue, kGenOut, kGenSide + n
};
constexpr uint32_t kGenTissue = 1u, kGenOut = 2u;
constexpr int kGenSide = 8;  // bits 8..15: neighbours W E N S SW NE SE NW usable (Dirichlet)

// The neighbours of a cell: the stage field W E N S SW NE SE NW, and the
// currents W E N S (lap4).
template <int MODEL>
struct GenNear {
  typename GenPair<MODEL>::type y[8], j[4];
};

// Increment of variable a in one stage at a cell, diffusion only (:97-490).
// Y2(a, dx, dy): the stage field two cells away (the anisotropic edges).
template <int MODEL, int KIND, bool LAP4, class Y2F>
__device__ __forceinline__ float g_diffusion(const GParams& g, const GenCell& q,
                                             const GenNear<MODEL>& n, const Y2F& Y2, int a, int i,
                                             int j, bool edges_x) {
  using P = GenPair<MODEL>;
  auto Y = [&](int k) { return P::get(n.y[k], a); };
  auto J = [&](int k) { return P::get(n.j[k], a); };
  const float c = q.y[a], I = q.I[a];
  float d;
  if (KIND == G_MASKED) {
    // :154-185 (lap4 and the anisotropic term are not applied, as in the reference)
    const float x = q.cxx * Y(0) - q.cxy * c + q.cxz * Y(1);
    const float y = q.cyx * Y(2) - q.cyy * c + q.cyz * Y(3);
    d = a == 0 ? x * g.rx + y * g.ry : x * g.rx * g.rscale + y * g.ry * g.rscale;
  } else if (KIND == G_DIRICHLET) {
    // :360-490: the field where the cell and the neighbour are tissue inside
    // the domain, else the boundary value
    auto B = [&](int k) { return ((q.flags >> (kGenSide + k)) & 1u) ? Y(k) : g.bval; };
    const float x = B(0) - 2.0f * c + B(1), y = B(2) - 2.0f * c + B(3);
    d = a == 0 ? x * g.rx + y * g.ry : x * g.rx * g.rscale + y * g.ry * g.rscale;
    if (g.aniso) {
      const float e = g.rxy * (B(4) + B(5) - B(6) - B(7));
      d += a == 0 ? e : e * g.rscale;
    }
  } else {
    // :188-199
    const float W = Y(0), E = Y(1), N = Y(2), S = Y(3);
    const float x = W - 2.0f * c + E, y = N - 2.0f * c + S;
    d = a == 0 ? x * g.rx + y * g.ry : x * g.rx * g.rscale + y * g.ry * g.rscale;
    if (LAP4) {
      // :201-247; J = the neighbours' currents in this stage
      const float z = (W - c + E) + (N - c + S);
      const float diag = Y(4) + Y(6) + Y(7) + Y(5);
      d += a == 0 ? -2.0f * g.q4 * z : -g.rscale * 2.0f * g.q4 * z;
      d += a == 0 ? g.q4 * diag : g.rscale * g.q4 * diag;
      d -= ((J(0) - 2.0f * I + J(1)) * g.fx4 + (J(2) - 2.0f * I + J(3)) * g.fy4);
    }
    if (KIND == G_ANISO || KIND == G_LAP4_ANISO) {
      auto YA = [&](int b, int dx, int dy) {
        return dx == 0 && dy == 0     ? c
               : dx == -1 && dy == 0  ? W
               : dx == 1 && dy == 0   ? E
               : dx == 0 && dy == 1   ? N
               : dx == 0 && dy == -1  ? S
               : dx == -1 && dy == -1 ? Y(4)
               : dx == 1 && dy == 1   ? Y(5)
               : dx == 1 && dy == -1  ? Y(6)
               : dx == -1 && dy == 1  ? Y(7)
                                      : Y2(b, dx, dy);
      };
      d += g_aniso_neumann(g, YA, a, i, j, a == 0 ? 1.0f : g.rscale, edges_x);
    }
  }
  return d;
}

template <int MODEL, int KIND, bool APD>
__global__ __launch_bounds__(kGenThreads) void k_general(
    const GParams g, const GenRun r, CFields in, Fields out, Fields vt, float* __restrict__ prev,
    const uint8_t* __restrict__ solid, const ApdState apd) {
  constexpr int NV = Model<MODEL>::NV;
  constexpr bool HOLES = KIND == G_MASKED || KIND == G_DIRICHLET;
  using L = GenLds<MODEL, KIND>;
  using P = GenPair<MODEL>;
  __shared__ L lds;
  const int tile = xcd_tile(blockIdx.x, r.ntiles);
  const int ty = tile / r.tiles_x, tx = tile - ty * r.tiles_x;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nx = g.nx, ny = g.ny;
  const int gx0 = tx * r.out_w - r.halo, gy0 = ty * r.out_h - r.halo;
  const int gi = gx0 + lane;
  const bool in_x = gi >= 0 && gi < nx;
  // the region holds cells of a domain edge (or beyond it)
  const bool edges_x = gx0 <= 0 || gx0 + 64 >= nx;
  const bool edges = edges_x || gy0 <= 0 || gy0 + r.rows >= ny;
  const bool vdiff = MODEL == M2V && g.vdiff != 0;
  // this lane's cell of the wave's first row, two rows and columns before it,
  // so every neighbour of every row lies at a constant offset >= 0
  const int l0 = wave * kGenStride + lane;
  auto off = [](int p, int dx, int dy) {
    return (p * kGenWaves + kGenPad + dy) * kGenStride + kGenPad + dx;
  };
  GenCell q[kGenPer];

  // The stage field (and currents) of row p's cell to LDS buffer b: at the
  // cell and, with no-flux boundaries, at its mirror images outside the domain
  // that lie in the region.
  auto put = [&](int b, int p, int lr, int gj, const GenCell& c) __attribute__((always_inline)) {
    const auto y = P::make(c.y[0], c.y[1]);
    const auto J = P::make(c.I[0], c.I[1]);
    auto at = [&](int dx, int dy) {
      const int l = l0 + off(p, 0, 0) + dy * kGenStride + dx;
      lds.y[b][l] = y;
      if (L::LAP4) lds.j[L::LAP4 ? b : 0][L::LAP4 ? l : 0] = J;
    };
    at(0, 0);
    if (KIND == G_DIRICHLET || !edges) return;
    // a cell next to an edge cell is the mirror image of the one past the
    // edge (helper_functions.cu:69-79)
    const int dx = gi == 1 ? -2 : gi == nx - 2 ? 2 : 0;
    const int dy = gj == 1 ? -2 : gj == ny - 2 ? 2 : 0;
    const bool hx = dx != 0 && lane + dx >= 0 && lane + dx < 64;
    const bool hy = dy != 0 && lr + dy >= 0 && lr + dy < r.rows;
    if (hx) at(dx, 0);
    if (hy) {
      at(0, dy);
      if (hx) at(dx, dy);
    }
  };
  auto currents = [&](GenCell& c) __attribute__((always_inline)) {
    g_currents<MODEL>(g, c.y[0], c.y[1], c.y[2], c.stim, c.I[0], c.I[1], c.I[2]);
  };

#pragma unroll
  for (int p = 0; p < kGenPer; ++p) {
    const int lr = wave + p * kGenWaves, gj = gy0 + lr;
    GenCell& c = q[p];
    c.flags = 0;
    c.stim = 0.0f;
#pragma unroll
    for (int a = 0; a < 3; ++a) c.y0[a] = c.rhs[a] = c.y[a] = c.I[a] = 0.0f;
    if (lr < r.rows && gj >= 0 && gj < ny && in_x) {
      const uint32_t idx = (uint32_t)gj * (uint32_t)nx + (uint32_t)gi;
#pragma unroll
      for (int a = 0; a < NV; ++a) c.y0[a] = c.y[a] = *at32(in.f[a], idx);
      if (g.stim_on) {  // :54-61: radius^2 < 400 cells
        const int di = gi - g.stim_x, dj = gj - g.stim_y;
        if (di * di + dj * dj < 400) c.stim = 24.7f;
      }
      c.flags = kGenTissue;
      if (lr >= r.halo && lr < r.halo + r.out_h && lane >= r.halo && lane < r.halo + r.out_w)
        c.flags |= kGenOut;
      if (KIND == G_MASKED) {
        const bool sc = solid[idx] != 0;
        const bool sw = solid[mirror(gi - 1, nx) + nx * gj] != 0;
        const bool se = solid[mirror(gi + 1, nx) + nx * gj] != 0;
        const bool sn = solid[gi + nx * mirror(gj + 1, ny)] != 0;
        const bool ss = solid[gi + nx * mirror(gj - 1, ny)] != 0;
        c.cxx = (sw && se) && (sw && sc) ? 1.0f : ((sw && sc) ? 2.0f : 0.0f);
        c.cxy = sc ? ((sw || se) ? 2.0f : 0.0f) : 0.0f;
        c.cxz = (sw && se) && (sc && se) ? 1.0f : ((sc && se) ? 2.0f : 0.0f);
        c.cyx = (sn && ss) && (sn && sc) ? 1.0f : ((sn && sc) ? 2.0f : 0.0f);
        c.cyy = sc ? ((sn || ss) ? 2.0f : 0.0f) : 0.0f;
        c.cyz = (sn && ss) && (sc && ss) ? 1.0f : ((sc && ss) ? 2.0f : 0.0f);
        if (!sc) c.flags &= ~kGenTissue;
      }
      if (KIND == G_DIRICHLET) {
        const bool sc = !solid || solid[idx] != 0;
        if (!sc) c.flags &= ~kGenTissue;
        const int ox[8] = {-1, 1, 0, 0, -1, 1, 1, -1}, oy[8] = {0, 0, 1, -1, -1, 1, -1, 1};
#pragma unroll
        for (int n = 0; n < 8; ++n) {
          if (n >= 4 && !g.aniso) break;  // only the cross term reads the diagonals
          const int ni = gi + ox[n], nj = gj + oy[n];
          const bool inside = ni >= 0 && ni < nx && nj >= 0 && nj < ny;
          if (inside && sc && (!solid || solid[ni + nx * nj] != 0))
            c.flags |= 1u << (kGenSide + n);
        }
      }
      currents(c);
      put(0, p, lr, gj, c);
    }
  }
  __syncthreads();

  const int T = r.K * r.order;
  int st = 0, step = 0;
  for (int t = 0; t < T; ++t) {
    const int b = t & 1;
    const bool last = st == r.order - 1, end = t == T - 1;
    const float wsum = r.sw[st], ki = r.ki[st + 1];
    const int lo = max(r.rad * (t + 1), -gy0), hi = min(r.rows - r.rad * (t + 1), ny - gy0);
    const auto* yb = lds.y[b] + l0;
    const auto* jb = lds.j[L::LAP4 ? b : 0] + (L::LAP4 ? l0 : 0);
    // Row p + 1's neighbours are read from LDS before row p's arithmetic, so
    // the LDS and the VALUs work at the same time (the reads are in bounds for
    // rows that take no part, too): 18.8 -> 16.1 us a launch of 8 lap4 stages
    // at 512 x 512.
    GenNear<MODEL> near;
    auto fetch = [&](int p) __attribute__((always_inline)) {
      constexpr bool diag = L::LAP4 || KIND == G_ANISO || KIND == G_DIRICHLET;
      const int ox[8] = {-1, 1, 0, 0, -1, 1, 1, -1}, oy[8] = {0, 0, 1, -1, -1, 1, -1, 1};
      GenNear<MODEL> n = {};
#pragma unroll
      for (int k = 0; k < (diag ? 8 : 4); ++k) n.y[k] = yb[off(p, ox[k], oy[k])];
      if (L::LAP4) {
#pragma unroll
        for (int k = 0; k < 4; ++k) n.j[k] = jb[L::LAP4 ? off(p, ox[k], oy[k]) : 0];
      }
      return n;
    };
    near = fetch(0);
#pragma unroll
    for (int p = 0; p < kGenPer; ++p) {
      const GenNear<MODEL> n = near;
      if (p + 1 < kGenPer) near = fetch(p + 1);
      const int lr = wave + p * kGenWaves, gj = gy0 + lr;
      if (lr < lo || lr >= hi) continue;
      GenCell& c = q[p];
      auto Y2 = [&](int a, int dx, int dy) { return P::get(yb[off(p, dx, dy)], a); };
      const float u0 = c.y0[0];
      // :498-499
      float d[3];
      d[0] = g_diffusion<MODEL, KIND, L::LAP4>(g, c, n, Y2, 0, gi, gj, edges_x) - g.dt * c.I[0];
      d[1] = vdiff ? g_diffusion<MODEL, KIND, L::LAP4>(g, c, n, Y2, 1, gi, gj, edges_x) -
                         g.dt * c.I[1]
                   : 0.0f - g.dt * c.I[1];
      d[2] = 0.0f - g.dt * c.I[2];
      // :501-503; the last stage gives y0 + tc*rhs, zero in holes (:506-561)
#pragma unroll
      for (int a = 0; a < NV; ++a) c.rhs[a] = c.rhs[a] + wsum * d[a];
      if (!last) {
#pragma unroll
        for (int a = 0; a < NV; ++a) c.y[a] = __builtin_fmaf(ki, d[a], c.y0[a]);
      } else {
        const bool sc = !HOLES || (c.flags & kGenTissue);
#pragma unroll
        for (int a = 0; a < NV; ++a) {
          const float x = c.y0[a] + g.tc * c.rhs[a];
          c.y0[a] = c.y[a] = sc ? x : 0.0f;
        }
        const bool owned = c.flags & kGenOut;
        const uint32_t idx = (uint32_t)gj * (uint32_t)nx + (uint32_t)gi;
        if (APD && owned && sc) apd_cell(apd, idx, u0, c.y[0], apd.count0 + step + 1);
        if (end && owned) {
#pragma unroll
          for (int a = 0; a < NV; ++a) {
            store_through(out.f[a], idx, c.y[a]);
            if (vt.f[0]) *at32(vt.f[a], idx) = sc ? c.rhs[a] / g.dt : 0.0f;
          }
          if (prev) store_through(prev, idx, u0);
        }
#pragma unroll
        for (int a = 0; a < NV; ++a) c.rhs[a] = 0.0f;
      }
      if (!end) {
        currents(c);
        if (in_x) put(b ^ 1, p, lr, gj, c);
      }
    }
    if (!end) __syncthreads();
    if (last) {
      st = 0;
      ++step;
    } else {
      ++st;
    }
  }
}

// Cells a stage reads to each side.
static int general_reach(const GParams& g) {
  return g.neumann && !g.masked && g.aniso ? 2 : 1;
}

static int general_depth(const GParams& g, int order, int halo) {
  return std::max(1, halo / (order * general_reach(g)));
}

// Steps to fuse and rows of a region on a device of `cus` compute units.  A
// launch takes about 4 us besides its stages and runs as many rounds as its
// workgroups fill, counted one a CU (16 waves; two of the square rule's without
// APD fit, of all others one); a row and stage costs c us on a CU.
// More steps a launch pay its fixed part less often and recompute a wider
// ring: RK4 with lap4 takes two steps a launch at 512 x 512 (17.3 against 2 x
// 10.1 us, one round either way) and one at 1024 x 1024 (22.2 us, two rounds,
// against 48.4, three).  The first choice is the pair with the least time per
// step, of up to 8 ring cells.  Where that fills one round, as up to about
// 512 x 512, 12 ring cells may pay too, and a call takes the depth whose full
// launches and remainder take the least time together, for an estimated gain of
// 4%, the estimate's spread (128 x 128, 5 steps of masked RK2: 11.7 us in
// launches of four and one, 9.2 in one; 40 RK4 steps 150.5 -> 138.9; 17
// Dirichlet steps at 512 x 512 31.3 -> 28.4).  With several rounds, which
// overlap in ways the estimate does not know, the same rule lost up to 9% as
// often as it gained.
GenTable general_table(int model, const GParams& g, int order, int steps, int cus) {
  const int rad = general_reach(g);
  const double fit = g.neumann && !g.masked ? (g.lap4 ? 0.025 : 0.0) + (g.aniso ? 0.04 : 0.0) : 0.0;
  auto rounds = [&](int K, int rows) {  // 0: no such region
    const int halo = K * order * rad, w = 64 - 2 * halo, h = rows - 2 * halo;
    if (h < 1) return 0;
    const int64_t tiles = (int64_t)((g.nx + w - 1) / w) * ((g.ny + h - 1) / h), n = std::max(1, cus);
    return (int)((tiles + n - 1) / n);
  };
  GenTable t;
  t.limit = std::min(steps, kGenDeepest);
  GenShape best{1, kGenRows};
  double least = 1e300;
  const double c = (model == M2V ? 0.025 : 0.05) + fit;
  for (int K = 1; K <= t.limit; ++K) {
    for (int rows = 8; rows <= kGenRows && K <= general_depth(g, order, 8); rows += 4) {
      const int n = rounds(K, rows);
      if (n == 0) continue;
      double us = 0.5;
      for (int s = 1; s <= K * order; ++s) us += std::max(0.2, c * (rows - 2 * rad * s));
      us = (4.0 + n * us) / K;
      if (us < least) {
        least = us;
        best = GenShape{K, rows};
      }
    }
    t.first[K] = best;
    t.round[K] = rounds(best.K, best.rows) == 1;
  }
  // one round: a stage is the chain of the wave with the most rows
  const double row = (model == M2V ? 0.33 : 0.75) + 16.0 * fit;
  for (int K = 1; K <= std::min(t.limit, general_depth(g, order, kGenHalo)); ++K) {
    int rows = 8;  // the fewest that do
    while (rows <= kGenRows && rounds(K, rows) != 1) rows += 4;
    if (rows > kGenRows) break;
    t.us[K] = 4.0;
    for (int s = 1; s <= K * order; ++s)
      t.us[K] += row * ((std::max(1, rows - 2 * rad * s) + kGenWaves - 1) / kGenWaves);
    t.rows[K] = rows;
    t.deepest = K;
  }
  return t;
}

// The next launch of a call with `steps` steps to go.
GenShape GenTable::next(int steps) const {
  const int n = std::min(steps, limit);
  if (!round[n] || first[n].K > deepest) return first[n];
  auto call = [&](int K) { return (steps / K) * us[K] + us[steps % K]; };
  GenShape best = first[n];
  double least = 0.96 * call(best.K);
  for (int K = 1; K <= std::min(n, deepest); ++K)
    if (call(K) < least) {
      least = call(K);
      best = GenShape{K, rows[K]};
    }
  return best;
}

hipError_t launch_general(int model, const GParams& g, int order, GenShape shape, CFields in, Fields out,
                          Fields vt, float* prev, const uint8_t* solid, hipStream_t s,
                          const ApdState* apd) {
  if (order != 1 && order != 2 && order != 4) return hipErrorInvalidValue;
  const int K = shape.K;
  if (K < 1 || K > general_depth(g, order, kGenHalo) || shape.rows > kGenRows) return hipErrorInvalidValue;
  // :70-95, RK4 weights as the reference writes them
  GenRun r = {};
  r.K = K;
  r.order = order;
  r.sw[0] = 1.0f;
  if (order == 2) {
    r.ki[1] = 0.5f;
    r.sw[0] = 0.0f;
    r.sw[1] = 1.0f;
  } else if (order == 4) {
    r.ki[1] = r.ki[2] = 0.5f;
    r.ki[3] = 1.0f;
    r.sw[0] = r.sw[3] = 0.166666666666667f;
    r.sw[1] = r.sw[2] = 0.333333333333333f;
  }
  r.rad = general_reach(g);
  r.halo = K * order * r.rad;
  r.out_w = 64 - 2 * r.halo;
  r.rows = shape.rows;
  r.out_h = r.rows - 2 * r.halo;
  if (r.out_w < 1 || r.out_h < 1) return hipErrorInvalidValue;
  r.tiles_x = (g.nx + r.out_w - 1) / r.out_w;
  r.ntiles = r.tiles_x * ((g.ny + r.out_h - 1) / r.out_h);
  const ApdState a = apd ? *apd : ApdState();
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(r.ntiles), dim3(kGenThreads), 0, s, g, r, in, out, vt, prev,
                       solid, a);
    return hipGetLastError();
  };
#define YH_GENERAL(KIND)                                                       \
  return model == M2V ? (apd ? go(k_general<M2V, KIND, true>) : go(k_general<M2V, KIND, false>)) \
                      : (apd ? go(k_general<MFK, KIND, true>) : go(k_general<MFK, KIND, false>))
  if (!g.neumann) YH_GENERAL(G_DIRICHLET);
  if (g.masked) YH_GENERAL(G_MASKED);
  if (g.lap4 && g.aniso) YH_GENERAL(G_LAP4_ANISO);
  if (g.lap4) YH_GENERAL(G_LAP4);
  if (g.aniso) YH_GENERAL(G_ANISO);
  YH_GENERAL(G_SQUARE);
#undef YH_GENERAL
}

}  // namespace yh
