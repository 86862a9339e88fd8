// fvwb_dgq.hip — the reference's own 2D modal DG program (2d/benchmark_2d_dg.f90
// with 2d/legendre.f90 and 2d/limiters.f90) on MI355X: the tensor-product (Q)
// Legendre basis of mx = my = O modes per direction, in FP64, equal to the
// reference bit for bit.
//
// What the reference evaluates with libm (the Gauss-Legendre rule by Newton's
// method, the basis values) is computed once on the host with the reference's
// expressions and handed to the kernels as a table; on the device there are
// only +, -, *, /, sqrt, min and max, written in the reference's order with
// contraction off, so they round as the reference's do.
//
// A stage of evolve, with its residual (compute_update, :1137-1479), its
// combination and its limiter (compute_positivity, 2d/limiters.f90:478-654), is
// one launch of dgq_stage_kernel; the dgq_speed_*_kernels are compute_max_speed
// (:826-870) with its bookkeeping and evolve's dt (:671), as exact block
// reductions.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <mutex>
#include <new>
#include <string>

#include "../../include/fvwb.h"
#include "fvwb_transfer.h"

#pragma clang fp contract(off)

namespace dgq {

constexpr int MAXO = 3;

// Basis and quadrature of one set-up (order O = mx = my).
struct Tab {
  double xq[MAXO], wq[MAXO];     // gl_quadrature(x_quad, w_quad, O)
  double L[MAXO][MAXO];          // L[a][n] = legendre(x_quad(a), n)
  double P[MAXO][MAXO];          // P[a][n] = legendre_prime(x_quad(a), n)
  double lm[MAXO], lp[MAXO];     // legendre(-1, n), legendre(+1, n)
  double Gl[MAXO][MAXO];         // Gl[c][n] = legendre(x_gll(c), n), compute_set's points
  int gll;
};

struct Geo {
  int nx, ny;
  int flux, source, gpc, bc, ninit, use_limiter;
  double gamma, boxlen_x, boxlen_y, odx, dx, eps, cfl, cmin;   // cmin = min(1/9, gll_w_1/2)
};

// The resident time loop's clock: dt of the current step, whether it runs, totals.
struct Clock {
  double t, dt, dt_last;
  long long steps;
  int active, err;
};

// One Runge-Kutta stage of evolve: out = (a X + am in) + (cdt dt) L, in that
// order, X or (own = 0) the stage's input absent from the sum; combine = 0
// writes L itself.  limit applies compute_positivity to the result.  With w5
// set, the stage also leaves w5 = ((b0 X + b1 Y) + bm in) + b4 out + (c5 dt) L,
// the last combination of 'RK4' and 'SS4' that takes the same L (the reference
// evaluates it twice, :700 and :723).  tick closes the step.
struct Epi {
  const double* X;
  double a, am, cdt;
  int combine, own, limit, tick;
  double* w5;
  const double* Y;
  double b0, b1, bm, b4, c5;
};

// ---- host: 2d/legendre.f90 as the reference evaluates it ------------------------
static double h_legendre(double x, int n) {
  x = std::min(std::max(x, -1.0), 1.0);
  const double x2 = x * x;
  double l = 0.0;
  switch (n) {
    case 0: l = 1.0; break;
    case 1: l = x; break;
    case 2: l = 0.5 * (3 * x2 - 1); break;
    case 3: l = 0.5 * (5.0 * (x2 * x) - 3.0 * x); break;
    case 4: l = 0.125 * (35.0 * (x2 * x2) - 30.0 * x2 + 3.0); break;
    case 5: l = 0.125 * (63.0 * (x2 * x2 * x) - 70.0 * (x2 * x) + 15.0 * x); break;
    case 6: l = 1.0 / 16.0 * (231.0 * (x2 * x2 * x2) - 315.0 * (x2 * x2) + 105.0 * x2 - 5.0); break;
    default: l = 0.0;
  }
  return std::sqrt(2.0 * (double)n + 1.0) * l;
}
static double h_legendre_prime(double x, int n) {
  x = std::min(std::max(x, -1.0), 1.0);
  const double x2 = x * x;
  double l = 0.0;
  switch (n) {
    case 0: l = 0.0; break;
    case 1: l = 1.0; break;
    case 2: l = 3.0 * x; break;
    case 3: l = 0.5 * (15.0 * x2 - 3.0); break;
    case 4: l = 0.125 * (140.0 * (x2 * x) - 60.0 * x); break;
    case 5: l = 0.125 * (315.0 * (x2 * x2) - 210.0 * x2 + 15.0); break;
    case 6: l = 1.0 / 16.0 * (1386.0 * (x2 * x2 * x) - 1260.0 * (x2 * x) + 210.0 * x); break;
    default: l = 0.0;
  }
  return std::sqrt(2.0 * (double)n + 1.0) * l;
}
// gl_quadrature (:77-108): the initial guess's coefficient in default REAL,
// 500 Newton steps, nodes sign-flipped, weights 2(2n+1)/((1-x^2) L'(x)^2),
// the second half mirrored.
static void h_gl_quadrature(int n, double* xq, double* wq) {
  const double dpi = std::acos(-1.0);
  for (int i = 1; i <= n; ++i) {
    const float nf = (float)n;
    const float c = (1.0f - 0.125f / nf / nf) + 0.125f / nf / nf / nf;
    double xx = (double)c * std::cos(dpi * (4.0 * (double)i - 1.0) / (4.0 * (double)n + 2.0));
    for (int it = 0; it < 500; ++it) xx = xx - h_legendre(xx, n) / h_legendre_prime(xx, n);
    xq[i - 1] = -xx;
    const double lp = h_legendre_prime(xq[i - 1], n);
    wq[i - 1] = 2 * (2.0 * (double)n + 1.0) / (1.0 - xq[i - 1] * xq[i - 1]) / (lp * lp);
  }
  for (int i = n / 2 + 1; i <= n; ++i) {
    xq[i - 1] = -xq[n - i];
    wq[i - 1] = wq[n - i];
  }
}

static Tab make_tab(int o) {
  Tab T{};
  h_gl_quadrature(o, T.xq, T.wq);
  for (int n = 0; n < o; ++n) {
    T.lm[n] = h_legendre(-1.0, n);
    T.lp[n] = h_legendre(1.0, n);
    for (int a = 0; a < o; ++a) {
      T.L[a][n] = h_legendre(T.xq[a], n);
      T.P[a][n] = h_legendre_prime(T.xq[a], n);
    }
  }
  // compute_positivity's point set uses gll_quadrature's points: (-1, 0) for
  // two points and (-1, 0, 1) for three (2d/legendre.f90:111-170 as written)
  T.gll = (2 * (o - 1) + 3) / 2;
  const double xg[3] = {-1.0, 0.0, 1.0};
  for (int c = 0; c < T.gll; ++c)
    for (int n = 0; n < o; ++n) T.Gl[c][n] = h_legendre(xg[c], n);
  return T;
}

// ---- device: the reference's point functions ------------------------------------
__device__ __forceinline__ double fmax_r(double a, double b) { return a > b ? a : b; }
__device__ __forceinline__ double fmin_r(double a, double b) { return a < b ? a : b; }

// compute_primitive (:891-902): density floored at the default-real 10e-10
__device__ __forceinline__ void prim(double gamma, const double u[4], double w[4]) {
  const double fl = (double)10e-10f;
  w[0] = u[0] > fl ? u[0] : fl;
  w[1] = u[1] / w[0];
  w[2] = u[2] / w[0];
  w[3] = (gamma - 1.0) * (u[3] - 0.5 * w[0] * (w[1] * w[1] + w[2] * w[2]));
}

// compute_flux (:919-944): f1 along x, f2 along y
__device__ __forceinline__ void flux_full(double gamma, const double u[4], double f1[4], double f2[4]) {
  double w[4];
  prim(gamma, u, w);
  f2[0] = w[0] * w[2];
  f2[1] = w[0] * w[1] * w[2];
  f2[2] = w[2] * u[2] + w[3];
  f2[3] = w[2] * u[3] + w[2] * w[3];
  f1[0] = w[0] * w[1];
  f1[1] = w[1] * u[1] + w[3];
  f1[2] = w[0] * w[1] * w[2];
  f1[3] = w[1] * u[3] + w[1] * w[3];
}

// compute_flux_int (:946-965) in one direction: dir 0 along x, 1 along y
__device__ __forceinline__ void flux_int(double gamma, const double u[4], int dir, double f[4]) {
  double w[4];
  prim(gamma, u, w);
  if (dir == 0) {
    f[0] = w[1] * u[0];
    f[1] = w[1] * u[1] + w[3];
    f[2] = w[0] * w[1] * w[2];
    f[3] = w[1] * u[3] + w[1] * w[3];
  } else {
    f[0] = w[2] * u[0];
    f[1] = w[0] * w[1] * w[2];
    f[2] = w[2] * u[2] + w[3];
    f[3] = w[2] * u[3] + w[2] * w[3];
  }
}

// compute_speed (:873-889)
__device__ __forceinline__ void speed(double gamma, const double u[4], double& cs, double& vx, double& vy,
                                      double& sp) {
  double w[4];
  prim(gamma, u, w);
  cs = sqrt(gamma * fmax(w[3], 1e-10) / fmax(w[0], 1e-10));
  vx = w[1];
  vy = w[2];
  sp = sqrt(w[1] * w[1] + w[2] * w[2]) + cs;
}

// compute_num_flux (:991-1006); flag 1 along x, 2 along y.  A flux_type of no
// branch (the shipped 'llf') and an HLLC state of no branch leave out at zero,
// the value the reference's F and G start from (:1317-1318).  HLLC is an
// instantiation of its own: its star states hold the stage kernel's registers
// (O = 2: 142 against 114, a wave per SIMD less).
template <bool HLLC>
__device__ __forceinline__ void num_flux(const Geo& g, const double ul[4], const double ur[4], const double fl[4],
                         const double fr[4], int flag, double out[4]) {
  out[0] = out[1] = out[2] = out[3] = 0.0;
  const double gamma = g.gamma;
  if (!HLLC && g.flux == FVWB_DGQ_FLUX_LLF1) {            // compute_llflux (:968-988)
    double csl, vxl, vyl, spl, csr, vxr, vyr, spr;
    speed(gamma, ul, csl, vxl, vyl, spl);
    speed(gamma, ur, csr, vxr, vyr, spr);
    const double cmax = flag == 1 ? fmax_r(fabs(vxr + csr), fabs(vxl + csl)) : fmax_r(fabs(vyr + csr), fabs(vyl + csl));
#pragma unroll
    for (int v = 0; v < 4; ++v) out[v] = 0.5 * (fr[v] + fl[v]) + 0.5 * cmax * (ul[v] - ur[v]);
  } else if (!HLLC && g.flux == FVWB_DGQ_FLUX_HLL2) {     // compute_hllflux (:1008-1026)
    double csl, vxl, vyl, spl, csr, vxr, vyr, spr;
    speed(gamma, ul, csl, vxl, vyl, spl);
    speed(gamma, ur, csr, vxr, vyr, spr);
    const double ap = fmax_r(0.0, fmax_r(csl + sqrt(vxl * vxl + vyl * vyl), csr + sqrt(vxr * vxr + vyr * vyr)));
    const double am = fmax_r(0.0, fmax_r(-(csl - sqrt(vxl * vxl + vyl * vyl)), -(csr - sqrt(vxr * vxr + vyr * vyr))));
#pragma unroll
    for (int v = 0; v < 4; ++v) out[v] = (ap * fl[v] + am * fr[v] - ap * am * (ur[v] - ul[v])) / (ap + am);
  } else if (HLLC) {     // compute_hllcflux (:1030-1134) as written
    double wl[4], wr[4], csl, vxl, vyl, spl, csr, vxr, vyr, spr;
    prim(gamma, ul, wl);
    prim(gamma, ur, wr);
    speed(gamma, ul, csl, vxl, vyl, spl);
    speed(gamma, ur, csr, vxr, vyr, spr);
    const double vl = flag == 1 ? vxl : vyl, vr = flag == 1 ? vxr : vyr;
    const double SL = fmin_r(vl, vr) - fmax_r(csl, csr);
    const double SR = fmax_r(vl, vr) + fmax_r(csl, csr);
    const double SM = (wr[0] * vr * (SR - vr) - wl[0] * vl * (SL - vl) + wl[3] - wr[3]) /
                      (wr[0] * (SR - vr) - wl[0] * (SL - vl));
    double usl[4], usr[4];
    usl[0] = ul[0] * (SL - vl) / (SL - SM);
    usr[0] = ur[0] * (SR - vr) / (SR - SM);
    if (flag == 1) {
      usl[1] = usl[0] * SM;
      usl[2] = usl[0] * wl[2];
      usl[3] = usl[0] * (ul[3] / ul[0] + (SM - wl[1]) * (SM + wl[3] / (wl[0] * (SL - wl[1]))));
      usr[1] = usr[0] * SM;
      usr[2] = usr[0] * wr[2];
      usr[3] = usr[0] * (ur[3] / ur[0] + (SM - wr[1] * (SM + wr[3] / (wr[0] * (SR - wr[1])))));
    } else {
      usl[1] = usl[0] * wl[1];
      usl[2] = usl[0] * SM;
      usl[3] = usl[0] * (ul[3] / ul[0] + (SM - wl[2]) * (SM + wl[3] / (wl[0] * (SL - wl[2]))));
      usr[1] = usr[0] * wl[1];                   // the left tangential velocity, as written
      usr[2] = usr[0] * SM;
      usr[3] = usr[0] * (ur[3] / ur[0] + (SM - wr[2] * (SM + wr[3] / (wr[0] * (SR - wr[2])))));
    }
    double f1[4], f2[4];
    int branch = 0;
    if (SL > 0.0) branch = 1;
    else if (SL <= 0.0 && SM > 0.0) branch = 2;
    else if (SR >= 0.0 && SM <= 0.0) branch = 3;
    else if (SR < 0.0) branch = 4;
    if (branch) {
      flux_full(gamma, branch <= 2 ? ul : ur, f1, f2);
      const double* f = flag == 1 ? f1 : f2;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if (branch == 1 || branch == 4) out[v] = f[v];
        else if (branch == 2) out[v] = f[v] + SL * (usl[v] - ul[v]);
        else out[v] = f[v] + SR * (usr[v] - ur[v]);
      }
    }
  }
}

// grad_phi (:1599-1644) at one point
__device__ __forceinline__ void grad_phi(int gcase, double x, double y, double& g0, double& g1) {
  if (gcase == 1) {
    g0 = x;
    g1 = y;
  } else if (gcase == 2) {
    const double epsilon = 0.25, delta_r = (double)0.1f, xd = x - 3., yd = y - 3.;
    const double r = sqrt(xd * xd + yd * yd);
    if (r > 0.5 - 0.5 * delta_r) {
      const double r3 = r * r * r;
      g0 = -(xd) / r3;
      g1 = -(yd) / r3;
    } else {
      g0 = -(xd) / (r * (r * r + epsilon * epsilon));
      g1 = -(yd) / (r * (r * r + epsilon * epsilon));
    }
  } else {
    g0 = g1 = 0.0;
  }
}

// ---- kernels ------------------------------------------------------------------
// Element (v, cell c, a, b) of a modal or nodal array at v + 4*(c + nc*(a + O*b)).
template <int O>
__device__ __forceinline__ long long at(int v, long long c, long long nc, int a, int b) {
  return (long long)v + 4 * (c + nc * ((long long)a + O * b));
}

// Lane layout of the stage and limiter kernels: lane 4 col + v holds the modes
// of variable v of the wave's cell col, which is the order of the arrays, so
// every load and store of a wave is one run of 16 cells x 4 variables.  Where a
// point needs all four variables (a node's fluxes, a pressure), the four lanes
// of a cell pass their values through a few KB of LDS of their own wave and
// take one point each.
constexpr int TX = 16;                             // cells of a wave, and of a tile in x

// orders a wave's own LDS writes before its other lanes' reads (and the reverse);
// the LDS serves one wave's accesses in order, so only the compiler is held
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ void get4(const double* s, double u[4]) {
#pragma unroll
  for (int v = 0; v < 4; ++v) u[v] = s[v];
}
__device__ __forceinline__ void put4(double* s, const double u[4]) {
#pragma unroll
  for (int v = 0; v < 4; ++v) s[v] = u[v];
}

// Products with the basis values.  Three exact properties of make_tab's values
// spare multiplications and registers without changing a result: the constant
// mode's value is 1; the points and weights are mirrored, so that mode n at the
// mirrored point is (-1)^n times its value here; and gll_quadrature's outer
// points are the cell's edges.  A product at a mirrored point is written as the
// sign of the other one, and the compiler forms it once.
// x legendre(x_quad(a), n)
template <int O>
__device__ __forceinline__ double times_l(const Tab& T, double x, int a, int n) {
  if (n == 0) return x;
  const bool mirror = a > (O - 1) / 2;
  const double r = x * T.L[mirror ? O - 1 - a : a][n];
  return mirror && n % 2 == 1 ? -r : r;
}
// the same for a point known only at run time
__device__ __forceinline__ double times_row(const Tab& T, double x, int a, int n) { return n == 0 ? x : x * T.L[a][n]; }
// x legendre(-1, n) or x legendre(+1, n)
__device__ __forceinline__ double times_edge(const Tab& T, double x, bool plus, int n) {
  if (n == 0) return x;
  const double r = x * T.lp[n];
  return !plus && n % 2 == 1 ? -r : r;
}
// x legendre(x_gll(c), n)
__device__ __forceinline__ double times_g(const Tab& T, double x, int c, int n) {
  if (n == 0) return x;
  return c == 1 ? x * T.Gl[1][n] : times_edge(T, x, c == 2, n);
}
// x legendre_prime(x_quad(a), n) w_quad(a), n >= 1
template <int O>
__device__ __forceinline__ double times_pw(const Tab& T, double x, int a, int n) {
  const bool mirror = a > (O - 1) / 2;
  const int k = mirror ? O - 1 - a : a;
  const double r = x * T.P[n == 1 ? 0 : k][n];
  return (mirror && n % 2 == 0 ? -r : r) * T.wq[k];
}
template <int O>
__device__ __forceinline__ double weight(const Tab& T, int a) {
  return T.wq[a > (O - 1) / 2 ? O - 1 - a : a];
}

// sum over the modes, i outer and j inner, of second(first(m[i][j])), in the
// reference's order of the factors
template <int O, class First, class Second>
__device__ __forceinline__ double expand(const double m[O][O], First first, Second second) {
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < O; ++i)
#pragma unroll
    for (int j = 0; j < O; ++j) s = s + second(first(m[i][j], i, j), i, j);
  return s;
}
// the trace at point q of a cell's x edge, of a cell's y edge, and the value at node (a, b)
template <int O>
__device__ __forceinline__ double trace_x(const Tab& T, const double m[O][O], bool plus, int q) {
  return expand<O>(m, [&](double x, int i, int) { return times_edge(T, x, plus, i); },
                   [&](double x, int, int j) { return times_l<O>(T, x, q, j); });
}
template <int O>
__device__ __forceinline__ double trace_y(const Tab& T, const double m[O][O], bool plus, int q) {
  return expand<O>(m, [&](double x, int, int j) { return times_edge(T, x, plus, j); },
                   [&](double x, int i, int) { return times_l<O>(T, x, q, i); });
}
template <int O>
__device__ __forceinline__ double node_value(const Tab& T, const double m[O][O], int a, int b) {
  return expand<O>(m, [&](double x, int i, int) { return times_row(T, x, a, i); },
                   [&](double x, int, int j) { return times_l<O>(T, x, b, j); });
}

// Mode (i, j) of a lane: a plane that is the same for the whole wave plus the
// lane's byte offset 8 (v + 4 c), which stays below 2^30 (2^24 cells).  One
// 32-bit register then addresses every plane of every array; as 64-bit indexes
// per plane the compiler kept 18 registers of addresses through the kernel.
template <int O>
__device__ __forceinline__ double& mode(double* u, unsigned lane_at, long long nc, int i, int j) {
  return *(double*)((char*)(u + 4 * nc * (i + O * j)) + lane_at);
}
template <int O>
__device__ __forceinline__ double mode(const double* u, unsigned lane_at, long long nc, int i, int j) {
  return *(const double*)((const char*)(u + 4 * nc * (i + O * j)) + lane_at);
}
template <int O>
__device__ __forceinline__ void load_modes(const double* __restrict__ u, unsigned lane_at, long long nc, double m[O][O]) {
#pragma unroll
  for (int j = 0; j < O; ++j)
#pragma unroll
    for (int i = 0; i < O; ++i) m[i][j] = mode<O>(u, lane_at, nc, i, j);
}
// element k of a per-cell array
__device__ __forceinline__ double cell_value(const double* plane, unsigned k) {
  return *(const double*)((const char*)plane + 8u * k);
}

// solve_for_t (2d/limiters.f90:312-362): the root in [0,1] of the quadratic
// whose zero puts the pressure of (1-t) u_avg + t u at eps
__device__ double solve_for_t(double gamma, double eps, const double u[4], const double ua[4]) {
  const double pa = ua[0], mxa = ua[1], mya = ua[2], ea = ua[3];
  const double pj = u[0], mxj = u[1], myj = u[2], ej = u[3];
  const double a = 2.0 * (pj - pa) * (ej - ea) - (mxj - mxa) * (mxj - mxa) - (myj - mya) * (myj - mya);
  double b = 2.0 * (pj - pa) * (ea - eps / (gamma - 1)) + 2.0 * pa * (ej - ea) -
             2.0 * (mxa * (mxj - mxa) + mya * (myj - mya));
  double cc = 2.0 * pa * ea - (mxa * mxa + mya * mya) - 2.0 * eps * pa / (gamma - 1.0);
  b = b / a;
  cc = cc / a;
  const double D = sqrt(fabs(b * b - 4 * cc));
  const double t1 = 0.5 * (-b - D), t2 = 0.5 * (-b + D);
  double t;
  if (t1 > -eps && t1 < 1.0 + eps) t = t1;
  else if (t2 > -eps && t2 < 1.0 + eps) t = t2;
  else t = 0.0;
  t = fmin(1.0, t);
  t = fmax(0.0, t);
  return t;
}

// compute_set's points (2d/limiters.f90:438-475): O x O at (x_gll(c), y_gl(q)),
// k = q O + c, then O x O at (x_gl(q), y_gll(c)); gll_quadrature gives O points
template <int O>
__device__ __forceinline__ double set_value(const Tab& T, const double m[O][O], int k) {
  const int q = k % (O * O) / O, c = k % O;
  return k < O * O ? expand<O>(m, [&](double x, int i, int) { return times_g(T, x, c, i); },
                               [&](double x, int, int j) { return times_l<O>(T, x, q, j); })
                   : expand<O>(m, [&](double x, int i, int) { return times_l<O>(T, x, q, i); },
                               [&](double x, int, int j) { return times_g(T, x, c, j); });
}

// compute_positivity (2d/limiters.f90:478-654) on the wave's 16 cells, m in the
// lane layout above: theta over the set's densities scales the non-mean density
// modes, then the smallest solve_for_t over the set points whose pressure
// (density floored at the default-real 10e-10) is not above eps scales every
// non-mean mode.  Both minima are exact, so the points may go in any order.
// The second minimum is formed beside the first, as if theta were 1; only a
// wave that has a theta below 1 goes over the set again with its scaled density.
struct LimitLds {
  double pts[4][TX][4];                            // four set points x cells x variables
  double avg[TX][4];
};

template <int O>
__device__ void limit_cells(const Geo& g, const Tab& T, LimitLds& s, double m[O][O]) {
  constexpr int NP = 2 * O * O;
  const int lane = threadIdx.x & 63, col = lane >> 2, v = lane & 3;
  const double eps = g.eps, gamma = g.gamma;
  double theta = 1.0, tmin = 1.;
  s.avg[col][v] = m[0][0];
#pragma unroll 1
  for (int pass = 0; pass < 2; ++pass) {
    double pmin = 0.0;
#pragma unroll
    for (int k0 = 0; k0 < NP; k0 += 4) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (k0 + k < NP) {
          const double p = set_value<O>(T, m, k0 + k);
          pmin = k0 + k == 0 ? p : fmin(pmin, p);
          s.pts[k][col][v] = p;
        }
      wave_lds_sync();
      if (k0 + v < NP) {
        double q[4];
        get4(s.pts[v][col], q);
        const double r = fmax(q[0], (double)10e-10f);
        const double vx = q[1] / r, vy = q[2] / r;
        const double pr = (gamma - 1.0) * (q[3] - 0.5 * r * (vx * vx + vy * vy));
        double t = 1.;
        if (!(pr > eps)) {
          double avg[4];
          get4(s.avg[col], avg);
          t = solve_for_t(gamma, eps, q, avg);
        }
        if (tmin >= t) tmin = t;
      }
      wave_lds_sync();
      __builtin_amdgcn_sched_barrier(0);           // a few values at a time
    }
    if (pass == 0 && v == 0) theta = fmin(fabs((m[0][0] - eps) / (m[0][0] - pmin)), 1.0);
    if (pass == 1 || !__any(theta != 1.0)) break;
    tmin = 1.;
#pragma unroll
    for (int i = 0; i < O; ++i)
#pragma unroll
      for (int j = 0; j < O; ++j)
        if (i != 0 || j != 0) m[i][j] = theta * m[i][j];
  }
#pragma unroll
  for (int x = 1; x < 4; x <<= 1) {
    const double t = __shfl_xor(tmin, x);
    if (tmin >= t) tmin = t;
  }
#pragma unroll
  for (int i = 0; i < O; ++i)
#pragma unroll
    for (int j = 0; j < O; ++j)
      if (i != 0 || j != 0) m[i][j] = tmin * m[i][j];
}

template <int O>
__global__ __launch_bounds__(256) void dgq_limit_kernel(Geo g, Tab T, double* __restrict__ u) {
  __shared__ LimitLds s[4];
  const long long nc = (long long)g.nx * g.ny;
  const int w = threadIdx.x >> 6, v = threadIdx.x & 3;
  const long long c = (long long)blockIdx.x * (4 * TX) + (threadIdx.x >> 2);
  double m[O][O];
  const unsigned la = 8u * (unsigned)(v + 4 * (c < nc ? c : nc - 1));   // lanes past the end repeat the last cell
  load_modes<O>(u, la, nc, m);
  limit_cells<O>(g, T, s[w], m);
  if (c >= nc) return;
#pragma unroll
  for (int j = 0; j < O; ++j)
#pragma unroll
    for (int i = 0; i < O; ++i) mode<O>(u, la, nc, i, j) = m[i][j];
}

// grad_phi at the nodes: it depends on the coordinates alone, so the resident
// loop forms it once per upload
__global__ __launch_bounds__(256) void dgq_grad_kernel(int gcase, long long n, const double* __restrict__ x,
                                                       const double* __restrict__ y, double* __restrict__ gx,
                                                       double* __restrict__ gy) {
  const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
  if (k < n) grad_phi(gcase, x[k], y[k], gx[k], gy[k]);
}

// One stage on a tile of TX x TY cells, a wave per row of 16 cells:
//   1. every lane expands its variable's modes to the cell's four traces
//      (:1253-1314); waves 0 to 2 also do the one trace that each neighbour of
//      the tile owes it (get_boundary_conditions :777-824 at the domain's edge);
//   2. a thread per face point: the traces' fluxes (compute_flux_int :946-965)
//      and compute_num_flux, written over the lower trace, which no other
//      thread reads;
//   3. O (or, for O = 2, all four) nodes at a time: node values, fluxes and
//      source by one lane per node, then every lane adds them to its variable's
//      volume and source integrals, a outer, b inner;
//   4. edge integrals, assembly (:1448-1466), special_boundary_conditions, the
//      Runge-Kutta combination, compute_positivity, and for the fourth 'RK4'
//      stage w5.
// Every sum takes its terms in the reference's order.
//
// Bound by FP64 issue: about 2,800 vector instructions per wave, 61 % of the
// issue slots at 512^2 and O = 3, 2.9 TB/s.  One launch instead of the four
// (traces, faces, cells, limiter) that moved 400 MB of traces and face fluxes
// and the state three more times per stage: 125 against 390 us per stage at
// 512^2, 8 against 32 at 16^2.  Tiles of 16 x 8 cells share more halo but hold
// twice the waves at each barrier: 165 us.  Four waves per SIMD (128
// registers) against three: 4 % faster.
template <int O, int TY>
struct StageLds {
  static constexpr int NB = O == 2 ? 4 : O;        // nodes per pass
  double yt[O][TY + 1][TX][4];                     // top traces of rows -1 .. TY-1, then the y face fluxes
  double xr[O][TY][TX + 1][4];                     // right traces of columns -1 .. TX-1, then the x face fluxes
  union {
    struct {
      double yb[O][TY + 1][TX][4];                 // bottom traces of rows 0 .. TY
      double xl[O][TY][TX + 1][4];                 // left traces of columns 0 .. TX
    } tr;
    union {
      double nodes[NB][3][TX][4];                  // f1 (first the node values), f2, s
      LimitLds lim;
    } wave[TY];
  } u;
};

template <int O, int TY, bool HLLC>
__global__ __launch_bounds__(64 * TY, 4) void dgq_stage_kernel(Geo g, Tab T, const double* __restrict__ in,
                                                            const double* __restrict__ x, const double* __restrict__ y,
                                                            const double* __restrict__ gx,
                                                            const double* __restrict__ gy, Epi e, double* out,
                                                            Clock* __restrict__ ck) {
  if (ck && !ck->active) return;
  using S = StageLds<O, TY>;
  __shared__ S s;
  const int nx = g.nx, ny = g.ny;
  const long long nc = (long long)nx * ny;
  const double dt = ck ? ck->dt : 0.0;
  // consecutive tiles on one XCD, whose L2 then holds the halo rows they share
  const int ntx = (nx + TX - 1) / TX, nt = gridDim.x, per = nt / 8, extra = nt % 8, xcd = blockIdx.x % 8;
  const int tile = xcd * per + (xcd < extra ? xcd : extra) + blockIdx.x / 8;
  const int i0 = (tile % ntx) * TX, j0 = (tile / ntx) * TY;
  const int wl = nx - i0 < TX ? nx - i0 : TX, hl = ny - j0 < TY ? ny - j0 : TY;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, col = lane >> 2, v = lane & 3;
  const bool own = col < wl && w < hl;
  // lanes outside the tile repeat its last cell and store nothing
  const unsigned c = (unsigned)(i0 + (col < wl ? col : wl - 1) + nx * (j0 + (w < hl ? w : hl - 1)));
  const unsigned la = 8u * (v + 4u * c);

  double m[O][O];
  load_modes<O>(in, la, nc, m);
  if (w < 3) {
    int hc = 0;
    bool has;
    if (w < 2) {                                   // the row below, the row above
      const int jh = w == 0 ? (j0 > 0 ? j0 - 1 : g.bc == 1 ? ny - 1 : 0)
                            : (j0 + hl < ny ? j0 + hl : g.bc == 1 ? 0 : ny - 1);
      has = col < wl;
      hc = i0 + (has ? col : 0) + nx * jh;
    } else {                                       // columns left and right
      const int r = col % TY;
      const int ih = col < TY ? (i0 > 0 ? i0 - 1 : g.bc == 1 ? nx - 1 : 0)
                              : (i0 + wl < nx ? i0 + wl : g.bc == 1 ? 0 : nx - 1);
      has = col < 2 * TY && r < hl;
      hc = ih + nx * (j0 + (has ? r : 0));
    }
    double mh[O][O];
    load_modes<O>(in, 8u * (v + 4u * hc), nc, mh);
    if (w < 2) {
#pragma unroll
      for (int q = 0; q < O; ++q) {
        const double lo = trace_y<O>(T, mh, false, q), hi = trace_y<O>(T, mh, true, q);
        if (has) *(w == 0 ? &s.yt[q][0][col][v] : &s.u.tr.yb[q][hl][col][v]) = w == 0 ? hi : lo;
      }
    } else {
      const bool left = col < TY;
#pragma unroll
      for (int q = 0; q < O; ++q) {
        const double lo = trace_x<O>(T, mh, false, q), hi = trace_x<O>(T, mh, true, q);
        if (has) *(left ? &s.xr[q][col % TY][0][v] : &s.u.tr.xl[q][col % TY][wl][v]) = left ? hi : lo;
      }
    }
  }
#pragma unroll
  for (int q = 0; q < O; ++q) {
    const double l = trace_x<O>(T, m, false, q), r = trace_x<O>(T, m, true, q);
    const double b = trace_y<O>(T, m, false, q), t = trace_y<O>(T, m, true, q);
    if (own) {
      s.u.tr.xl[q][w][col][v] = l;
      s.xr[q][w][col + 1][v] = r;
      s.u.tr.yb[q][w][col][v] = b;
      s.yt[q][w + 1][col][v] = t;
    }
  }
  __syncthreads();

  constexpr int NY = O * (TY + 1) * TX, NX = O * TY * (TX + 1);
#pragma unroll 1
  for (int k = tid; k < NY + NX; k += 64 * TY) {
    const bool xdir = k >= NY;
    const int kx = k - NY;
    if (xdir ? (kx % (TX + 1) > wl || kx / (TX + 1) % TY >= hl) : (k % TX >= wl || k / TX % (TY + 1) > hl)) continue;
    double* lo = xdir ? &s.xr[0][0][0][0] + 4 * kx : &s.yt[0][0][0][0] + 4 * k;
    const double* hi = xdir ? &s.u.tr.xl[0][0][0][0] + 4 * kx : &s.u.tr.yb[0][0][0][0] + 4 * k;
    double ul[4], ur[4], fl[4], fr[4], f[4];
    get4(lo, ul);
    get4(hi, ur);
    flux_int(g.gamma, ul, xdir ? 0 : 1, fl);
    flux_int(g.gamma, ur, xdir ? 0 : 1, fr);
    num_flux<HLLC>(g, ul, ur, fl, fr, xdir ? 1 : 2, f);
    put4(lo, f);
  }
  __syncthreads();

  // f1 P(a,0) and f2 P(b,0) are products with zero: the integrals of the modes
  // i = 0 (along x) and j = 0 (along y) are 0, or NaN if a flux is not finite
  constexpr int NB = S::NB;
  double fv1[O][O], fv2[O][O], sv[O][O], z1 = 0.0, z2 = 0.0;
#pragma unroll
  for (int i = 0; i < O; ++i)
#pragma unroll
    for (int j = 0; j < O; ++j) fv1[i][j] = fv2[i][j] = sv[i][j] = 0.0;
  const bool has_s = g.source != 1;
  double(*nd)[3][TX][4] = s.u.wave[w].nodes;
#pragma unroll 1
  for (int a0 = 0; a0 < O; a0 += NB / O) {
    // this lane's node of the pass (lane 3 of a cell has none for O = 3)
    const int an = O == 2 ? v >> 1 : a0, bn = O == 2 ? v & 1 : v;
    double g0 = 0.0, g1 = 0.0;
    if (g.source == 2 && bn < O) {
      const unsigned k = c + (unsigned)nc * (an + O * bn);
      g0 = cell_value(gx, k);
      g1 = cell_value(gy, k);
    }
#pragma unroll
    for (int k = 0; k < NB; ++k) {                 // get_nodes_from_modes (:544-592)
      const int a = O == 2 ? k / O : a0, b = k % O;
      nd[k][0][col][v] = node_value<O>(T, m, a, b);
    }
    wave_lds_sync();
    if (v < NB) {
      double u[4], f1[4], f2[4], sq[4] = {0.0, 0.0, 0.0, 0.0};
      get4(nd[v][0][col], u);
      flux_full(g.gamma, u, f1, f2);
      if (g.source == 2) {                         // get_source (:1558-1576)
        double p[4];
        prim(g.gamma, u, p);
        sq[1] = p[0] * g0;
        sq[2] = p[0] * g1;
        sq[3] = p[0] * (p[1] * g0 + p[2] * g1);
      } else if (g.source == 3) {                  // get_adv_source (:1579-1596)
        sq[0] = -1.0 * u[0];
      }
      put4(nd[v][0][col], f1);
      put4(nd[v][1][col], f2);
      if (has_s) put4(nd[v][2][col], sq);
    }
    wave_lds_sync();
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const int a = O == 2 ? k / O : a0, b = k % O;
      const double f1 = nd[k][0][col][v], f2 = nd[k][1][col][v];
      z1 = z1 + f1 * 0.0;
      z2 = z2 + f2 * 0.0;
#pragma unroll
      for (int i = 1; i < O; ++i) {
        const double f1i = f1 * T.P[a][i] * T.wq[a], f2j = times_pw<O>(T, f2, b, i);
#pragma unroll
        for (int j = 0; j < O; ++j) {
          fv1[i][j] = fv1[i][j] + times_l<O>(T, f1i, b, j) * weight<O>(T, b);
          fv2[j][i] = fv2[j][i] + times_row(T, f2j, a, j) * T.wq[a];
        }
      }
      if (has_s) {
        const double sq = nd[k][2][col][v];
#pragma unroll
        for (int i = 0; i < O; ++i) {
          const double si = times_row(T, sq, a, i) * T.wq[a];
#pragma unroll
          for (int j = 0; j < O; ++j) sv[i][j] = sv[i][j] + times_l<O>(T, si, b, j) * weight<O>(T, b);
        }
      }
    }
    wave_lds_sync();
  }

  // :1455-1462 (oneoverdx for the y terms too), the volume, x edge and y edge
  // terms one after the other so that few values are live at a time
  const double odx = g.odx;
  double d[O][O];
#pragma unroll
  for (int i = 0; i < O; ++i)
#pragma unroll
    for (int j = 0; j < O; ++j) d[i][j] = odx * (i == 0 ? z1 : fv1[i][j]) + odx * (j == 0 ? z2 : fv2[i][j]);
  __builtin_amdgcn_sched_barrier(0);
  {
    double fl[O], fr[O];
#pragma unroll
    for (int q = 0; q < O; ++q) {
      fl[q] = s.xr[q][w][col][v];
      fr[q] = s.xr[q][w][col + 1][v];
    }
#pragma unroll
    for (int i = 0; i < O; ++i)
#pragma unroll
      for (int j = 0; j < O; ++j) {
        double e1 = 0.0, e2 = 0.0;
#pragma unroll
        for (int q = 0; q < O; ++q) {              // :1377-1386
          e1 = e1 + times_l<O>(T, times_edge(T, fr[q], true, i), q, j) * weight<O>(T, q);
          e2 = e2 + times_l<O>(T, times_edge(T, fl[q], false, i), q, j) * weight<O>(T, q);
        }
        d[i][j] = d[i][j] - odx * (e1 - e2);
      }
  }
  __builtin_amdgcn_sched_barrier(0);
  {
    double gb[O], gt[O];
#pragma unroll
    for (int q = 0; q < O; ++q) {
      gb[q] = s.yt[q][w][col][v];
      gt[q] = s.yt[q][w + 1][col][v];
    }
#pragma unroll
    for (int j = 0; j < O; ++j)
#pragma unroll
      for (int i = 0; i < O; ++i) {
        double e3 = 0.0, e4 = 0.0;
#pragma unroll
        for (int q = 0; q < O; ++q) {              // :1391-1408
          e3 = e3 + times_l<O>(T, times_edge(T, gt[q], true, j), q, i) * weight<O>(T, q);
          e4 = e4 + times_l<O>(T, times_edge(T, gb[q], false, j), q, i) * weight<O>(T, q);
        }
        d[i][j] = (d[i][j] - odx * (e3 - e4)) / 2. + sv[i][j] / 4.;
      }
  }
  __builtin_amdgcn_sched_barrier(0);
  if (g.ninit == 12) {                             // special_boundary_conditions (:1481-1514)
#pragma unroll
    for (int i = 0; i < O; ++i)
#pragma unroll
      for (int j = 0; j < O; ++j) {
        const double xd = cell_value(x + nc * (i + O * j), c) - g.boxlen_x / 2.;
        const double yd = cell_value(y + nc * (i + O * j), c) - g.boxlen_y / 2.;
        if (sqrt(xd * xd + yd * yd) > 2.0) d[i][j] = 0.0;
      }
  }

  // w5 needs L and its leading terms once the result is limited: they wait in
  // their lane's elements of out and w5, which no other lane reads, and not in
  // registers
  if (own && e.w5) {
#pragma unroll
    for (int j = 0; j < O; ++j)
#pragma unroll
      for (int i = 0; i < O; ++i) {
        mode<O>(e.w5, la, nc, i, j) =
            e.b0 * mode<O>(e.X, la, nc, i, j) + e.b1 * mode<O>(e.Y, la, nc, i, j) + e.bm * m[i][j];
        mode<O>(out, la, nc, i, j) = d[i][j];
      }
  }
  if (e.combine) {
    if (e.X) {
      const double* X = e.X;
#pragma unroll
      for (int j = 0; j < O; ++j)
#pragma unroll
        for (int i = 0; i < O; ++i) {
          const double ax = e.a * mode<O>(X, la, nc, i, j);
          m[i][j] = e.own ? ax + e.am * m[i][j] : ax;
        }
    } else {
#pragma unroll
      for (int j = 0; j < O; ++j)
#pragma unroll
        for (int i = 0; i < O; ++i) m[i][j] = e.am * m[i][j];
    }
#pragma unroll
    for (int j = 0; j < O; ++j)
#pragma unroll
      for (int i = 0; i < O; ++i) d[i][j] = m[i][j] + e.cdt * dt * d[i][j];
  }
  if (e.limit) limit_cells<O>(g, T, s.u.wave[w].lim, d);
  if (own && e.w5) {
#pragma unroll
    for (int j = 0; j < O; ++j)
#pragma unroll
      for (int i = 0; i < O; ++i) {
        const double part = mode<O>(e.w5, la, nc, i, j), l = mode<O>(out, la, nc, i, j);
        mode<O>(e.w5, la, nc, i, j) = part + e.b4 * d[i][j] + e.c5 * dt * l;
      }
  }
  if (own) {
#pragma unroll
    for (int j = 0; j < O; ++j)
#pragma unroll
      for (int i = 0; i < O; ++i) mode<O>(out, la, nc, i, j) = d[i][j];
  }
  if (e.tick && blockIdx.x == 0 && tid == 0) {     // t = t + dt (:749); no block reads these
    ck->t = ck->t + dt;
    ck->dt_last = dt;
    ck->steps += 1;
  }
}

// the state of 'DEB', whose stage reads the neighbours of what it replaces
__global__ __launch_bounds__(256) void dgq_copy_kernel(long long n, const double* __restrict__ src,
                                                       double* __restrict__ dst, const Clock* __restrict__ ck) {
  if (!ck->active) return;
  for (long long k = (long long)blockIdx.x * 256 + threadIdx.x; k < n; k += (long long)gridDim.x * 256) dst[k] = src[k];
}

// get_nodes_from_modes / get_modes_from_nodes (:497-592) per cell, in the
// reference's loop order (modes a' outer, b' inner; for the modes the nodes
// a outer, b inner with 0.25 first)
template <int O, bool TO_NODES>
__global__ __launch_bounds__(256) void dgq_project_kernel(Geo g, Tab T, const double* __restrict__ src,
                                                          double* __restrict__ dst) {
  const long long nc = (long long)g.nx * g.ny;
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nc) return;
  double s[4][O][O];
#pragma unroll
  for (int i = 0; i < O; ++i)
#pragma unroll
    for (int j = 0; j < O; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) s[v][i][j] = src[at<O>(v, c, nc, i, j)];
#pragma unroll
  for (int i = 0; i < O; ++i)
#pragma unroll
    for (int j = 0; j < O; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        double acc = 0.0;
#pragma unroll
        for (int a = 0; a < O; ++a)
#pragma unroll
          for (int b = 0; b < O; ++b) {
            if (TO_NODES)
              acc = acc + s[v][a][b] * T.L[i][a] * T.L[j][b];
            else
              acc = acc + 0.25 * s[v][a][b] * T.L[a][i] * T.L[b][j] * T.wq[a] * T.wq[b];
          }
        dst[at<O>(v, c, nc, i, j)] = acc;
      }
}

// compute_max_speed (:826-870) over the cells in the reference's order
// k = i ny + j (x outer) and, with a clock, evolve's dt (:668-671).  The
// maximum speed S, the last k whose speed equals S (the last update of the
// reference's running ">=" test) and the smallest sound speed from that cell
// on (cs_max restarts there and only decreases) are each exact reductions, so
// their order does not matter.  Three launches: per block the pair (S_b, last
// k with speed S_b); per block the smallest sound speed at k >= k* (every
// block first combines the pairs itself); one block that combines everything,
// re-evaluates the cell k* and sets dt.  res = (cs_max, v_xmax, v_ymax,
// speed_max); part holds three doubles per block.
constexpr int SPEED_THREADS = 256;
constexpr int SPEED_MAX_BLOCKS = 1024;

__device__ __forceinline__ void cell_speed(const Geo& g, const double* __restrict__ u, long long m, double& cs,
                                           double& vx, double& vy, double& sp) {
  double q[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) q[v] = u[4 * m + v];
  speed(g.gamma, q, cs, vx, vy, sp);
}

// (s, k) pairs: the larger speed wins, equal speeds keep the larger k
__device__ __forceinline__ void pair_max(double& s, long long& k, double so, long long ko) {
  if (so > s) { s = so; k = ko; }
  else if (so == s && ko > k) k = ko;
}

__device__ __forceinline__ void wave_pair_max(double& s, long long& k) {
  for (int off = 32; off > 0; off >>= 1) {
    const double so = __shfl_xor(s, off);
    const long long ko = __shfl_xor(k, off);
    pair_max(s, k, so, ko);
  }
}

// a step that will not run (clock stopped or past t_end) skips the passes
__device__ __forceinline__ bool speed_runs(const Clock* ck, double t_end) {
  return !ck || (!ck->err && ck->t < t_end);
}

// the pairs of every block combined (each thread of the block strides over
// them, then the block reduces): S and k* (-1 when no speed reached S >= 0)
__device__ void combine_pairs(const double* part, int nblk, double& S, long long& ks) {
  __shared__ double sd[SPEED_THREADS / 64];
  __shared__ long long sk[SPEED_THREADS / 64];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  double s = 0.0;
  long long k = -1;
  for (int b = tid; b < nblk; b += SPEED_THREADS) pair_max(s, k, part[3 * b], (long long)part[3 * b + 1]);
  wave_pair_max(s, k);
  if (lane == 0) { sd[wv] = s; sk[wv] = k; }
  __syncthreads();
  s = sd[0];
  k = sk[0];
  for (int w = 1; w < SPEED_THREADS / 64; ++w) pair_max(s, k, sd[w], sk[w]);
  S = s;
  ks = k;
  __syncthreads();
}

__device__ void speed_pairs(const Geo& g, const double* __restrict__ u, double* part) {
  __shared__ double sd[SPEED_THREADS / 64];
  __shared__ long long sk[SPEED_THREADS / 64];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const long long nc = (long long)g.nx * g.ny;
  // speeds start at 0 with k = -1: a speed that is 0 joins the pair at 0, a
  // NaN never compares, as in the reference's running test from 0
  double s = 0.0;
  long long k = -1;
  for (long long m = (long long)blockIdx.x * SPEED_THREADS + tid; m < nc; m += (long long)gridDim.x * SPEED_THREADS) {
    double cs, vx, vy, sp;
    cell_speed(g, u, m, cs, vx, vy, sp);
    const long long km = (m % g.nx) * g.ny + m / g.nx;
    if (sp > s) { s = sp; k = km; }
    else if (sp == s && km > k) k = km;
  }
  wave_pair_max(s, k);
  if (lane == 0) { sd[wv] = s; sk[wv] = k; }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < SPEED_THREADS / 64; ++w) pair_max(s, k, sd[w], sk[w]);
    part[3 * blockIdx.x] = s;
    part[3 * blockIdx.x + 1] = (double)k;   // exact: k < 2^53
  }
}

__device__ void speed_csmin(const Geo& g, const double* __restrict__ u, double* part) {
  __shared__ double sd[SPEED_THREADS / 64];
  double S;
  long long ks;
  combine_pairs(part, gridDim.x, S, ks);
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const long long nc = (long long)g.nx * g.ny;
  double csm = INFINITY;
  if (ks >= 0)
    for (long long m = (long long)blockIdx.x * SPEED_THREADS + tid; m < nc; m += (long long)gridDim.x * SPEED_THREADS) {
      const long long km = (m % g.nx) * g.ny + m / g.nx;
      if (km < ks) continue;
      double cs, vx, vy, sp;
      cell_speed(g, u, m, cs, vx, vy, sp);
      if (csm > cs) csm = cs;
    }
  for (int off = 32; off > 0; off >>= 1) {
    const double o = __shfl_xor(csm, off);
    if (csm > o) csm = o;
  }
  if (lane == 0) sd[wv] = csm;
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < SPEED_THREADS / 64; ++w) if (csm > sd[w]) csm = sd[w];
    part[3 * blockIdx.x + 2] = csm;
  }
}

__device__ void speed_final(const Geo& g, const double* __restrict__ u, const double* part, int nblk,
                            double* __restrict__ res, Clock* __restrict__ ck, double t_end) {
  double S;
  long long ks;
  combine_pairs(part, nblk, S, ks);
  // the smallest of the blocks' sound-speed minima, in parallel
  __shared__ double sc[SPEED_THREADS / 64];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  double cmin = INFINITY;
  for (int b = tid; b < nblk; b += SPEED_THREADS) if (cmin > part[3 * b + 2]) cmin = part[3 * b + 2];
  for (int off = 32; off > 0; off >>= 1) {
    const double o = __shfl_xor(cmin, off);
    if (cmin > o) cmin = o;
  }
  if (lane == 0) sc[wv] = cmin;
  __syncthreads();
  if (tid != 0) return;
  for (int w = 1; w < SPEED_THREADS / 64; ++w) if (cmin > sc[w]) cmin = sc[w];
  double cs_max = 0.0, vxm = 0.0, vym = 0.0;
  if (ks >= 0) {
    const long long mb = (ks / g.ny) + (long long)g.nx * (ks % g.ny);
    double sp;
    cell_speed(g, u, mb, cs_max, vxm, vym, sp);
    if (cs_max > cmin) cs_max = cmin;
  }
  if (res) {
    res[0] = cs_max;
    res[1] = vxm;
    res[2] = vym;
    res[3] = S;
  }
  if (ck) {
    const double dtc = g.cfl * g.cmin / ((fabs(vxm) + (cs_max)) / g.dx + (fabs(vym) + (cs_max)) / g.dx);
    const double rest = t_end - ck->t;
    const double dt = rest < dtc ? rest : dtc;
    if (!(dt > 0.0) || !isfinite(dt)) {
      ck->err = 1;
      ck->active = 0;
      return;
    }
    ck->dt = dt;
    ck->active = 1;
  }
}

__global__ __launch_bounds__(SPEED_THREADS) void dgq_speed_pairs_kernel(Geo g, const double* __restrict__ u,
                                                                       double* __restrict__ part,
                                                                       const Clock* __restrict__ ck, double t_end) {
  if (speed_runs(ck, t_end)) speed_pairs(g, u, part);
}

__global__ __launch_bounds__(SPEED_THREADS) void dgq_speed_csmin_kernel(Geo g, const double* __restrict__ u,
                                                                       double* __restrict__ part,
                                                                       const Clock* __restrict__ ck, double t_end) {
  if (speed_runs(ck, t_end)) speed_csmin(g, u, part);
}

// the last of the three launches, or (alone: one block, small grids) all three
__global__ __launch_bounds__(SPEED_THREADS) void dgq_speed_final_kernel(Geo g, const double* __restrict__ u,
                                                                       double* part, int nblk, bool alone,
                                                                       double* __restrict__ res,
                                                                       Clock* __restrict__ ck, double t_end) {
  if (!speed_runs(ck, t_end)) {
    if (threadIdx.x == 0) ck->active = 0;
    return;
  }
  if (alone) {
    speed_pairs(g, u, part);
    __syncthreads();
    speed_csmin(g, u, part);
    __syncthreads();
  }
  speed_final(g, u, part, nblk, res, ck, t_end);
}

// compute_error (:23-89) per cell, then a fixed-order sum of the block
// partials: part[blk*12 + (0..3 max, 4..7 l1, 8..11 l2 sums)]
constexpr int ERR_THREADS = 256;

template <int O>
__global__ __launch_bounds__(ERR_THREADS) void dgq_error_kernel(Geo g, Tab T, const double* __restrict__ u,
                                                                const double* __restrict__ u0,
                                                                double* __restrict__ part) {
  __shared__ double sh[ERR_THREADS / 64][12];
  const long long nc = (long long)g.nx * g.ny;
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  double r[12];
  for (int k = 0; k < 12; ++k) r[k] = 0.0;
  if (c < nc) {
    const double cdx = 1. / (double)g.nx, cdy = 1. / (double)g.ny;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      double a1 = 0.0, a2 = 0.0, mx = 0.0;
#pragma unroll
      for (int a = 0; a < O; ++a)
#pragma unroll
        for (int b = 0; b < O; ++b) {
          const long long idx = at<O>(v, c, nc, a, b);
          const double d = u[idx] - u0[idx];
          mx = fmax(mx, fabs(d));
          a1 = a1 + fabs(d) * T.wq[a] * T.wq[b];
          a2 = a2 + d * d * T.wq[a] * T.wq[b];
        }
      r[v] = mx;
      r[4 + v] = a1 * (cdx * cdy) * 0.25;
      r[8 + v] = a2 * (cdx * cdy) * 0.25;
    }
  }
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (int k = 0; k < 12; ++k) {
    double x = r[k];
    for (int off = 32; off > 0; off >>= 1) {
      const double o = __shfl_xor(x, off);
      x = k < 4 ? fmax(x, o) : x + o;
    }
    if (lane == 0) sh[wv][k] = x;
  }
  __syncthreads();
  if (threadIdx.x < 12) {
    const int k = threadIdx.x;
    double x = sh[0][k];
    for (int w = 1; w < ERR_THREADS / 64; ++w) x = k < 4 ? fmax(x, sh[w][k]) : x + sh[w][k];
    part[(long long)blockIdx.x * 12 + k] = x;
  }
}

__global__ void dgq_error_final_kernel(const double* __restrict__ part, int nblk, double* __restrict__ res) {
  const int k = threadIdx.x;
  if (k >= 12) return;
  double x = 0.0;
  for (int b = 0; b < nblk; ++b) x = k < 4 ? fmax(x, part[(long long)b * 12 + k]) : x + part[(long long)b * 12 + k];
  res[k] = k >= 8 ? sqrt(x) : x;
}

}  // namespace dgq

using namespace dgq;

struct fvwb_dgq {
  fvwb_dgq_params p{};
  Geo g{};
  Tab T{};
  hipStream_t stream = nullptr;
  long long nc = 0, ns = 0;                  // cells, doubles per state
  double* du = nullptr;                      // resident state
  double* w[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};   // stage states
  double* s_in = nullptr;                    // drop-in staging
  double* s_out = nullptr;
  double *x = nullptr, *y = nullptr;         // resident coordinates
  double *xi = nullptr, *yi = nullptr;       // drop-in coordinates
  double *gx = nullptr, *gy = nullptr;       // grad_phi at the resident coordinates (source 2)
  double *gxi = nullptr, *gyi = nullptr;     // and at the drop-in's
  double* res = nullptr;                     // small results
  double* part = nullptr;                    // error partials
  Clock* clk = nullptr;
  bool loaded = false;
  fvwb_xfer::Staging xfer;  // large copies from and to host arrays
  std::string err;
};

static thread_local std::string g_errq;
// the message of the allocation-free entry point's last failure (a literal,
// so reporting it allocates nothing); cleared by every other failure
static thread_local const char* g_errq_static = nullptr;

static int failq(fvwb_dgq* h, int code, const std::string& msg) {
  (h ? h->err : g_errq) = msg;
  if (!h) g_errq_static = nullptr;
  return code;
}

#define HIPQ(h, call)                                                                                 \
  do {                                                                                                \
    hipError_t e_ = (call);                                                                           \
    if (e_ != hipSuccess) return failq(h, FVWB_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

extern "C" const char* fvwb_dgq_last_error(fvwb_dgq_handle h) {
  if (h) return h->err.c_str();
  return g_errq_static ? g_errq_static : g_errq.c_str();
}

extern "C" int fvwb_dgq_params_reference(fvwb_dgq_params* p) {
  if (!p) return failq(nullptr, FVWB_ERR_ARG, "NULL argument");
  *p = fvwb_dgq_params{};
  p->nx = p->ny = 8;
  p->order = 2;
  p->flux_type = FVWB_DGQ_FLUX_NONE;
  p->source = 1;
  p->grad_phi_case = 2;
  p->bc = 1;
  p->ninit = 1;
  p->solver = FVWB_DGQ_SOLVER_RK4;
  p->use_limiter = 1;
  p->gamma = (double)1.4f;
  p->boxlen_x = p->boxlen_y = 1.0;
  p->cfl = (double)0.2f;
  p->eps = (double)1e-10f;
  return FVWB_OK;
}

extern "C" int fvwb_dgq_destroy(fvwb_dgq_handle h) {
  if (!h) return FVWB_OK;
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  void* ps[] = {h->du, h->w[0], h->w[1], h->w[2], h->w[3], h->w[4], h->s_in, h->s_out, h->x, h->y, h->xi, h->yi,
                h->gx, h->gy, h->gxi, h->gyi, h->res, h->part, h->clk};
  for (void* q : ps)
    if (q) (void)hipFree(q);
  if (h->stream) (void)hipStreamDestroy(h->stream);
  delete h;
  return FVWB_OK;
}

static long long err_blocks(long long nc) { return (nc + ERR_THREADS - 1) / ERR_THREADS; }

// compute_max_speed (and, with a clock, evolve's dt) as three launches; the
// per-block partials use the handle's partial-sum buffer (3 doubles per block,
// at most err_blocks(nc) blocks)
static int speed_blocks(long long nc) {
  return (int)std::max(1LL, std::min<long long>((nc + SPEED_THREADS - 1) / SPEED_THREADS, SPEED_MAX_BLOCKS));
}
// up to four cells per thread of one block the one launch is the faster form:
// 45 against 52 us per 'RK4' step at 16^2, 76 against 78 at 32^2; at 64^2 the
// block is the bound (38 against 31 us per 'EQL' step)
static constexpr long long SPEED_ALONE_CELLS = 4 * SPEED_THREADS;
static void launch_speed(fvwb_dgq* h, const double* u, double* res, Clock* ck, double t_end) {
  const bool alone = h->nc <= SPEED_ALONE_CELLS;
  const int nb = alone ? 1 : speed_blocks(h->nc);
  if (!alone) {
    hipLaunchKernelGGL(dgq_speed_pairs_kernel, dim3(nb), dim3(SPEED_THREADS), 0, h->stream, h->g, u, h->part,
                       (const Clock*)ck, t_end);
    hipLaunchKernelGGL(dgq_speed_csmin_kernel, dim3(nb), dim3(SPEED_THREADS), 0, h->stream, h->g, u, h->part,
                       (const Clock*)ck, t_end);
  }
  hipLaunchKernelGGL(dgq_speed_final_kernel, dim3(1), dim3(SPEED_THREADS), 0, h->stream, h->g, u, h->part, nb, alone,
                     res, ck, t_end);
}

extern "C" int fvwb_dgq_create(fvwb_dgq_handle* out, const fvwb_dgq_params* p) {
  if (!out || !p) return failq(nullptr, FVWB_ERR_ARG, "NULL argument");
  *out = nullptr;
  // the reference passes dim = 2 to get_boundary_conditions for the x faces as
  // well (:1338-1339)
  if (p->nx < 1 || p->nx != p->ny)
    return failq(nullptr, FVWB_ERR_ARG,
                 "nx == ny >= 1 required (the reference's residual indexes the x faces with the y bounds)");
  if ((long long)p->nx * p->ny > (1ll << 24)) return failq(nullptr, FVWB_ERR_ARG, "more than 2^24 cells");
  if (p->order < 2 || p->order > 3) return failq(nullptr, FVWB_ERR_ARG, "order (mx = my) must be 2 or 3");
  if (p->flux_type < 0 || p->flux_type > 3) return failq(nullptr, FVWB_ERR_ARG, "flux_type must be 0..3");
  if (p->source < 1 || p->source > 3) return failq(nullptr, FVWB_ERR_ARG, "source must be 1, 2 or 3");
  if (p->grad_phi_case < 1 || p->grad_phi_case > 2) return failq(nullptr, FVWB_ERR_ARG, "grad_phi_case must be 1 or 2");
  if (p->bc < 1 || p->bc > 3) return failq(nullptr, FVWB_ERR_ARG, "bc must be 1, 2 or 3");
  if (p->solver < 0 || p->solver > 3) return failq(nullptr, FVWB_ERR_ARG, "solver must be 0..3");
  if (!(p->gamma > 1.0) || !(p->boxlen_x > 0.0) || !(p->boxlen_y > 0.0) || !(p->cfl > 0.0))
    return failq(nullptr, FVWB_ERR_ARG, "gamma > 1, positive box lengths and cfl required");
  fvwb_dgq* h = new (std::nothrow) fvwb_dgq;
  if (!h) return failq(nullptr, FVWB_ERR_OOM, "host allocation failed");
  h->p = *p;
  const int o = p->order;
  h->T = make_tab(o);
  const double dx = p->boxlen_x / (double)p->nx;
  const int gll = h->T.gll;
  // evolve's gll_w_1 (:650-655) in default REAL: 1e-10 vanishes against gll(gll-1)
  const double gll_w_1 = o == 1 ? 1. : 1. / (double)((float)(gll * (gll - 1)) + 1e-10f);
  const double c1 = 1. / (double)(2 * 4 + 1), c2 = gll_w_1 / 2.;
  h->g = Geo{p->nx, p->ny, p->flux_type, p->source, p->grad_phi_case, p->bc, p->ninit, p->use_limiter,
             p->gamma, p->boxlen_x, p->boxlen_y, 1. / dx, dx, p->eps, p->cfl, c1 < c2 ? c1 : c2};
  h->nc = (long long)p->nx * p->ny;
  h->ns = 4 * h->nc * o * o;
  const size_t sb = sizeof(double) * (size_t)h->ns, cb = sizeof(double) * (size_t)(h->nc * o * o);
  bool ok = hipStreamCreate(&h->stream) == hipSuccess && hipMalloc(&h->du, sb) == hipSuccess &&
            hipMalloc(&h->s_in, sb) == hipSuccess && hipMalloc(&h->s_out, sb) == hipSuccess &&
            hipMalloc(&h->x, cb) == hipSuccess && hipMalloc(&h->y, cb) == hipSuccess &&
            hipMalloc(&h->xi, cb) == hipSuccess && hipMalloc(&h->yi, cb) == hipSuccess &&
            hipMalloc(&h->res, 16 * sizeof(double)) == hipSuccess &&
            hipMalloc(&h->part, sizeof(double) * 12 * (size_t)err_blocks(h->nc)) == hipSuccess &&
            hipMalloc(&h->clk, sizeof(Clock)) == hipSuccess;
  for (int k = 0; ok && k < 5; ++k) ok = hipMalloc(&h->w[k], sb) == hipSuccess;
  if (p->source == 2)
    for (double** q : {&h->gx, &h->gy, &h->gxi, &h->gyi}) ok = ok && hipMalloc(q, cb) == hipSuccess;
  if (!ok) {
    fvwb_dgq_destroy(h);
    return failq(nullptr, FVWB_ERR_OOM, "device allocation failed");
  }
  *out = h;
  return FVWB_OK;
}

static dim3 cells_grid(const fvwb_dgq* h) { return dim3((unsigned)((h->nc + 255) / 256)); }

// the fields of the residual beside the state: coordinates and grad_phi
struct Coords {
  const double *x, *y, *gx, *gy;
};

static int gradients(fvwb_dgq* h, const double* x, const double* y, double* gx, double* gy) {
  if (h->p.source != 2) return FVWB_OK;
  const long long n = h->nc * h->p.order * h->p.order;
  hipLaunchKernelGGL(dgq_grad_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, h->stream, h->g.gpc, n, x, y, gx,
                     gy);
  HIPQ(h, hipGetLastError());
  return FVWB_OK;
}

template <int O, int TY>
static void launch_stage(fvwb_dgq* h, const double* in, const Coords& k, const Epi& e, double* out, Clock* ck) {
  const unsigned nt = (unsigned)(((h->p.nx + TX - 1) / TX) * ((h->p.ny + TY - 1) / TY));
  auto* kernel = h->p.flux_type == FVWB_DGQ_FLUX_HLLC ? dgq_stage_kernel<O, TY, true> : dgq_stage_kernel<O, TY, false>;
  hipLaunchKernelGGL(kernel, dim3(nt), dim3(64 * TY), 0, h->stream, h->g, h->T, in, k.x, k.y, k.gx, k.gy, e, out, ck);
}

// compute_update of `in` into `out` with the stage combination e (combine = 0:
// dudt itself); the clock gates and provides dt in the resident loop.  `out`
// may be e.X but not `in`, whose neighbours other tiles read.
static int stage(fvwb_dgq* h, const double* in, const Coords& k, const Epi& e, double* out, Clock* ck) {
  if (h->p.order == 2) launch_stage<2, 4>(h, in, k, e, out, ck);
  else launch_stage<3, 4>(h, in, k, e, out, ck);
  HIPQ(h, hipGetLastError());
  return FVWB_OK;
}

static int limit(fvwb_dgq* h, double* u) {
  if (!h->p.use_limiter) return FVWB_OK;
  const dim3 grid((unsigned)((h->nc + 4 * TX - 1) / (4 * TX)));
  if (h->p.order == 2)
    hipLaunchKernelGGL(dgq_limit_kernel<2>, grid, dim3(256), 0, h->stream, h->g, h->T, u);
  else
    hipLaunchKernelGGL(dgq_limit_kernel<3>, grid, dim3(256), 0, h->stream, h->g, h->T, u);
  HIPQ(h, hipGetLastError());
  return FVWB_OK;
}

static int project(fvwb_dgq* h, const double* src, double* dst, bool to_nodes) {
  if (h->p.order == 2) {
    if (to_nodes)
      hipLaunchKernelGGL((dgq_project_kernel<2, true>), cells_grid(h), dim3(256), 0, h->stream, h->g, h->T, src, dst);
    else
      hipLaunchKernelGGL((dgq_project_kernel<2, false>), cells_grid(h), dim3(256), 0, h->stream, h->g, h->T, src, dst);
  } else {
    if (to_nodes)
      hipLaunchKernelGGL((dgq_project_kernel<3, true>), cells_grid(h), dim3(256), 0, h->stream, h->g, h->T, src, dst);
    else
      hipLaunchKernelGGL((dgq_project_kernel<3, false>), cells_grid(h), dim3(256), 0, h->stream, h->g, h->T, src, dst);
  }
  HIPQ(h, hipGetLastError());
  return FVWB_OK;
}

static size_t state_bytes(const fvwb_dgq* h) { return sizeof(double) * (size_t)h->ns; }
static size_t coord_bytes(const fvwb_dgq* h) { return sizeof(double) * (size_t)(h->nc * h->p.order * h->p.order); }

extern "C" int fvwb_dgq_gl_quadrature(int32_t n, double* x_quad, double* w_quad) {
  if (!x_quad || !w_quad) return failq(nullptr, FVWB_ERR_ARG, "NULL argument");
  if (n < 1 || n > 6) return failq(nullptr, FVWB_ERR_ARG, "n must be 1..6 (legendre is defined up to 6)");
  h_gl_quadrature(n, x_quad, w_quad);
  return FVWB_OK;
}

extern "C" int fvwb_dgq_compute_update(fvwb_dgq_handle h, const double* delta_u, const double* x, const double* y,
                                       const double* u_eq, double* dudt) {
  (void)u_eq;      // unused by the reference (:1141)
  if (!h || !delta_u || !x || !y || !dudt) return failq(h, FVWB_ERR_ARG, "NULL argument");
  HIPQ(h, fvwb_xfer::to_device(h->xfer, h->s_in, delta_u, state_bytes(h), h->stream));
  HIPQ(h, fvwb_xfer::to_device(h->xfer, h->xi, x, coord_bytes(h), h->stream));
  HIPQ(h, fvwb_xfer::to_device(h->xfer, h->yi, y, coord_bytes(h), h->stream));
  int rc = gradients(h, h->xi, h->yi, h->gxi, h->gyi);
  if (rc || (rc = stage(h, h->s_in, Coords{h->xi, h->yi, h->gxi, h->gyi}, Epi{}, h->s_out, nullptr))) return rc;
  HIPQ(h, fvwb_xfer::to_host(h->xfer, dudt, h->s_out, state_bytes(h), h->stream));
  HIPQ(h, hipStreamSynchronize(h->stream));
  return FVWB_OK;
}

extern "C" int fvwb_dgq_compute_max_speed(fvwb_dgq_handle h, const double* u, double* cs_max, double* v_xmax,
                                          double* v_ymax, double* speed_max) {
  if (!h || !u || !cs_max || !v_xmax || !v_ymax || !speed_max) return failq(h, FVWB_ERR_ARG, "NULL argument");
  HIPQ(h, fvwb_xfer::to_device(h->xfer, h->s_in, u, sizeof(double) * 4 * (size_t)h->nc, h->stream));
  launch_speed(h, h->s_in, h->res, nullptr, 0.0);
  HIPQ(h, hipGetLastError());
  double r[4];
  HIPQ(h, hipMemcpyAsync(r, h->res, sizeof r, hipMemcpyDeviceToHost, h->stream));
  HIPQ(h, hipStreamSynchronize(h->stream));
  *cs_max = r[0];
  *v_xmax = r[1];
  *v_ymax = r[2];
  *speed_max = r[3];
  return FVWB_OK;
}

extern "C" int fvwb_dgq_apply_limiter(fvwb_dgq_handle h, double* u) {
  if (!h || !u) return failq(h, FVWB_ERR_ARG, "NULL argument");
  HIPQ(h, fvwb_xfer::to_device(h->xfer, h->s_in, u, state_bytes(h), h->stream));
  int rc = limit(h, h->s_in);
  if (rc) return rc;
  HIPQ(h, fvwb_xfer::to_host(h->xfer, u, h->s_in, state_bytes(h), h->stream));
  HIPQ(h, hipStreamSynchronize(h->stream));
  return FVWB_OK;
}

static int project_host(fvwb_dgq* h, const double* src, double* dst, bool to_nodes) {
  if (!h || !src || !dst) return failq(h, FVWB_ERR_ARG, "NULL argument");
  HIPQ(h, fvwb_xfer::to_device(h->xfer, h->s_in, src, state_bytes(h), h->stream));
  int rc = project(h, h->s_in, h->s_out, to_nodes);
  if (rc) return rc;
  HIPQ(h, fvwb_xfer::to_host(h->xfer, dst, h->s_out, state_bytes(h), h->stream));
  HIPQ(h, hipStreamSynchronize(h->stream));
  return FVWB_OK;
}

extern "C" int fvwb_dgq_modes_from_nodes(fvwb_dgq_handle h, const double* nodes, double* modes) {
  return project_host(h, nodes, modes, false);
}

extern "C" int fvwb_dgq_nodes_from_modes(fvwb_dgq_handle h, const double* modes, double* nodes) {
  return project_host(h, modes, nodes, true);
}

extern "C" int fvwb_dgq_upload(fvwb_dgq_handle h, const double* delta_u, const double* x, const double* y) {
  if (!h || !delta_u || !x || !y) return failq(h, FVWB_ERR_ARG, "NULL argument");
  const Clock zero{};
  HIPQ(h, fvwb_xfer::to_device(h->xfer, h->du, delta_u, state_bytes(h), h->stream));
  HIPQ(h, fvwb_xfer::to_device(h->xfer, h->x, x, coord_bytes(h), h->stream));
  HIPQ(h, fvwb_xfer::to_device(h->xfer, h->y, y, coord_bytes(h), h->stream));
  HIPQ(h, hipMemcpyAsync(h->clk, &zero, sizeof zero, hipMemcpyHostToDevice, h->stream));
  int rc = gradients(h, h->x, h->y, h->gx, h->gy);
  if (rc) return rc;
  HIPQ(h, hipStreamSynchronize(h->stream));
  h->loaded = true;
  return FVWB_OK;
}

static int read_clock(fvwb_dgq* h, Clock* c) {
  HIPQ(h, hipMemcpyAsync(c, h->clk, sizeof *c, hipMemcpyDeviceToHost, h->stream));
  HIPQ(h, hipStreamSynchronize(h->stream));
  return FVWB_OK;
}

// the 'RK4' (:683-710) and 'SS4' (:711-735) coefficients, default-real literals
static const float kRK4[16] = {0.391752226571890f, 0.444370493651235f, 0.555629506348765f, 0.368410593050371f,
                               0.620101851488403f, 0.379898148511597f, 0.251891774271694f, 0.178079954393132f,
                               0.821920045606868f, 0.544974750228521f, 0.00683325884039f,  0.51723167208978f,
                               0.12759831133288f,  0.34833675773694f,  0.08460416338212f,  0.22600748319395f};
static const float kSS4[16] = {0.39175222700392f, 0.44437049406734f, 0.55562950593266f, 0.36841059262959f,
                               0.6201018513854f,  0.37989814861460f, 0.25189177424738f, 0.17807995410773f,
                               0.82192004589227f, 0.54497475021237f, 0.00683325884039f, 0.51723167208978f,
                               0.12759831133288f, 0.34833675773694f, 0.08460416338212f, 0.22600748319395f};

// a X + am in + cdt dt L (X = nullptr, or am = 0: without that term)
static Epi epi(const fvwb_dgq* h, double a, const double* X, double am, double cdt, bool last = false) {
  Epi e{};
  e.X = X;
  e.a = a;
  e.am = am;
  e.cdt = cdt;
  e.combine = 1;
  e.own = am != 0.0;
  e.limit = h->p.use_limiter;
  e.tick = last;
  return e;
}

// One step of evolve's loop (:666-769): dt, the configured solver with
// apply_limiter after its stages, t = t + dt.
static int step(fvwb_dgq* h, double t_end) {
  Clock* ck = h->clk;
  double* du = h->du;
  double *w1 = h->w[0], *w2 = h->w[1], *w3 = h->w[2], *w4 = h->w[3], *w5 = h->w[4];
  launch_speed(h, du, nullptr, ck, t_end);
  HIPQ(h, hipGetLastError());
  int rc = 0;
  const Coords k{h->x, h->y, h->gx, h->gy};
  if (h->p.solver == FVWB_DGQ_SOLVER_EQL) {        // :672-681
    if ((rc = stage(h, du, k, epi(h, 0.0, nullptr, 1.0, 1.0), w1, ck))) return rc;
    return stage(h, w1, k, epi(h, 0.5, du, 0.5, 0.5, true), du, ck);
  }
  if (h->p.solver == FVWB_DGQ_SOLVER_DEB) {        // :737-747: w1 = du + dt L(du), limited, becomes du
    if ((rc = stage(h, du, k, epi(h, 0.0, nullptr, 1.0, 1.0, true), w1, ck))) return rc;
    hipLaunchKernelGGL(dgq_copy_kernel, dim3((unsigned)std::min<long long>((h->ns + 255) / 256, 8192)), dim3(256), 0,
                       h->stream, h->ns, (const double*)w1, du, (const Clock*)ck);
    HIPQ(h, hipGetLastError());
    return FVWB_OK;
  }
  const float* cf = h->p.solver == FVWB_DGQ_SOLVER_SS4 ? kSS4 : kRK4;   // 'RK4' / 'SS4'
  double c[16];
  for (int q = 0; q < 16; ++q) c[q] = (double)cf[q];
  if ((rc = stage(h, du, k, epi(h, 0.0, nullptr, 1.0, c[0]), w1, ck))) return rc;
  if ((rc = stage(h, w1, k, epi(h, c[1], du, c[2], c[3]), w2, ck))) return rc;
  if ((rc = stage(h, w2, k, epi(h, c[4], du, c[5], c[6]), w3, ck))) return rc;
  // w4 = c7 u + c8 w3 + c9 dt L(w3), and with w4 limited
  // w5 = c10 u + c11 w2 + c12 w3 + c13 w4 + c14 dt L(w3)
  Epi e4 = epi(h, c[7], du, c[8], c[9]);
  e4.w5 = w5;
  e4.Y = w2;
  e4.b0 = c[10]; e4.b1 = c[11]; e4.bm = c[12]; e4.b4 = c[13]; e4.c5 = c[14];
  if ((rc = stage(h, w3, k, e4, w4, ck))) return rc;
  // then L(w4) for the new state
  return stage(h, w4, k, epi(h, 1.0, w5, 0.0, c[15], true), du, ck);
}

static constexpr int32_t kGroupQ = 32;

extern "C" int fvwb_dgq_advance(fvwb_dgq_handle h, int32_t nsteps, double t_end) {
  if (!h) return failq(h, FVWB_ERR_ARG, "NULL handle");
  if (!h->loaded) return failq(h, FVWB_ERR_STATE, "advance before upload");
  if (nsteps < 0) return failq(h, FVWB_ERR_ARG, "nsteps must be >= 0");
  Clock c{};
  int rc = read_clock(h, &c);
  if (rc) return rc;
  int32_t done = 0;
  while (done < nsteps && !c.err && c.t < t_end) {
    const int32_t k = std::min(kGroupQ, nsteps - done);
    for (int32_t s = 0; s < k; ++s)
      if ((rc = step(h, t_end))) return rc;
    done += k;
    if ((rc = read_clock(h, &c))) return rc;
  }
  if (c.err) return failq(h, FVWB_ERR_NONPHYSICAL, "time step not finite and positive");
  return FVWB_OK;
}

extern "C" int fvwb_dgq_download(fvwb_dgq_handle h, double* delta_u) {
  if (!h || !delta_u) return failq(h, FVWB_ERR_ARG, "NULL argument");
  if (!h->loaded) return failq(h, FVWB_ERR_STATE, "download before upload");
  HIPQ(h, fvwb_xfer::to_host(h->xfer, delta_u, h->du, state_bytes(h), h->stream));
  HIPQ(h, hipStreamSynchronize(h->stream));
  return FVWB_OK;
}

extern "C" int fvwb_dgq_get_time(fvwb_dgq_handle h, double* t, double* dt_last, int64_t* steps) {
  if (!h) return failq(h, FVWB_ERR_ARG, "NULL handle");
  Clock c{};
  if (h->loaded) {
    int rc = read_clock(h, &c);
    if (rc) return rc;
  }
  if (t) *t = c.t;
  if (dt_last) *dt_last = c.dt_last;
  if (steps) *steps = c.steps;
  return FVWB_OK;
}

extern "C" int fvwb_dgq_compute_error(fvwb_dgq_handle h, const double* nodes, const double* u_init, double* linf,
                                      double* l1, double* l2) {
  if (!h || !u_init || !linf || !l1 || !l2) return failq(h, FVWB_ERR_ARG, "NULL argument");
  if (!nodes && !h->loaded) return failq(h, FVWB_ERR_STATE, "no nodal values and no uploaded state");
  if (nodes) {
    HIPQ(h, fvwb_xfer::to_device(h->xfer, h->s_out, nodes, state_bytes(h), h->stream));
  } else {
    int rc = project(h, h->du, h->s_out, true);
    if (rc) return rc;
  }
  HIPQ(h, fvwb_xfer::to_device(h->xfer, h->s_in, u_init, state_bytes(h), h->stream));
  const long long nb = err_blocks(h->nc);
  if (h->p.order == 2)
    hipLaunchKernelGGL(dgq_error_kernel<2>, dim3((unsigned)nb), dim3(ERR_THREADS), 0, h->stream, h->g, h->T,
                       h->s_out, h->s_in, h->part);
  else
    hipLaunchKernelGGL(dgq_error_kernel<3>, dim3((unsigned)nb), dim3(ERR_THREADS), 0, h->stream, h->g, h->T,
                       h->s_out, h->s_in, h->part);
  hipLaunchKernelGGL(dgq_error_final_kernel, dim3(1), dim3(64), 0, h->stream, h->part, (int)nb, h->res);
  HIPQ(h, hipGetLastError());
  double r[12];
  HIPQ(h, hipMemcpyAsync(r, h->res, sizeof r, hipMemcpyDeviceToHost, h->stream));
  HIPQ(h, hipStreamSynchronize(h->stream));
  for (int v = 0; v < 4; ++v) {
    linf[v] = r[v];
    l1[v] = r[4 + v];
    l2[v] = r[8 + v];
  }
  return FVWB_OK;
}

// ---- compute_error without allocation ------------------------------------------
// The block partials of dgq_error_kernel live in this file-scope array instead
// of a handle's allocation.  Its host-side name is only a stand-in: the device
// address comes from hipGetSymbolAddress, once per device, and only that
// address is handed to kernels.  Every call on a GPU shares that GPU's array;
// each block overwrites its own 12 partials and the final pass reads only the
// blocks of the current call, so nothing needs clearing, but calls that
// overlap on one GPU race.
static __device__ __align__(256) double scratch[12 * (FVWB_DGQ_NOALLOC_MAX_CELLS / ERR_THREADS)];

namespace {
constexpr int kMaxDevices = 64;
std::atomic<double*> g_scratch_ptr[kMaxDevices];
std::mutex g_scratch_mu;

// the device address of `scratch` on the current device (nullptr on failure)
double* scratch_address(int dev) {
  double* ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (ptr) return ptr;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  ptr = g_scratch_ptr[dev].load(std::memory_order_relaxed);
  if (ptr) return ptr;
  void* a = nullptr;
  if (hipGetSymbolAddress(&a, HIP_SYMBOL(scratch)) != hipSuccess || !a) return nullptr;
  ptr = static_cast<double*>(a);
  g_scratch_ptr[dev].store(ptr, std::memory_order_release);
  return ptr;
}

int fail_static(int code, const char* msg) {
  g_errq_static = msg;
  return code;
}
}  // namespace

extern "C" int fvwb_dgq_compute_error_noalloc(int32_t nx, int32_t ny, int32_t order, const double* nodes,
                                              const double* u_init, double* out, void* stream) {
  if (!nodes || !u_init || !out) return fail_static(FVWB_ERR_ARG, "NULL argument");
  if (nx < 1 || ny < 1) return fail_static(FVWB_ERR_ARG, "nx, ny >= 1 required");
  if (order < 2 || order > 3) return fail_static(FVWB_ERR_ARG, "order must be 2 or 3");
  const long long nc = (long long)nx * ny;
  if (nc > FVWB_DGQ_NOALLOC_MAX_CELLS)
    return fail_static(FVWB_ERR_ARG, "more cells than FVWB_DGQ_NOALLOC_MAX_CELLS (2^20): the scratch array "
                                     "holds the partial sums of that many cells");
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return fail_static(FVWB_ERR_HIP, "hipGetDevice failed or device index out of range");
  double* part = scratch_address(dev);
  if (!part) return fail_static(FVWB_ERR_HIP, "hipGetSymbolAddress of the scratch array failed");
  hipStream_t st = static_cast<hipStream_t>(stream);
  Geo g{};
  g.nx = nx;
  g.ny = ny;
  const Tab T = make_tab(order);
  const long long nb = err_blocks(nc);
  if (order == 2)
    hipLaunchKernelGGL(dgq_error_kernel<2>, dim3((unsigned)nb), dim3(ERR_THREADS), 0, st, g, T, nodes, u_init, part);
  else
    hipLaunchKernelGGL(dgq_error_kernel<3>, dim3((unsigned)nb), dim3(ERR_THREADS), 0, st, g, T, nodes, u_init, part);
  hipLaunchKernelGGL(dgq_error_final_kernel, dim3(1), dim3(64), 0, st, (const double*)part, (int)nb, out);
  if (hipGetLastError() != hipSuccess) return fail_static(FVWB_ERR_HIP, "kernel launch failed");
  return FVWB_OK;
}
