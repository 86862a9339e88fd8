// fvwb_fv2d_stage.h — the 2D finite-volume stage (gfx950, wave64): one wave's
// strip, and the kernel of one problem.
//
// One fused kernel per Runge-Kutta stage computes, for every cell, the
// well-balanced residual of compute_update_exact (benchmark_2d.f90:465-618) —
// reconstruction of the deviation dU at faces, numerical flux minus the
// equilibrium flux, source deviation — and the stage combination
// out = alpha*dU^n + beta*(dU_in + dt*L(dU_in)).  The last stage also reduces
// max(|v|+c) of the new state for the next dt (compute_max_speed,
// benchmark_2d.f90:264-279), so a whole run is enqueued without host syncs.
//
// Work decomposition: a wave owns a strip of 64 columns (2H of them halo,
// H = 1 first order, 2 MUSCL) and `rows` rows, and marches upward with a
// sliding register window.  x-neighbours come from DPP lane moves; y-neighbours
// from the window; each row is one coalesced 64-wide load per variable plane.
// Face fluxes are computed once: the x face on a lane's left, the y face above
// the current row (carried to the next row).
#pragma once

#include <type_traits>

#include "fvwb_device.h"
#include "fvwb_internal.h"

namespace fvwb {

enum { BC_FROZEN = 0, BC_REFLECT = 1 };
enum { MODE_RESIDUAL = 0, MODE_STAGE1 = 1, MODE_STAGE = 2 };

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// Read of a table that no kernel writes while a stage runs, through the
// constant address space: at a wave-uniform index it becomes a scalar load,
// which waits on its own counter and so never holds up on the row loads in
// flight (a vector load would, as vector loads complete in order).
__device__ __forceinline__ double table_at(const double* t, int k) {
  return ((const __attribute__((address_space(4))) double*)t)[k];
}

// Blocks are dealt round-robin to the 8 XCDs; renumber them so that each XCD
// receives a contiguous range of strips (neighbouring halos share its L2).
__device__ __forceinline__ int xcd_block(int b, int nb) {
  int xcd = b & 7, idx = b >> 3, base = nb >> 3, rem = nb & 7;
  return xcd * base + (xcd < rem ? xcd : rem) + idx;
}

// Row access through a buffer descriptor built on the scalar unit: base = the
// row's first element (uniform), extent = one variable's row, per-lane
// 32-bit byte offset.  No vector address arithmetic, and the hardware range
// check bounds every access to the row.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_rsrc(const void* row, int row_bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)row, 0, row_bytes, 0x00020000);
}
template <typename T>
__device__ __forceinline__ T ld1(const T* row, unsigned boff, int row_bytes) {
  if constexpr (sizeof(T) == 4)
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(row_rsrc(row, row_bytes), boff, 0, 0));
  else
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(row_rsrc(row, row_bytes), boff, 0, 0));
}

// A lane's block of C consecutive columns of one variable: one 4-, 8- or 16-byte load.
template <typename T, int C>
struct Lanes { T v[C]; };
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
// AUX is the buffer instruction's cache policy (0 = default).  Nontemporal
// policies were measured and did not help the stage kernels.
template <typename T, int C, int AUX = 0>
__device__ __forceinline__ Lanes<T, C> ldv(const T* row, unsigned boff, int row_bytes) {
  static_assert(C * sizeof(T) == 4 || C * sizeof(T) == 8 || C * sizeof(T) == 16, "block of 4, 8 or 16 bytes");
  if constexpr (C * sizeof(T) == 16)
    return __builtin_bit_cast(Lanes<T, C>, __builtin_amdgcn_raw_buffer_load_b128(row_rsrc(row, row_bytes), boff, 0, AUX));
  else if constexpr (C * sizeof(T) == 8)
    return __builtin_bit_cast(Lanes<T, C>, __builtin_amdgcn_raw_buffer_load_b64(row_rsrc(row, row_bytes), boff, 0, AUX));
  else
    return __builtin_bit_cast(Lanes<T, C>, __builtin_amdgcn_raw_buffer_load_b32(row_rsrc(row, row_bytes), boff, 0, AUX));
}
template <typename T, int C, int AUX = 0>
__device__ __forceinline__ void stv(T* row, unsigned boff, int row_bytes, Lanes<T, C> x) {
  if constexpr (C * sizeof(T) == 16)
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, x), row_rsrc(row, row_bytes), boff, 0, AUX);
  else if constexpr (C * sizeof(T) == 8)
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, x), row_rsrc(row, row_bytes), boff, 0, AUX);
  else
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, x), row_rsrc(row, row_bytes), boff, 0, AUX);
}

// Deviation state of a lane's C columns on one row.
template <typename T, int C>
struct Blk { Vec4<T> c[C]; };

// One wave computes one strip ("tile") of one instance.  The wave that owns
// tile 0 of an instance also does that instance's step bookkeeping: the first
// stage clears the next step's speed slots, the last stage advances t.  LAST
// (the step's last stage, a.last) is a template parameter so that the other
// stages carry no wave-speed code at all.
//
// SHORT is the form for strips of one or two rows, which small grids use: their
// few waves leave the chip idle, so a stage lasts as long as one wave, and a
// row costs a wave 1.1 us in FP32 and 1.6 us in FP64 (MUSCL, HLL) beside 5.5 us
// for the launch, the step control and the first rows' way from memory.  It
// sweeps upward only and ends with its last row instead of a ring's four.
template <typename T, int RECON, int FLUX, int BC, int FORM, int MODE, int CPL, bool LAST, bool SHORT = false>
__device__ __forceinline__ void stage_tile(const StageArgs<T>& a, const int tile, const int lane, const int slot) {
  // each lane owns CPL adjacent columns (8 or 16 bytes per variable plane);
  // lanes 0 and 63 are halo, so a wave produces 62*CPL columns
  constexpr int COLS = 62 * CPL;

  // ---- step control (dt from the previous step's reduction) -----------------
  double dt = 0.0;
  const int p = a.parity, q = p ^ 1;
  if (MODE != MODE_RESIDUAL) {
    const Ctrl* c = a.ctrl;
    const double t = c->t[p];
    const bool active = t < a.t_end;
    unsigned long long m = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) m = c->cmax[p][k].v > m ? c->cmax[p][k].v : m;
    // dt = 0.5*dx/cmax*cfl (benchmark_2d.f90:242)
    dt = 0.5 * a.h / __longlong_as_double((long long)m) * a.cfl;
    if (tile == 0 && lane < 8) {
      Ctrl* cw = a.ctrl;
      // a step past t_end changes nothing and carries the wave-speed maximum to
      // the next parity, so a later call with a larger t_end resumes from it
      if (a.first) cw->cmax[q][lane].v = active ? 0ull : c->cmax[p][lane].v;
      if (LAST && lane == 0) {
        cw->t[q] = active ? t + dt : t;
        if (active) { cw->steps_done += 1; cw->dt_last = dt; }
      }
    }
    if (!active) return;
  }

  const int tx = tile % a.ntx, ty = tile / a.ntx;
  const int nx = a.nx, ny = a.ny;
  const int xw = tx * COLS - CPL;              // first column of lane 0 (uniform)
  const int x0 = xw + CPL * lane;              // first column of this lane's block
  const int y0 = ty * a.rows;
  const int y1 = min(y0 + a.rows, ny);
  const bool own = lane >= 1 && lane <= 62 && x0 < nx;
  // interior strips read whole blocks; strips touching a side wall build their
  // halo column by column (mirror for walls, clamp for the frozen ring)
  const bool fast = xw >= 0 && xw + 64 * CPL <= nx;
  const long long plane = a.plane;
  const int pitch = a.pitch;
  // one variable's row holds min(pitch, plane) elements: pitch when the
  // variables are separate planes (plane = pitch * ny), plane when their rows
  // lie side by side (pitch = 4 * plane); every row access is bounded to it
  const int rowl = (long long)pitch < plane ? pitch : (int)plane;
  const int rowb = rowl * (int)sizeof(T);
  const unsigned vboff = (unsigned)clampi(x0, 0, rowl - CPL) * (unsigned)sizeof(T);

  auto load_row = [&](const T* base, int j) -> Blk<T, CPL> {
    int jc;
    bool flip = false;
    if (BC == BC_REFLECT) {
      jc = j < 0 ? -1 - j : (j >= ny ? 2 * ny - 1 - j : j);
      flip = j < 0 || j >= ny;
      jc = clampi(jc, 0, ny - 1);
    } else {
      jc = clampi(j, 0, ny - 1);
    }
    const T* r = base + (long long)jc * pitch;
    Blk<T, CPL> b;
    if (fast) {
      Lanes<T, CPL> v0 = ldv<T, CPL>(r, vboff, rowb), v1 = ldv<T, CPL>(r + plane, vboff, rowb),
                    v2 = ldv<T, CPL>(r + 2 * plane, vboff, rowb), v3 = ldv<T, CPL>(r + 3 * plane, vboff, rowb);
#pragma unroll
      for (int k = 0; k < CPL; ++k) b.c[k] = Vec4<T>{v0.v[k], v1.v[k], v2.v[k], v3.v[k]};
    } else {
#pragma unroll
      for (int k = 0; k < CPL; ++k) {
        int col = x0 + k, mc;
        T sxk = T(1);
        if (BC == BC_REFLECT) {
          mc = col < 0 ? -1 - col : (col >= nx ? 2 * nx - 1 - col : col);
          if (col < 0 || col >= nx) sxk = T(-1);
          mc = clampi(mc, 0, nx - 1);
        } else {
          mc = clampi(col, 0, nx - 1);
        }
        const unsigned o = (unsigned)mc * (unsigned)sizeof(T);
        b.c[k] = Vec4<T>{ld1(r, o, rowb), sxk * ld1(r + plane, o, rowb), ld1(r + 2 * plane, o, rowb),
                         ld1(r + 3 * plane, o, rowb)};
      }
    }
    if (BC == BC_REFLECT && flip) {
#pragma unroll
      for (int k = 0; k < CPL; ++k) b.c[k].my = -b.c[k].my;
    }
    return b;
  };
  // interior strips: every row and column read lies inside the grid, so a row
  // is four plain block loads with nothing applied to the loaded values (no
  // mirror, no per-column path), which lets the loads stay in flight until the
  // row that uses them
  auto load_row_interior = [&](const T* base, int j) -> Blk<T, CPL> {
    const T* r = base + (long long)clampi(j, 0, ny - 1) * pitch;
    Lanes<T, CPL> v0 = ldv<T, CPL>(r, vboff, rowb), v1 = ldv<T, CPL>(r + plane, vboff, rowb),
                  v2 = ldv<T, CPL>(r + 2 * plane, vboff, rowb), v3 = ldv<T, CPL>(r + 3 * plane, vboff, rowb);
    Blk<T, CPL> b;
#pragma unroll
    for (int k = 0; k < CPL; ++k) b.c[k] = Vec4<T>{v0.v[k], v1.v[k], v2.v[k], v3.v[k]};
    return b;
  };
  // U^n rows: only owned cells of the tile's own rows use them, so halo lanes,
  // lanes past nx and the ring's row beyond the tile read 0 through an offset
  // past the extent instead of memory (0.7 % faster in FP32, no result changes)
  auto load_cell = [&](const T* base, int j) -> Blk<T, CPL> {
    const T* r = base + (long long)clampi(j, 0, ny - 1) * pitch;
    const unsigned uo = (own && j >= y0 && j < y1) ? vboff : 0x80000000u;
    Lanes<T, CPL> v0 = ldv<T, CPL>(r, uo, rowb), v1 = ldv<T, CPL>(r + plane, uo, rowb),
                  v2 = ldv<T, CPL>(r + 2 * plane, uo, rowb), v3 = ldv<T, CPL>(r + 3 * plane, uo, rowb);
    Blk<T, CPL> b;
#pragma unroll
    for (int k = 0; k < CPL; ++k) b.c[k] = Vec4<T>{v0.v[k], v1.v[k], v2.v[k], v3.v[k]};
    return b;
  };

  // a face state D + h*s of a reconstruction (h = +-1/2).  The deviation form
  // writes it as one fused multiply-add per variable, so every launch shape
  // rounds it the same way: h*s is exact for normal numbers, but not for
  // subnormal ones, where a separate product would round first.  The FP64
  // form keeps the reference's product-then-sum.
  auto face_state = [](const Vec4<T>& D, T h, const Vec4<T>& s) -> Vec4<T> {
    if constexpr (FORM == FORM_DEV) {
      auto fm = [](T x, T y, T z) -> T {
        if constexpr (sizeof(T) == 4) return __builtin_fmaf(x, y, z);
        else return __builtin_fma(x, y, z);
      };
      return {fm(h, s.r, D.r), fm(h, s.mx, D.mx), fm(h, s.my, D.my), fm(h, s.e, D.e)};
    } else {
      return D + scale(h, s);
    }
  };

  Phys<T> P;
  P.gamma = T(a.gamma);
  P.gm1 = T(a.gamma - 1.0);
  P.half = T(0.5);
  P.g = T(a.g);
  P.ggm1 = T(a.gamma * (a.gamma - 1.0));
  P.gfloor = T(a.gamma * 1e-10);
  const T odx = T(a.odx), ody = T(a.ody);
  // stage combination out = alpha*U^n + beta*D + (beta*dt)*L
  const T alpha = T(a.alpha), beta = T(a.beta), bdt = T(a.beta * dt);
  // the deviation form folds beta*dt into the residual's factors
  const T kx = T(a.beta * dt * a.odx), ky = T(a.beta * dt * a.ody), kg = T(a.beta * dt * a.g);

  // separable FP64 equilibrium: rho = (rho0 e^{-kx}) e^{-ky} is formed in FP64
  // and rounded once; p, E and E+p scale with rho by constant ratios.
  double rxf[CPL], rxc[CPL];
#pragma unroll
  for (int k = 0; k < CPL; ++k) {
    rxf[k] = a.rxf[clampi(x0 + k, 0, nx)];        // left x face of column x0+k
    rxc[k] = a.rxc[clampi(x0 + k, 0, nx - 1)];
  }
  const T por = T(a.p_over_rho), eor = T(a.p_over_rho * a.inv_gm1);
  const T epor = T(a.p_over_rho * a.gamma * a.inv_gm1);
  const T gpor = T(a.p_over_rho * a.gamma);
  auto face_eq = [&](double rx, double ey) -> FaceEq<T> {
    FaceEq<T> f;
    f.rho = T(rx * ey);
    f.p = f.rho * por;
    f.e = f.rho * eor;
    f.ep = f.rho * epor;
    f.gp = f.rho * gpor;
    return f;
  };

  // the wave-speed maximum in the working precision (exact when widened)
  T smax = T(0);
  bool bad = false;

  // ---- the sweep ------------------------------------------------------------------
  // Even tile rows sweep upward, odd ones downward, so two vertically adjacent
  // tiles reach their shared halo rows at the same time and one of them finds
  // the rows in L2.  Both directions compute every face flux from the same two
  // states in the same order (lower, upper), so the results of the two agree
  // to an ulp (each is an instantiation whose products and sums may be fused
  // differently: Rusanov's are from the first stage on, HLL's in FP32 now and
  // then).
  // A ring of RING rows holds rows j, j+DIR, j+2DIR while row j is computed and
  // receives row j+(RING-1)DIR (one row in flight ahead of use); U^n uses a ring
  // of URING.  The body is unrolled RING times with rotated roles, so the rings
  // never move data.  (A deeper ring measured no faster: the strip sweep is
  // limited by its memory access pattern, not by loads in flight per wave.)
  auto sweep = [&](auto dirc, auto interiorc) {
    constexpr int DIR = decltype(dirc)::value;
    auto load_row_s = [&](const T* base, int j) -> Blk<T, CPL> {
      if constexpr (decltype(interiorc)::value) return load_row_interior(base, j);
      else return load_row(base, j);
    };
    constexpr int RING = 4;
    // FP64 holds U^n for one row only (loaded as the row starts, used as it
    // ends): that keeps its stage-2/3 kernel under 256 VGPRs, two waves per
    // SIMD instead of one.  FP32 keeps two rows at three waves, which measured
    // faster than one row at four.
    constexpr int URING = sizeof(T) == 8 ? 1 : 2;
    // slopes are differences along the sweep (minmod2(-a,-b) = -minmod2(a,b)), so a
    // row's state toward the next row is D + sy/2 and toward the previous D - sy/2
    const T hd = P.half;
    const int js = DIR > 0 ? y0 : y1 - 1;      // first row of the sweep
    Blk<T, CPL> R[RING], Ur[URING], sy, Gp;
    // flux through the face between row jb (behind, state Db) and row ja (ahead, Da)
    auto yface = [&](const FaceEq<T>& qy, const Vec4<T>& Db, const Vec4<T>& Da) {
      if constexpr (DIR > 0) return face_flux<T, FLUX, 1, FORM>(P, qy, Db, Da);
      else return face_flux<T, FLUX, 1, FORM>(P, qy, Da, Db);
    };
    {
      const double eyf0 = table_at(a.eyf, clampi(js + (DIR < 0), 0, ny));
      Blk<T, CPL> Dm1 = load_row_s(a.in, js - DIR);
#pragma unroll
      for (int k = 0; k < RING - 1; ++k) R[k] = load_row_s(a.in, js + k * DIR);
      Blk<T, CPL> Dm2;
      if (RECON) Dm2 = load_row_s(a.in, js - 2 * DIR);
#pragma unroll
      for (int k = 0; k < CPL; ++k) {
        FaceEq<T> qy = face_eq(rxc[k], eyf0);
        if (RECON) {
          Vec4<T> sym1 = minmod2(Dm1.c[k] - Dm2.c[k], R[0].c[k] - Dm1.c[k]);
          sy.c[k] = minmod2(R[0].c[k] - Dm1.c[k], R[1].c[k] - R[0].c[k]);
          Gp.c[k] = yface(qy, face_state(Dm1.c[k], hd, sym1), face_state(R[0].c[k], -hd, sy.c[k]));
        } else {
          Gp.c[k] = yface(qy, Dm1.c[k], R[0].c[k]);
        }
      }
#pragma unroll
      for (int k = 0; k < URING; ++k) Ur[k] = Blk<T, CPL>{};
      if (MODE == MODE_STAGE) {
#pragma unroll
        for (int k = 0; k < URING - 1; ++k) Ur[k] = load_cell(a.un, js + k * DIR);
      }
    }

    // one row: A = row j, B = row j+DIR, C = row j+2DIR; S receives row
    // j+(RING-1)DIR; UA holds U^n(j) and US receives U^n(j+(URING-1)DIR).
    auto row_step = [&](int j, const Blk<T, CPL>& A, const Blk<T, CPL>& B, const Blk<T, CPL>& C,
                        Blk<T, CPL>& S, const Blk<T, CPL>& UA, Blk<T, CPL>& US) {
      S = load_row_s(a.in, j + (RING - 1) * DIR);
      if (MODE == MODE_STAGE) US = load_cell(a.un, j + (URING - 1) * DIR);
      const int jt = clampi(j, 0, ny - 1);
      const double eyc = table_at(a.eyc, jt);
      const double eyf = table_at(a.eyf, jt + (DIR > 0));

      // y faces between row j and row j+DIR
      Blk<T, CPL> Gn;
#pragma unroll
      for (int k = 0; k < CPL; ++k) {
        FaceEq<T> qy = face_eq(rxc[k], eyf);
        if (RECON) {
          Vec4<T> syn = minmod2(B.c[k] - A.c[k], C.c[k] - B.c[k]);
          Gn.c[k] = yface(qy, face_state(A.c[k], hd, sy.c[k]), face_state(B.c[k], -hd, syn));
          sy.c[k] = syn;
        } else {
          Gn.c[k] = yface(qy, A.c[k], B.c[k]);
        }
      }
      // x faces on the left of each column; the first takes its left state from
      // the neighbouring lane's last column, the last column's right face is the
      // right neighbour's first
      Vec4<T> xr[CPL], xl[CPL];
      if (RECON) {
        Vec4<T> lm = from_left(A.c[CPL - 1]), rp = from_right(A.c[0]);
#pragma unroll
        for (int k = 0; k < CPL; ++k) {
          Vec4<T> am = k == 0 ? lm : A.c[k - 1];
          Vec4<T> ap = k == CPL - 1 ? rp : A.c[k + 1];
          Vec4<T> sx = minmod2(A.c[k] - am, ap - A.c[k]);
          xr[k] = face_state(A.c[k], P.half, sx);
          xl[k] = face_state(A.c[k], -P.half, sx);
        }
      } else {
#pragma unroll
        for (int k = 0; k < CPL; ++k) xr[k] = xl[k] = A.c[k];
      }
      Vec4<T> F[CPL + 1];
      const Vec4<T> xr_left = from_left(xr[CPL - 1]);
#pragma unroll
      for (int k = 0; k < CPL; ++k)
        F[k] = face_flux<T, FLUX, 0, FORM>(P, face_eq(rxf[k], eyc), k == 0 ? xr_left : xr[k - 1], xl[k]);
      F[CPL] = from_right(F[0]);

      Blk<T, CPL> O;
#pragma unroll
      for (int k = 0; k < CPL; ++k) {
        const Vec4<T>& D = A.c[k];
        // residual: -dF/dx - dG/dy + (s(U) - s(U_eq)), s = (0, -rho g, -rho g, -g (m_x+m_y));
        // the same expression in both directions, on the flux above (Ga) and below (Gb)
        const Vec4<T>& Ga = DIR > 0 ? Gn.c[k] : Gp.c[k];
        const Vec4<T>& Gb = DIR > 0 ? Gp.c[k] : Gn.c[k];
        const bool frozen =
            BC == BC_FROZEN && (x0 + k == 0 || x0 + k == nx - 1 || j == 0 || j == ny - 1);
        if (FORM == FORM_DEV && MODE != MODE_RESIDUAL) {
          // out = base - kx dF - ky dG + kg s, base = D (stage 1) or alpha U^n + beta D
          Vec4<T> B = D;
          if (MODE == MODE_STAGE) B = scale(alpha, UA.c[k]) + scale(beta, D);
          Vec4<T> Q;
          Q.r = B.r - kx * (F[k + 1].r - F[k].r) - ky * (Ga.r - Gb.r);
          Q.mx = B.mx - kx * (F[k + 1].mx - F[k].mx) - ky * (Ga.mx - Gb.mx) - kg * D.r;
          Q.my = B.my - kx * (F[k + 1].my - F[k].my) - ky * (Ga.my - Gb.my) - kg * D.r;
          Q.e = B.e - kx * (F[k + 1].e - F[k].e) - ky * (Ga.e - Gb.e) - kg * (D.mx + D.my);
          O.c[k] = frozen ? B : Q;
        } else {
          Vec4<T> L;
          L.r = -(F[k + 1].r - F[k].r) * odx - (Ga.r - Gb.r) * ody;
          L.mx = (-(F[k + 1].mx - F[k].mx) * odx - (Ga.mx - Gb.mx) * ody) - P.g * D.r;
          L.my = (-(F[k + 1].my - F[k].my) * odx - (Ga.my - Gb.my) * ody) - P.g * D.r;
          L.e = (-(F[k + 1].e - F[k].e) * odx - (Ga.e - Gb.e) * ody) - P.g * (D.mx + D.my);
          if (frozen) L = {T(0), T(0), T(0), T(0)};
          if (MODE == MODE_RESIDUAL) {
            O.c[k] = L;
          } else if (MODE == MODE_STAGE1) {
            O.c[k] = D + scale(bdt, L);
          } else {
            O.c[k] = scale(alpha, UA.c[k]) + (scale(beta, D) + scale(bdt, L));
          }
        }
      }
      Gp = Gn;
      // The stores are issued on every row and lane, without a branch: a lane
      // or row that owns nothing gets an offset past the row's extent, which
      // the buffer range check discards.  A branch around them would make the
      // wait for the next row's loads (issued before these stores) also wait
      // for the stores, since vector loads and stores share one in-order
      // counter and the two paths would be merged pessimistically.
      const bool row_ok = j >= y0 && j < y1;
      {
        T* d = a.out + (long long)jt * pitch;
        const unsigned soff = (own && row_ok) ? vboff : 0x80000000u;
        Lanes<T, CPL> o0, o1, o2, o3;
#pragma unroll
        for (int k = 0; k < CPL; ++k) {
          o0.v[k] = O.c[k].r; o1.v[k] = O.c[k].mx; o2.v[k] = O.c[k].my; o3.v[k] = O.c[k].e;
        }
        // a block may run past nx into the row padding, which is never read as data
        stv<T, CPL>(d, soff, rowb, o0);
        stv<T, CPL>(d + plane, soff, rowb, o1);
        stv<T, CPL>(d + 2 * plane, soff, rowb, o2);
        stv<T, CPL>(d + 3 * plane, soff, rowb, o3);
      }
      if (MODE != MODE_RESIDUAL && LAST && row_ok) {
#pragma unroll
        for (int k = 0; k < CPL; ++k) {
          if (own && x0 + k < nx) {
            bool ok;
            T rct = T(rxc[k] * eyc);
            T sp = cell_speed(P, rct, rct * eor, O.c[k], ok);
            smax = tmax(smax, sp);
            bad |= !ok;
          }
        }
      }
    };

    const int nrows = y1 - y0;
    if constexpr (SHORT) {
      row_step(js, R[0], R[1], R[2], R[3], Ur[0], Ur[URING - 1]);
      if (nrows > 1) row_step(js + DIR, R[1], R[2], R[3], R[0], Ur[1 % URING], Ur[0]);
      return;
    }
    for (int n = 0; n < nrows; n += RING) {
#pragma unroll
      for (int k = 0; k < RING; ++k)
        row_step(js + (n + k) * DIR, R[k % RING], R[(k + 1) % RING], R[(k + 2) % RING], R[(k + RING - 1) % RING],
                 Ur[k % URING], Ur[(k + URING - 1) % URING]);
    }
  };
  // rows read: y0-3 .. y1+2 (the ring runs one row past each end of the strip)
  const bool interior = fast && y0 >= 3 && y1 + 3 <= ny;
  if (!SHORT && (ty & 1)) {
    if (interior) sweep(std::integral_constant<int, -1>{}, std::true_type{});
    else sweep(std::integral_constant<int, -1>{}, std::false_type{});
  } else {
    if (interior) sweep(std::integral_constant<int, 1>{}, std::true_type{});
    else sweep(std::integral_constant<int, 1>{}, std::false_type{});
  }

  if (MODE != MODE_RESIDUAL && LAST) {
    if (bad) atomicOr(&a.ctrl->err, 1u);
    double sm = (double)smax;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) sm = fmax(sm, __shfl_xor(sm, off));
    if (lane == 0) atomicMax(&a.ctrl->cmax[q][slot].v, (unsigned long long)__double_as_longlong(sm));
  }
}

template <typename T, int RECON, int FLUX, int BC, int FORM, int MODE, int CPL, bool LAST, bool SHORT = false>
__global__ __launch_bounds__(256) void fv2d_stage_kernel(StageArgs<T> a) {
  const int lane = threadIdx.x & 63;
  // wave index made explicitly uniform so that strip, row and row pointers
  // live in scalar registers
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tile = xcd_block(blockIdx.x, gridDim.x) * 4 + wave;
  if (tile >= a.ntiles) return;
  stage_tile<T, RECON, FLUX, BC, FORM, MODE, CPL, LAST, SHORT>(a, tile, lane, blockIdx.x & 7);
}

// Persistent batched stage: every wave walks the global tile list of all
// instances (static stride, each XCD taking contiguous runs) and finds each
// tile's instance by binary search over the tile prefix sums.
template <typename T, int RECON, int FLUX, int BC, int FORM, int MODE, int CPL, bool LAST, bool SHORT = false>
__global__ __launch_bounds__(256) void fv2d_batch_stage_kernel(BatchArgs<T> b) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int stride = gridDim.x * 4;
  for (int t = xcd_block(blockIdx.x, gridDim.x) * 4 + wave; t < b.ntiles; t += stride) {
    int lo = 0, hi = b.ninst - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (b.tile_start[mid] <= t) lo = mid; else hi = mid - 1;
    }
    const InstDesc& d = b.inst[lo];
    StageArgs<T> a;
    a.in = b.in + d.off;
    a.un = b.un ? b.un + d.off : nullptr;
    a.out = b.out + d.off;
    a.rxf = b.tabx + d.tx_off;
    a.rxc = b.tabx + d.tx_off + d.nx + 1;
    a.eyc = b.taby + d.ty_off;
    a.eyf = b.taby + d.ty_off + d.ny;
    a.ctrl = b.ctrl + lo;
    a.plane = d.plane;
    a.pitch = d.pitch; a.nx = d.nx; a.ny = d.ny;
    a.rows = d.rows; a.ntx = d.ntx; a.ntiles = d.ntiles;
    a.parity = b.parity; a.first = b.first; a.last = b.last;
    a.t_end = b.t_end; a.h = d.h; a.cfl = d.cfl;
    a.gamma = d.gamma; a.g = d.g; a.p_over_rho = d.p_over_rho; a.inv_gm1 = d.inv_gm1;
    a.odx = d.odx; a.ody = d.ody;
    a.alpha = b.alpha; a.beta = b.beta;
    stage_tile<T, RECON, FLUX, BC, FORM, MODE, CPL, LAST, SHORT>(a, t - b.tile_start[lo], lane, blockIdx.x & 7);
  }
}

// ---- host-side launchers ----------------------------------------------------------

template <typename T, int RECON, int FLUX, int BC, int FORM, int MODE, int CPL, bool SHORT = false>
static hipError_t launch_stage_t(const StageArgs<T>& a, hipStream_t s) {
  int blocks = (a.ntiles + 3) / 4;
  if (MODE == MODE_STAGE && a.last)
    hipLaunchKernelGGL((fv2d_stage_kernel<T, RECON, FLUX, BC, FORM, MODE, CPL, true, SHORT>), dim3(blocks), dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((fv2d_stage_kernel<T, RECON, FLUX, BC, FORM, MODE, CPL, false, SHORT>), dim3(blocks), dim3(256), 0, s, a);
  return hipGetLastError();
}

template <typename T, int FORM, int MODE, int CPL, bool SHORT = false>
static hipError_t dispatch_scheme(const StageArgs<T>& a, int recon, int flux, int bc, hipStream_t s) {
#define FVWB_CASE(R, F, B)                                              \
  if (recon == R && flux == F && bc == B) return launch_stage_t<T, R, F, B, FORM, MODE, CPL, SHORT>(a, s);
  FVWB_CASE(0, 0, 0) FVWB_CASE(0, 0, 1) FVWB_CASE(0, 1, 0) FVWB_CASE(0, 1, 1)
  FVWB_CASE(1, 0, 0) FVWB_CASE(1, 0, 1) FVWB_CASE(1, 1, 0) FVWB_CASE(1, 1, 1)
#undef FVWB_CASE
  return hipErrorInvalidValue;
}

template <typename T, int RECON, int FLUX, int BC, int FORM, int MODE, int CPL, bool SHORT = false>
static hipError_t launch_batch_t(const BatchArgs<T>& b, int blocks, hipStream_t s) {
  if (MODE == MODE_STAGE && b.last)
    hipLaunchKernelGGL((fv2d_batch_stage_kernel<T, RECON, FLUX, BC, FORM, MODE, CPL, true, SHORT>), dim3(blocks), dim3(256), 0,
                       s, b);
  else
    hipLaunchKernelGGL((fv2d_batch_stage_kernel<T, RECON, FLUX, BC, FORM, MODE, CPL, false, SHORT>), dim3(blocks), dim3(256), 0,
                       s, b);
  return hipGetLastError();
}

template <typename T, int FORM, int MODE, int CPL, bool SHORT = false>
static hipError_t dispatch_batch(const BatchArgs<T>& b, int blocks, int recon, int flux, int bc, hipStream_t s) {
#define FVWB_CASE(R, F, B)                                              \
  if (recon == R && flux == F && bc == B) return launch_batch_t<T, R, F, B, FORM, MODE, CPL, SHORT>(b, blocks, s);
  FVWB_CASE(0, 0, 0) FVWB_CASE(0, 0, 1) FVWB_CASE(0, 1, 0) FVWB_CASE(0, 1, 1)
  FVWB_CASE(1, 0, 0) FVWB_CASE(1, 0, 1) FVWB_CASE(1, 1, 0) FVWB_CASE(1, 1, 1)
#undef FVWB_CASE
  return hipErrorInvalidValue;
}

}  // namespace fvwb
