// fvwb_rd.hip — the reference's 2D residual distribution (benchmark_rd.f90,
// solver 'RD1') on MI355X.
//
// compute_update_rd (:612-745) scatters four corner residuals of every quad
// cell into its nodes.  Here a wave marches up a strip of node columns, forms
// each node's quantities once, each cell's corner residuals once, and every
// node adds its own four in the order the reference's cell loop (x outer, y
// inner) adds them, so the sums round identically without atomics.  The
// reference's boundary copies (:722-737) are stores of the node they copy.
// FP64 with contraction off and the reference's expression order throughout:
// the results equal the oracle's bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <string>

#include "../../include/fvwb.h"
#include "fvwb_checkpoint.h"
#include "fvwb_device.h"
#include "fvwb_transfer.h"

#pragma clang fp contract(off)

namespace rd {

using fvwb::lane_from_left;
using fvwb::lane_from_right;

struct Geo {
  int nx, ny, bc;
  double gamma, dx, dy;
};

__device__ __forceinline__ void primitive(double gamma, const double u[4], double w[4]) {
  w[0] = u[0];
  w[1] = u[1] / u[0];
  w[2] = u[2] / u[0];
  w[3] = (gamma - 1.0) * (u[3] - 0.5 * w[0] * (w[1] * w[1] + w[2] * w[2]));
}

// compute_speed (:478-493) of the vector it is handed
__device__ __forceinline__ double speed(double gamma, const double u[4]) {
  double w[4];
  primitive(gamma, u, w);
  const double cs = sqrt(gamma * fmax(w[3], 1e-10) / fmax(w[0], 1e-10));
  return sqrt(w[1] * w[1] + w[2] * w[2]) + cs;
}

__device__ __forceinline__ void load4(const double* a, int nx, int i, int j, double v[4]) {
  const double4 q = *reinterpret_cast<const double4*>(a + 4 * ((long long)j * nx + i));
  v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
}
__device__ __forceinline__ void store4(double* a, int nx, int i, int j, const double v[4]) {
  *reinterpret_cast<double4*>(a + 4 * ((long long)j * nx + i)) = double4{v[0], v[1], v[2], v[3]};
}

// The resident time loop's clock, on the device so that steps follow each
// other without a host round trip: dt of the current step, whether it runs
// (t < t_end and no failure), and the running totals.
struct Clock {
  double t, dt, dt_last;
  long long steps;
  int active, err;
};

// The node that the boundary copies make node `t` of 0..n-1 equal to, along x
// (:722-729: the lower end first) and along y (:730-737: the upper end first).
__host__ __device__ __forceinline__ int source_x(int bc, int n, int t) {
  if (bc == FVWB_RD_BC_PERIODIC) return t == 0 ? n - 1 : t;
  if (t == n - 1 && n > 2) return n - 2;
  return t == 0 || n == 2 ? 1 : t;
}
__host__ __device__ __forceinline__ int source_y(int bc, int n, int t) {
  if (bc == FVWB_RD_BC_PERIODIC) return t == n - 1 ? 0 : t;
  if (t == 0 && n > 2) return 1;
  return t == n - 1 || n == 2 ? n - 2 : t;
}

// What a cell needs of one of its nodes.
struct Node {
  double u[4], f[4], g[4];   // state, flux along x and along y
  double s3, sp;             // energy source (the momentum ones are -u[0]), speed
  double d[4];               // correction
};

__device__ __forceinline__ void node_values(double gamma, Node& n) {
  // compute_flux (:549-571): f along x, g along y
  double w[4], w2[4];
  primitive(gamma, n.u, w);
  n.g[0] = w[0] * w[2];
  n.g[1] = w[0] * w[1] * w[2];
  n.g[2] = w[2] * n.u[2] + w[3];
  n.g[3] = w[2] * n.u[3] + w[2] * w[3];
  n.f[0] = w[0] * w[1];
  n.f[1] = w[1] * n.u[1] + w[3];
  n.f[2] = w[0] * w[1] * w[2];
  n.f[3] = w[1] * n.u[3] + w[1] * w[3];
  // get_source (:747-767), grad_p = (1, 1): it receives the primitive vector
  // (:681-684) and converts it once more (:756), so its velocities are
  // w[1]/w[0] and w[2]/w[0]; compute_speed gets the primitive vector as well
  // (:692-695)
  primitive(gamma, w, w2);
  n.s3 = -w2[0] * (w2[1] * 1.0 + w2[2] * 1.0);
  const double cs = sqrt(gamma * fmax(w2[3], 1e-10) / fmax(w2[0], 1e-10));
  n.sp = sqrt(w2[1] * w2[1] + w2[2] * w2[2]) + cs;
}

// UPDATE: dudt of (u, diff), the drop-in.  FIRST and SECOND are the two passes
// of an 'RD1' step (evolve, :351-356) with their element-wise ends: FIRST has
// diff = 0 and leaves up = u - dudt/(dx dy); SECOND has diff = up - u, leaves
// the new u = up - dudt/(dx dy) and reduces its maximum speed.
enum { UPDATE = 0, FIRST = 1, SECOND = 2 };

constexpr int OWN = 62;                         // node columns a wave owns
constexpr int SLOTS = 64, SLOT_STRIDE = 16;     // 16 x 8 B = one 128-byte line

// A wave owns 62 node columns (lanes 1..62; lane l holds column x0 - 1 + l) and
// `rows` node rows, and marches up them.  A lane forms the quantities of its
// node of a row once, takes the node's on its right from the next lane (DPP),
// and with the row below has everything of its cell (a, r-1); what a cell adds
// to its right-hand nodes goes one lane on.  Each node's divisions and square
// roots are so evaluated once (and once more in a strip's two halo rows and
// columns), where a thread per cell evaluates them four times, and no value
// goes through LDS.  At 2049^2 the two updates with their element-wise passes,
// copies and speed pass took 570 us per step as separate kernels with a thread
// per cell; see the launch rule in strip_rows() for what they take now.
// PACKED: a grid of up to 30 columns leaves most lanes without a node, so the
// wave holds several strips of rows side by side, in groups of 1 << lw >= nx + 2
// lanes; the end lanes of a group own no cell and take nothing from the next.
template <int MODE, bool PACKED>
__global__ __launch_bounds__(256) void rd_sweep_kernel(Geo g, double area, const double* __restrict__ u0,
                                                       const double* __restrict__ u1, double* __restrict__ up,
                                                       const double* __restrict__ diff, double dt, int rows, int lw,
                                                       const Clock* __restrict__ ck, double* __restrict__ o0,
                                                       double* __restrict__ o1,
                                                       unsigned long long* __restrict__ smax) {
  const double* u = u0;
  double* out = o0;
  if constexpr (MODE != UPDATE) {
    if (!ck->active) return;
    dt = ck->dt;
    // the state alternates between two buffers, by the parity of the steps taken
    const bool odd = ck->steps & 1;
    u = odd ? u1 : u0;
    out = MODE == FIRST ? up : (odd ? o0 : o1);
  }
  const int wave = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = PACKED ? threadIdx.x & ((1 << lw) - 1) : threadIdx.x & 63;
  const int strips = PACKED ? 1 : (g.nx + OWN - 1) / OWN;
  const int tile = PACKED ? (wave << (6 - lw)) + ((threadIdx.x & 63) >> lw) : wave;
  if ((PACKED ? (wave << (6 - lw)) * rows : tile / strips * rows) >= g.ny) return;
  const int b0 = tile / strips * rows;                   // of PACKED's last groups perhaps past the grid
  const int b1 = min(b0 + rows, g.ny);
  const int a = tile % strips * OWN - 1 + lane;          // this lane's node column
  const int ac = min(max(a, 0), g.nx - 1);
  const bool cell_x = a >= 0 && a < g.nx - 1;            // cell (a, .) exists
  const bool own = lane >= 1 && (PACKED || lane <= OWN) && a < g.nx;
  // a strip that touches no end of the grid has no copies to make
  const bool inner = !PACKED && b0 > 1 && b1 < g.ny - 1 && tile % strips > 0 && tile % strips * OWN + OWN < g.nx - 1;
  const double dx = g.dx, dy = g.dy;

  auto load = [&](int r, Node& n) {
    const int rc = min(max(r, 0), g.ny - 1);
    load4(u, g.nx, ac, rc, n.u);
    if constexpr (MODE == UPDATE) load4(diff, g.nx, ac, rc, n.d);
    if constexpr (MODE == SECOND) load4(up, g.nx, ac, rc, n.d);     // up itself until node() takes u off
  };
  auto node = [&](Node& n) {
    node_values(g.gamma, n);
  };
  auto right4 = [&](const double v[4], double r[4]) {
#pragma unroll
    for (int k = 0; k < 4; ++k) r[k] = lane_from_right(v[k]);
  };
  // u - dudt/area of one node (or dudt itself) to node (ta, tb); base is the
  // value that dudt is taken off
  double speed_max = 0.0;
  auto put = [&](int ta, int tb, const double s[4], const double base[4]) {
    if constexpr (MODE == UPDATE) {
      store4(out, g.nx, ta, tb, s);
    } else {
      double x[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) x[v] = base[v] - s[v] / area;
      store4(out, g.nx, ta, tb, x);
      if constexpr (MODE == SECOND) speed_max = fmax(speed_max, speed(g.gamma, x));
    }
  };

  Node P, next;            // the row below, and the row in flight
  double pr_u[4], pr_d[4], pr_s3, pr_sp;   // the row below: its right neighbour
  double gsum[4];          // g of the row below plus its right neighbour's
  double c2[4] = {0.0, 0.0, 0.0, 0.0}, c3[4] = {0.0, 0.0, 0.0, 0.0};   // corners of cell (a, r-2) at row r-1
  double base[4];          // what dudt of row r-1 is taken off
  load(b0 - 1, P);
  load(b0, next);
  auto settle = [&](Node& n, double b[4]) {
    if constexpr (MODE == SECOND) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        b[v] = n.d[v];
        n.d[v] = n.d[v] - n.u[v];
      }
    } else {
#pragma unroll
      for (int v = 0; v < 4; ++v) b[v] = n.u[v];
    }
  };
  settle(P, base);
  node(P);
  right4(P.u, pr_u);
  if constexpr (MODE != FIRST) right4(P.d, pr_d);
  pr_s3 = lane_from_right(P.s3);
  pr_sp = lane_from_right(P.sp);
#pragma unroll
  for (int v = 0; v < 4; ++v) gsum[v] = P.g[v] + lane_from_right(P.g[v]);

  // r: the row that closes cell row r-1 and completes node row r-1; every group
  // of PACKED goes through as many rows
  const int last = PACKED ? b0 + rows : b1;
  for (int r = b0; r <= last; ++r) {
    Node N = next;
    load(r + 1, next);
    double nbase[4];
    settle(N, nbase);
    node(N);
    double nr_u[4], nr_d[4], gs[4];
    right4(N.u, nr_u);
    if constexpr (MODE != FIRST) right4(N.d, nr_d);
    const double nr_s3 = lane_from_right(N.s3), nr_sp = lane_from_right(N.sp);
    const bool cell = cell_x && r >= 1 && r < g.ny;      // cell (a, r-1) exists
    double alpha = P.sp;
    if (pr_sp > alpha) alpha = pr_sp;
    if (N.sp > alpha) alpha = N.sp;
    if (nr_sp > alpha) alpha = nr_sp;
    double q[4], k0[4], k2[4], k3[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      // :673-678, corners 11, 12, 21, 22 = P, its right neighbour, N, its right neighbour
      gs[v] = N.g[v] + lane_from_right(N.g[v]);
      const double fa = P.f[v] + N.f[v];
      const double fb = lane_from_right(fa);
      const double src = v == 0 ? 0.0
                         : v == 3 ? P.s3 + N.s3 + pr_s3 + nr_s3
                                  : -P.u[0] + -N.u[0] + -pr_u[0] + -nr_u[0];
      const double totalphi = -0.5 * fa + 0.5 * fb - 0.5 * gs[v] + 0.5 * gsum[v] - 0.25 * src * dx * dy;
      const double ubar = 0.25 * (P.u[v] + nr_u[v] + N.u[v] + pr_u[v]);
      // :688-697
      double k1;
      if constexpr (MODE == FIRST) {
        // diff = 0: its term is +0, which changes no sum that starts from +0
        k0[v] = dt * (totalphi * 0.25 + alpha * (P.u[v] - ubar) * dy);
        k1 = dt * (totalphi * 0.25 + alpha * (pr_u[v] - ubar) * dy);
        k2[v] = dt * (totalphi * 0.25 + alpha * (N.u[v] - ubar) * dx);
        k3[v] = dt * (totalphi * 0.25 + alpha * (nr_u[v] - ubar) * dx);
      } else {
        k0[v] = dy * dx * P.d[v] * 0.25 + dt * (totalphi * 0.25 + alpha * (P.u[v] - ubar) * dy);
        k1 = dy * dx * pr_d[v] * 0.25 + dt * (totalphi * 0.25 + alpha * (pr_u[v] - ubar) * dy);
        k2[v] = dy * dx * N.d[v] * 0.25 + dt * (totalphi * 0.25 + alpha * (N.u[v] - ubar) * dx);
        k3[v] = dy * dx * nr_d[v] * 0.25 + dt * (totalphi * 0.25 + alpha * (nr_u[v] - ubar) * dx);
      }
      if (!cell) k0[v] = k1 = k2[v] = k3[v] = 0.0;
      // what cell column a adds to node (a+1, r-1): cells (a, r-2) and (a, r-1)
      q[v] = 0.0 + c3[v] + k1;
    }
    // node (a, r-1): cells (a-1, r-2), (a-1, r-1), (a, r-2), (a, r-1) in that
    // order; a cell that does not exist counts as +0, which changes nothing
    double s[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      s[v] = lane_from_left(q[v]) + c2[v] + k0[v];
      c2[v] = k2[v];
      c3[v] = k3[v];
    }
    const int b = r - 1;
    if (b >= b0 && own && (!PACKED || b < b1)) {
      if (inner) {
        put(a, b, s, base);
      } else {
        // every node whose value the copies take from this one: itself, and
        // nodes of the four edges
        const int xs[3] = {a, 0, g.nx - 1}, ys[3] = {b, 0, g.ny - 1};
        for (int p = 0; p < 3; ++p) {
          if (source_x(g.bc, g.nx, xs[p]) != a || (p > 0 && xs[p] == a) || (p == 2 && g.nx == 1)) continue;
          for (int w = 0; w < 3; ++w) {
            if (source_y(g.bc, g.ny, ys[w]) != b || (w > 0 && ys[w] == b)) continue;
            if (MODE == UPDATE || (p == 0 && w == 0)) {
              put(xs[p], ys[w], s, base);
            } else {
              double tb[4];
              load4(MODE == FIRST ? u : up, g.nx, xs[p], ys[w], tb);
              put(xs[p], ys[w], s, tb);
            }
          }
        }
      }
    }
    P = N;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      pr_u[v] = nr_u[v];
      if constexpr (MODE != FIRST) pr_d[v] = nr_d[v];
      gsum[v] = gs[v];
      base[v] = nbase[v];
    }
    pr_s3 = nr_s3;
    pr_sp = nr_sp;
  }
  if constexpr (MODE == SECOND) {
    for (int off = 32; off > 0; off >>= 1) speed_max = fmax(speed_max, __shfl_xor(speed_max, off));
    if ((threadIdx.x & 63) == 0)
      atomicMax(smax + (blockIdx.x % SLOTS) * SLOT_STRIDE, (unsigned long long)__double_as_longlong(speed_max));
  }
}

// compute_max_speed (:448-475): the maximum of the nodes' speeds (a NaN speed
// never passes the reference's ">=" test, and fmax ignores it likewise).
// Speeds are >= 0, so their bit patterns order as unsigned integers.  Each
// workgroup reduces its nodes and adds one atomicMax to one of SLOTS slots, a
// cache line apart, so the atomics do not queue on one line; the host takes
// the maximum of the slots.
__global__ __launch_bounds__(256) void rd_speed_kernel(Geo g, const double* __restrict__ u,
                                                       unsigned long long* __restrict__ smax) {
  __shared__ double part[4];
  const long long n = (long long)g.nx * g.ny;
  double m = 0.0;
  for (long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (long long)gridDim.x * blockDim.x) {
    double v[4];
    const double4 q = *reinterpret_cast<const double4*>(u + 4 * k);
    v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
    m = fmax(m, speed(g.gamma, v));
  }
  for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off));
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    m = fmax(fmax(part[0], part[1]), fmax(part[2], part[3]));
    atomicMax(smax + (blockIdx.x % SLOTS) * SLOT_STRIDE, (unsigned long long)__double_as_longlong(m));
  }
}

// t = t + dt (:366), after a step that ran
__device__ __forceinline__ void tick(Clock* ck) {
  if (!ck->active) return;
  ck->t = ck->t + ck->dt;
  ck->dt_last = ck->dt;
  ck->steps += 1;
}
// dt = min(cfl dx dy/cmax/3, t_end - t) (evolve, :348-349) from the speed
// slots, which it clears for the next step; a maximum that is not finite and
// positive stops the run with the error flag set.  One wave, a slot per lane;
// `ticks` closes the step before this one first.
__global__ __launch_bounds__(64) void rd_dt_kernel(Geo g, double cfl, double t_end, int ticks,
                                                   unsigned long long* __restrict__ smax, Clock* __restrict__ ck) {
  static_assert(SLOTS == 64, "a slot per lane");
  const int k = threadIdx.x * SLOT_STRIDE;
  double cmax = __longlong_as_double((long long)smax[k]);
  smax[k] = 0;
  for (int off = 32; off > 0; off >>= 1) cmax = fmax(cmax, __shfl_xor(cmax, off));
  if (threadIdx.x != 0) return;
  if (ticks) tick(ck);
  if (ck->err || !(ck->t < t_end)) {
    ck->active = 0;
    return;
  }
  if (!(cmax > 0.0) || !isfinite(cmax)) {
    ck->err = 1;
    ck->active = 0;
    return;
  }
  ck->dt = fmin(cfl * g.dy * g.dx / cmax / (2.0 * 1.0 + 1.0), t_end - ck->t);
  ck->active = 1;
}
__global__ void rd_tick_kernel(Clock* __restrict__ ck) {
  if (threadIdx.x == 0) tick(ck);
}

}  // namespace rd

using namespace rd;

struct fvwb_rd {
  fvwb_rd_params p{};
  Geo g{};
  fvwb_xfer::Staging xfer;  // large copies from and to host arrays
  hipStream_t stream = nullptr;
  double* buf[2] = {nullptr, nullptr};   // state, AoS(4,nx,ny): buf[par], the other one is the next step's
  int par = 0;                           // parity of the clock's step count
  double* d_up = nullptr;
  double* d_dudt = nullptr;
  unsigned long long* d_smax = nullptr;
  Clock* d_clk = nullptr;
  bool loaded = false;
  std::string err;
};

static thread_local std::string g_errrd;

static int failrd(fvwb_rd* h, int code, const std::string& msg) {
  (h ? h->err : g_errrd) = msg;
  return code;
}

#define HIPR(h, call)                                                                                  \
  do {                                                                                                 \
    hipError_t e_ = (call);                                                                            \
    if (e_ != hipSuccess) return failrd(h, FVWB_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

extern "C" const char* fvwb_rd_last_error(fvwb_rd_handle h) { return h ? h->err.c_str() : g_errrd.c_str(); }

extern "C" int fvwb_rd_destroy(fvwb_rd_handle h) {
  if (!h) return FVWB_OK;
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  void* ps[] = {h->buf[0], h->buf[1], h->d_up, h->d_dudt, h->d_smax, h->d_clk};
  for (void* q : ps)
    if (q) (void)hipFree(q);
  if (h->stream) (void)hipStreamDestroy(h->stream);
  delete h;
  return FVWB_OK;
}

extern "C" int fvwb_rd_create(fvwb_rd_handle* out, const fvwb_rd_params* p) {
  if (!out || !p) return failrd(nullptr, FVWB_ERR_ARG, "NULL argument");
  *out = nullptr;
  if (p->nx < 2 || p->ny < 2) return failrd(nullptr, FVWB_ERR_ARG, "nx and ny must be >= 2");
  if ((long long)p->nx * p->ny > (1ll << 28)) return failrd(nullptr, FVWB_ERR_ARG, "more than 2^28 nodes");
  // a limit of the interface, not of these launches: it has always been refused
  if (p->ny > 458745) return failrd(nullptr, FVWB_ERR_ARG, "ny must be <= 458745");
  if (p->bc != FVWB_RD_BC_PERIODIC && p->bc != FVWB_RD_BC_TRANSMISSIVE)
    return failrd(nullptr, FVWB_ERR_ARG, "bc must be 2 (periodic copies) or 3 (transmissive copies)");
  if (!(p->gamma > 1.0) || !(p->boxlen_x > 0.0) || !(p->boxlen_y > 0.0) || !(p->cfl > 0.0))
    return failrd(nullptr, FVWB_ERR_ARG, "gamma > 1 and positive box lengths and cfl required");
  fvwb_rd* h = new (std::nothrow) fvwb_rd;
  if (!h) return failrd(nullptr, FVWB_ERR_OOM, "host allocation failed");
  h->p = *p;
  h->g = Geo{p->nx, p->ny, p->bc, p->gamma, p->boxlen_x / (double)(p->nx - 1), p->boxlen_y / (double)(p->ny - 1)};
  const size_t nb = sizeof(double) * 4 * (size_t)p->nx * (size_t)p->ny;
  bool ok = hipStreamCreate(&h->stream) == hipSuccess && hipMalloc(&h->buf[0], nb) == hipSuccess &&
            hipMalloc(&h->buf[1], nb) == hipSuccess && hipMalloc(&h->d_up, nb) == hipSuccess &&
            hipMalloc(&h->d_dudt, nb) == hipSuccess &&
            hipMalloc(&h->d_smax, sizeof(unsigned long long) * SLOTS * SLOT_STRIDE) == hipSuccess &&
            hipMalloc(&h->d_clk, sizeof(Clock)) == hipSuccess;
  if (!ok) {
    fvwb_rd_destroy(h);
    return failrd(nullptr, FVWB_ERR_OOM, "device allocation failed");
  }
  *out = h;
  return FVWB_OK;
}

// Rows of a strip, of so many one-row strips: about 4096 strips (two rounds of the two waves per SIMD that
// SECOND runs at), between 2 and 12 rows each.  A strip marches 2 rows more than
// it owns, so short ones repeat work and long ones leave the chip idle on small
// grids.  Measured us per step with 2 / 4 / 8 / 12 / 16 / 24 rows: 129^2 18.8 /
// 24.6 / 37.3 / 49.9 / 62.7 / 87.3, 513^2 35.2 / 37.7 / 39.7 / 51.7 / 64.4 /
// 89.1, 1025^2 80.4 / 73.1 / 77.2 / 75.7 / 93.5 / 90.1, 2049^2 275 / 231 / 209 /
// 201 / 211 / 205.
static int strip_rows(long long strips) { return (int)std::max(2LL, std::min(12LL, strips / 4096)); }

// One sweep: dudt of (u0, diff) into o0, or a pass of an 'RD1' step between the
// state's two buffers.  Up to 30 columns the strips are packed into waves: 2 x
// 200,000 nodes take 62 us per step (502 with a wave per strip, 400 with a thread
// per cell), 16 x 100,000 172 (274 and 280), 30 x 1000 20 (21 and 36).
template <int MODE>
static int sweep(fvwb_rd* h, const double* u0, const double* u1, double* up, const double* diff, double dt,
                 const Clock* ck, double* o0, double* o1) {
  const long long nx = h->p.nx, ny = h->p.ny;
  int lw = 2;
  while (lw < 6 && (1 << lw) < nx + 2) ++lw;
  const bool packed = lw < 6;
  const long long across = (nx + OWN - 1) / OWN, groups = 64 >> lw;
  const int rows = strip_rows(packed ? ny / groups : across * ny);
  const long long strips = across * ((ny + rows - 1) / rows), waves = packed ? (strips + groups - 1) / groups : strips;
  hipLaunchKernelGGL((packed ? rd_sweep_kernel<MODE, true> : rd_sweep_kernel<MODE, false>),
                     dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, h->stream, h->g, h->g.dx * h->g.dy, u0, u1, up,
                     diff, dt, rows, lw, ck, o0, o1, h->d_smax);
  HIPR(h, hipGetLastError());
  return FVWB_OK;
}

static void launch_speed(fvwb_rd* h, const double* u) {
  const long long n = (long long)h->p.nx * h->p.ny;
  const unsigned blocks = (unsigned)std::min<long long>((n + 255) / 256, 16384);
  hipLaunchKernelGGL(rd_speed_kernel, dim3(blocks), dim3(256), 0, h->stream, h->g, u, h->d_smax);
}

static int max_speed(fvwb_rd* h, const double* u, double* cmax) {
  const size_t sb = sizeof(unsigned long long) * SLOTS * SLOT_STRIDE;
  HIPR(h, hipMemsetAsync(h->d_smax, 0, sb, h->stream));
  launch_speed(h, u);
  HIPR(h, hipGetLastError());
  unsigned long long bits[SLOTS * SLOT_STRIDE];
  HIPR(h, hipMemcpyAsync(bits, h->d_smax, sb, hipMemcpyDeviceToHost, h->stream));
  HIPR(h, hipStreamSynchronize(h->stream));
  unsigned long long m = 0;
  for (int k = 0; k < SLOTS; ++k) m = std::max(m, bits[k * SLOT_STRIDE]);
  std::memcpy(cmax, &m, sizeof m);
  return FVWB_OK;
}

extern "C" int fvwb_rd_compute_update(fvwb_rd_handle h, const double* u, const double* diff, double dt,
                                      double* dudt) {
  if (!h || !u || !diff || !dudt) return failrd(h, FVWB_ERR_ARG, "NULL argument");
  const size_t nb = sizeof(double) * 4 * (size_t)h->p.nx * (size_t)h->p.ny;
  // the update works in the step's scratch arrays; an uploaded state stays as it is
  HIPR(h, fvwb_xfer::to_device(h->xfer, h->d_up, u, nb, h->stream));
  double* d_diff = h->buf[h->par ^ 1];
  HIPR(h, fvwb_xfer::to_device(h->xfer, d_diff, diff, nb, h->stream));
  int rc = sweep<UPDATE>(h, h->d_up, nullptr, nullptr, d_diff, dt, nullptr, h->d_dudt, nullptr);
  if (rc) return rc;
  HIPR(h, fvwb_xfer::to_host(h->xfer, dudt, h->d_dudt, nb, h->stream));
  HIPR(h, hipStreamSynchronize(h->stream));
  return FVWB_OK;
}

extern "C" int fvwb_rd_compute_max_speed(fvwb_rd_handle h, const double* u, double* cmax) {
  if (!h || !u || !cmax) return failrd(h, FVWB_ERR_ARG, "NULL argument");
  const size_t nb = sizeof(double) * 4 * (size_t)h->p.nx * (size_t)h->p.ny;
  HIPR(h, fvwb_xfer::to_device(h->xfer, h->d_up, u, nb, h->stream));
  return max_speed(h, h->d_up, cmax);
}

extern "C" int fvwb_rd_upload(fvwb_rd_handle h, const double* u) {
  if (!h || !u) return failrd(h, FVWB_ERR_ARG, "NULL argument");
  const size_t nb = sizeof(double) * 4 * (size_t)h->p.nx * (size_t)h->p.ny;
  const Clock zero{};
  h->par = 0;
  HIPR(h, fvwb_xfer::to_device(h->xfer, h->buf[0], u, nb, h->stream));
  HIPR(h, hipMemcpyAsync(h->d_clk, &zero, sizeof zero, hipMemcpyHostToDevice, h->stream));
  HIPR(h, hipStreamSynchronize(h->stream));
  h->loaded = true;
  return FVWB_OK;
}

static int read_clock(fvwb_rd* h, Clock* c) {
  HIPR(h, hipMemcpyAsync(c, h->d_clk, sizeof *c, hipMemcpyDeviceToHost, h->stream));
  HIPR(h, hipStreamSynchronize(h->stream));
  h->par = (int)(c->steps & 1);
  return FVWB_OK;
}

// Steps are queued in groups of this many between reads of the clock.
static constexpr int32_t kGroup = 64;

// evolve (:356-385) with solver 'RD1': while t < t_end, at most nsteps steps.
// dt, t and the step count live on the device; the host reads them once per
// group of steps to stop early, and each kernel of a step past t_end (or
// after a failure) does nothing.
extern "C" int fvwb_rd_advance(fvwb_rd_handle h, int32_t nsteps, double t_end) {
  if (!h) return failrd(h, FVWB_ERR_ARG, "NULL handle");
  if (!h->loaded) return failrd(h, FVWB_ERR_STATE, "advance before upload");
  if (nsteps < 0) return failrd(h, FVWB_ERR_ARG, "nsteps must be >= 0");
  Clock c{};
  int rc = read_clock(h, &c);
  if (rc) return rc;
  // the state's maximum speed; every step leaves its new state's
  HIPR(h, hipMemsetAsync(h->d_smax, 0, sizeof(unsigned long long) * SLOTS * SLOT_STRIDE, h->stream));
  launch_speed(h, h->buf[h->par]);
  double *b0 = h->buf[0], *b1 = h->buf[1];
  int32_t done = 0;
  while (done < nsteps && !c.err && c.t < t_end) {
    const int32_t k = std::min(kGroup, nsteps - done);
    for (int32_t s = 0; s < k; ++s) {
      hipLaunchKernelGGL(rd_dt_kernel, dim3(1), dim3(64), 0, h->stream, h->g, h->p.cfl, t_end, s > 0 ? 1 : 0,
                         h->d_smax, h->d_clk);
      if ((rc = sweep<FIRST>(h, b0, b1, h->d_up, nullptr, 0.0, h->d_clk, nullptr, nullptr))) return rc;
      if ((rc = sweep<SECOND>(h, b0, b1, h->d_up, nullptr, 0.0, h->d_clk, b0, b1))) return rc;
    }
    hipLaunchKernelGGL(rd_tick_kernel, dim3(1), dim3(64), 0, h->stream, h->d_clk);
    HIPR(h, hipGetLastError());
    done += k;
    if ((rc = read_clock(h, &c))) return rc;
  }
  if (c.err) return failrd(h, FVWB_ERR_NONPHYSICAL, "wave-speed maximum not finite and positive");
  return FVWB_OK;
}

extern "C" int fvwb_rd_download(fvwb_rd_handle h, double* u) {
  if (!h || !u) return failrd(h, FVWB_ERR_ARG, "NULL argument");
  if (!h->loaded) return failrd(h, FVWB_ERR_STATE, "download before upload");
  const size_t nb = sizeof(double) * 4 * (size_t)h->p.nx * (size_t)h->p.ny;
  HIPR(h, fvwb_xfer::to_host(h->xfer, u, h->buf[h->par], nb, h->stream));
  HIPR(h, hipStreamSynchronize(h->stream));
  return FVWB_OK;
}

// ---- checkpoint / resume: the state and the clock -----------------------------------
extern "C" int fvwb_rd_checkpoint_save(fvwb_rd_handle h, const char* path) {
  if (!h || !path) return failrd(h, FVWB_ERR_ARG, "NULL argument");
  if (!h->loaded) return failrd(h, FVWB_ERR_STATE, "checkpoint before upload");
  const fvwb_ckpt::Segment seg[2] = {{h->buf[h->par], sizeof(double) * 4 * (size_t)h->p.nx * (size_t)h->p.ny},
                                     {h->d_clk, sizeof(Clock)}};
  std::string err;
  const int rc = fvwb_ckpt::save(path, fvwb_ckpt::RD, &h->p, sizeof h->p, 0, seg, 2, h->stream, err);
  if (rc) h->err = err;
  return rc;
}

extern "C" int fvwb_rd_checkpoint_load(fvwb_rd_handle h, const char* path) {
  if (!h || !path) return failrd(h, FVWB_ERR_ARG, "NULL argument");
  const fvwb_ckpt::Segment seg[2] = {{h->buf[0], sizeof(double) * 4 * (size_t)h->p.nx * (size_t)h->p.ny},
                                     {h->d_clk, sizeof(Clock)}};
  std::string err;
  int32_t parity = 0;
  const int rc = fvwb_ckpt::load(path, fvwb_ckpt::RD, &h->p, sizeof h->p, &parity, seg, 2, h->stream, err);
  h->loaded = rc == FVWB_OK;
  h->par = 0;
  if (rc) {
    h->err = err;
    return rc;
  }
  // the state lies in buf[0]; the clock's step count says which of the two it is
  Clock c{};
  const int rc2 = read_clock(h, &c);
  if (rc2) return rc2;
  if (h->par) std::swap(h->buf[0], h->buf[1]);
  return FVWB_OK;
}

extern "C" int fvwb_rd_get_time(fvwb_rd_handle h, double* t, double* dt_last, int64_t* steps) {
  if (!h) return failrd(h, FVWB_ERR_ARG, "NULL handle");
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
