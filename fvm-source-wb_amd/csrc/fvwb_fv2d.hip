// fvwb_fv2d.hip — 2D finite-volume kernels (gfx950, wave64): the stage kernels of
// strips of four rows and more, of one problem and of batches, and the
// conversion, reduction and initial-state kernels.
#include "fvwb_fv2d_stage.h"

namespace fvwb {

// ---- auxiliary kernels ---------------------------------------------------------

// dU = u - conservative(w_eq) (benchmark_2d.f90:496-499), FP64, into planes of T.
template <typename T>
__global__ void aos_to_dev_kernel(const double* __restrict__ u, const double* __restrict__ w,
                                  T* __restrict__ out, int nx, int ny, int pitch, long long plane,
                                  double gamma) {
  long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= (long long)nx * ny) return;
  int i = (int)(c % nx), j = (int)(c / nx);
  const double* uc = u + 4 * c;
  const double* wc = w + 4 * c;
  double ue0 = wc[0], ue1 = wc[0] * wc[1], ue2 = wc[0] * wc[2];
  double ue3 = wc[3] / (gamma - 1.0) + 0.5 * (wc[0] * (wc[1] * wc[1] + wc[2] * wc[2]));
  long long o = (long long)j * pitch + i;
  out[o] = T(uc[0] - ue0);
  out[o + plane] = T(uc[1] - ue1);
  out[o + 2 * plane] = T(uc[2] - ue2);
  out[o + 3 * plane] = T(uc[3] - ue3);
}

// AoS(4,nx,ny) FP64 = [conservative(w_eq) +] planes (widened exactly).
template <typename T, bool ADD_EQ>
__global__ void dev_to_aos_kernel(const T* __restrict__ in, const double* __restrict__ w,
                                  double* __restrict__ u, int nx, int ny, int pitch, long long plane,
                                  double gamma) {
  long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= (long long)nx * ny) return;
  int i = (int)(c % nx), j = (int)(c / nx);
  long long o = (long long)j * pitch + i;
  double d0 = (double)in[o], d1 = (double)in[o + plane], d2 = (double)in[o + 2 * plane],
         d3 = (double)in[o + 3 * plane];
  if (ADD_EQ) {
    const double* wc = w + 4 * c;
    double ue0 = wc[0], ue1 = wc[0] * wc[1], ue2 = wc[0] * wc[2];
    double ue3 = wc[3] / (gamma - 1.0) + 0.5 * (wc[0] * (wc[1] * wc[1] + wc[2] * wc[2]));
    d0 += ue0; d1 += ue1; d2 += ue2; d3 += ue3;
  }
  double* uc = u + 4 * c;
  uc[0] = d0; uc[1] = d1; uc[2] = d2; uc[3] = d3;
}

// compute_max_speed (benchmark_2d.f90:264-279) over an AoS FP64 state.
__global__ void max_speed_aos_kernel(const double* __restrict__ u, long long n, double gamma,
                                     unsigned long long* __restrict__ out) {
  double m = 0.0;
  for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < n;
       c += (long long)gridDim.x * blockDim.x) {
    const double* s = u + 4 * c;
    double w0 = s[0], w1 = s[1] / w0, w2 = s[2] / w0;
    double w3 = (gamma - 1.0) * (s[3] - 0.5 * w0 * (w1 * w1 + w2 * w2));
    double cs = sqrt(gamma * fmax(w3, 1e-10) / fmax(w0, 1e-10));
    m = fmax(m, sqrt(w1 * w1 + w2 * w2) + cs);
  }
  for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off));
  if ((threadIdx.x & 63) == 0) atomicMax(out, (unsigned long long)__double_as_longlong(m));
}

// Initial reduction of max(|v|+c) of the stored state into ctrl->cmax[0].
template <typename T>
__global__ void cfl_init_kernel(const T* __restrict__ in, const double* __restrict__ rxc,
                                const double* __restrict__ eyc, Ctrl* ctrl, int nx, int ny,
                                int pitch, long long plane, double gamma, double p_over_rho,
                                double inv_gm1) {
  Phys<T> P;
  P.gamma = T(gamma); P.gm1 = T(gamma - 1.0); P.half = T(0.5); P.g = T(0);
  P.ggm1 = T(gamma * (gamma - 1.0)); P.gfloor = T(gamma * 1e-10);
  double m = 0.0;
  bool bad = false;
  for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < (long long)nx * ny;
       c += (long long)gridDim.x * blockDim.x) {
    int i = (int)(c % nx), j = (int)(c / nx);
    long long o = (long long)j * pitch + i;
    Vec4<T> d = {in[o], in[o + plane], in[o + 2 * plane], in[o + 3 * plane]};
    double rc = rxc[i] * eyc[j];
    bool ok;
    T sp = cell_speed(P, T(rc), T(rc * p_over_rho * inv_gm1), d, ok);
    m = fmax(m, (double)sp);
    bad |= !ok;
  }
  if (bad) atomicOr(&ctrl->err, 1u);
  for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off));
  if ((threadIdx.x & 63) == 0)
    atomicMax(&ctrl->cmax[0][blockIdx.x & 7].v, (unsigned long long)__double_as_longlong(m));
}

// Device-side initial condition: w_eq = closed-form equilibrium at centres
// (get_equilibrium_solution, benchmark_2d.f90:195-202) and dU = (0,0,0,dp/(gamma-1))
// with dp = amp*exp(-width*((x-x0)^2+(y-y0)^2)).
template <typename T>
__global__ void init_gaussian_kernel(T* __restrict__ out, double* __restrict__ w, int nx, int ny,
                                     int pitch, long long plane, double dx, double dy, double rho0,
                                     double p0, double kk, double gamma, double amp, double x0,
                                     double y0, double width) {
  long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= (long long)nx * ny) return;
  int i = (int)(c % nx), j = (int)(c / nx);
  double x = ((double)i + 0.5) * dx, y = ((double)j + 0.5) * dy;
  double e = exp(-(kk * (x + y)));
  double* wc = w + 4 * c;
  wc[0] = rho0 * e; wc[1] = 0.0; wc[2] = 0.0; wc[3] = p0 * e;
  double dp = amp * exp(-width * ((x - x0) * (x - x0) + (y - y0) * (y - y0)));
  long long o = (long long)j * pitch + i;
  out[o] = T(0); out[o + plane] = T(0); out[o + 2 * plane] = T(0);
  out[o + 3 * plane] = T(dp / (gamma - 1.0));
}

// ---- host-side launchers ----------------------------------------------------------

hipError_t launch_fv2d_batch_f64(const BatchArgs<double>& b, int blocks, int recon, int flux, int bc, int mode,
                                 hipStream_t s) {
  if (mode == MODE_STAGE1) return dispatch_batch<double, FORM_PLAIN, MODE_STAGE1, 2>(b, blocks, recon, flux, bc, s);
  if (mode == MODE_STAGE) return dispatch_batch<double, FORM_PLAIN, MODE_STAGE, 2>(b, blocks, recon, flux, bc, s);
  return hipErrorInvalidValue;
}

hipError_t launch_fv2d_batch_f32(const BatchArgs<float>& b, int blocks, int recon, int flux, int bc, int mode,
                                 int cpl, hipStream_t s) {
  if (cpl == 4) {
    if (mode == MODE_STAGE1) return dispatch_batch<float, FORM_DEV, MODE_STAGE1, 4>(b, blocks, recon, flux, bc, s);
    if (mode == MODE_STAGE) return dispatch_batch<float, FORM_DEV, MODE_STAGE, 4>(b, blocks, recon, flux, bc, s);
  } else if (cpl == 2) {
    if (mode == MODE_STAGE1) return dispatch_batch<float, FORM_DEV, MODE_STAGE1, 2>(b, blocks, recon, flux, bc, s);
    if (mode == MODE_STAGE) return dispatch_batch<float, FORM_DEV, MODE_STAGE, 2>(b, blocks, recon, flux, bc, s);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_fv2d_short_f64(const StageArgs<double>& a, int recon, int flux, int bc, int mode, hipStream_t s);
hipError_t launch_fv2d_short_f32(const StageArgs<float>& a, int recon, int flux, int bc, int mode, hipStream_t s);

// Stage modes: 0 residual (FP64 plain only), 1 first stage, 2 later stages.
// Strips of one or two rows go to the short form (fvwb_fv2d_short.hip).
// FP64 lanes own 2 columns (16-byte loads); FP32 lanes own `cpl` = 2 or 4.
hipError_t launch_fv2d_stage_f64(const StageArgs<double>& a, int recon, int flux, int bc, int mode,
                                 hipStream_t s) {
  if (a.rows <= 2) return launch_fv2d_short_f64(a, recon, flux, bc, mode, s);
  if (mode == MODE_RESIDUAL) return dispatch_scheme<double, FORM_PLAIN, MODE_RESIDUAL, 2>(a, recon, flux, bc, s);
  if (mode == MODE_STAGE1) return dispatch_scheme<double, FORM_PLAIN, MODE_STAGE1, 2>(a, recon, flux, bc, s);
  return dispatch_scheme<double, FORM_PLAIN, MODE_STAGE, 2>(a, recon, flux, bc, s);
}

hipError_t launch_fv2d_stage_f32(const StageArgs<float>& a, int recon, int flux, int bc, int mode, int cpl,
                                 hipStream_t s) {
  if (a.rows <= 2) return launch_fv2d_short_f32(a, recon, flux, bc, mode, s);
  if (cpl == 4) {
    if (mode == MODE_STAGE1) return dispatch_scheme<float, FORM_DEV, MODE_STAGE1, 4>(a, recon, flux, bc, s);
    if (mode == MODE_STAGE) return dispatch_scheme<float, FORM_DEV, MODE_STAGE, 4>(a, recon, flux, bc, s);
  } else if (cpl == 2) {
    if (mode == MODE_STAGE1) return dispatch_scheme<float, FORM_DEV, MODE_STAGE1, 2>(a, recon, flux, bc, s);
    if (mode == MODE_STAGE) return dispatch_scheme<float, FORM_DEV, MODE_STAGE, 2>(a, recon, flux, bc, s);
  }
  return hipErrorInvalidValue;
}

static inline unsigned grid1d(long long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

template <typename T>
hipError_t launch_aos_to_dev(const double* u, const double* w, T* out, int nx, int ny, int pitch,
                             long long plane, double gamma, hipStream_t s) {
  long long n = (long long)nx * ny;
  hipLaunchKernelGGL((aos_to_dev_kernel<T>), dim3(grid1d(n, 256)), dim3(256), 0, s, u, w, out, nx, ny,
                     pitch, plane, gamma);
  return hipGetLastError();
}
template hipError_t launch_aos_to_dev<double>(const double*, const double*, double*, int, int, int, long long, double, hipStream_t);
template hipError_t launch_aos_to_dev<float>(const double*, const double*, float*, int, int, int, long long, double, hipStream_t);

template <typename T>
hipError_t launch_dev_to_aos(const T* in, const double* w, double* u, int nx, int ny, int pitch,
                             long long plane, double gamma, bool add_eq, hipStream_t s) {
  long long n = (long long)nx * ny;
  if (add_eq)
    hipLaunchKernelGGL((dev_to_aos_kernel<T, true>), dim3(grid1d(n, 256)), dim3(256), 0, s, in, w, u, nx,
                       ny, pitch, plane, gamma);
  else
    hipLaunchKernelGGL((dev_to_aos_kernel<T, false>), dim3(grid1d(n, 256)), dim3(256), 0, s, in, w, u, nx,
                       ny, pitch, plane, gamma);
  return hipGetLastError();
}
template hipError_t launch_dev_to_aos<double>(const double*, const double*, double*, int, int, int, long long, double, bool, hipStream_t);
template hipError_t launch_dev_to_aos<float>(const float*, const double*, double*, int, int, int, long long, double, bool, hipStream_t);

hipError_t launch_max_speed_aos(const double* u, long long n, double gamma, unsigned long long* out,
                                hipStream_t s) {
  unsigned blocks = grid1d(n, 256);
  if (blocks > 2048) blocks = 2048;
  hipLaunchKernelGGL(max_speed_aos_kernel, dim3(blocks), dim3(256), 0, s, u, n, gamma, out);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_cfl_init(const T* in, const double* rxc, const double* eyc, Ctrl* ctrl, int nx, int ny,
                           int pitch, long long plane, double gamma, double p_over_rho, double inv_gm1,
                           hipStream_t s) {
  unsigned blocks = grid1d((long long)nx * ny, 256);
  if (blocks > 2048) blocks = 2048;
  hipLaunchKernelGGL((cfl_init_kernel<T>), dim3(blocks), dim3(256), 0, s, in, rxc, eyc, ctrl, nx, ny, pitch,
                     plane, gamma, p_over_rho, inv_gm1);
  return hipGetLastError();
}
template hipError_t launch_cfl_init<double>(const double*, const double*, const double*, Ctrl*, int, int, int, long long, double, double, double, hipStream_t);
template hipError_t launch_cfl_init<float>(const float*, const double*, const double*, Ctrl*, int, int, int, long long, double, double, double, hipStream_t);

template <typename T>
hipError_t launch_init_gaussian(T* out, double* w, int nx, int ny, int pitch, long long plane, double dx,
                                double dy, double rho0, double p0, double kk, double gamma, double amp,
                                double x0, double y0, double width, hipStream_t s) {
  long long n = (long long)nx * ny;
  hipLaunchKernelGGL((init_gaussian_kernel<T>), dim3(grid1d(n, 256)), dim3(256), 0, s, out, w, nx, ny, pitch,
                     plane, dx, dy, rho0, p0, kk, gamma, amp, x0, y0, width);
  return hipGetLastError();
}
template hipError_t launch_init_gaussian<double>(double*, double*, int, int, int, long long, double, double, double, double, double, double, double, double, double, double, hipStream_t);
template hipError_t launch_init_gaussian<float>(float*, double*, int, int, int, long long, double, double, double, double, double, double, double, double, double, double, hipStream_t);

}  // namespace fvwb

namespace fvwb {

// Plain streaming copy (16 B per lane): the calibration point for
// the achieved-bandwidth and HBM-counter figures of the solver kernels.
__global__ __launch_bounds__(256) void copy_probe_kernel(const float4* __restrict__ src, float4* __restrict__ dst,
                                                         long long n4) {
  // one float4 per thread over a grid that covers the buffer: the fastest plain
  // device copy pattern on MI355X (measured against grid-stride variants)
  const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n4) dst[k] = src[k];
}

hipError_t launch_copy_probe(const void* src, void* dst, long long bytes, hipStream_t s) {
  const long long n4 = bytes / 16;
  const long long blocks = (n4 + 255) / 256;
  if (blocks < 1 || blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL(copy_probe_kernel, dim3((unsigned)blocks), dim3(256), 0, s, (const float4*)src, (float4*)dst, n4);
  return hipGetLastError();
}

}  // namespace fvwb
