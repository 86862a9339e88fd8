// fvwb_fv2d_short.hip — the 2D stage on strips of one or two rows, two columns
// per lane (small grids; see SHORT in fvwb_fv2d_stage.h).
#include "fvwb_fv2d_stage.h"

namespace fvwb {

hipError_t launch_fv2d_short_f64(const StageArgs<double>& a, int recon, int flux, int bc, int mode, hipStream_t s) {
  if (mode == MODE_RESIDUAL) return dispatch_scheme<double, FORM_PLAIN, MODE_RESIDUAL, 2, true>(a, recon, flux, bc, s);
  if (mode == MODE_STAGE1) return dispatch_scheme<double, FORM_PLAIN, MODE_STAGE1, 2, true>(a, recon, flux, bc, s);
  return dispatch_scheme<double, FORM_PLAIN, MODE_STAGE, 2, true>(a, recon, flux, bc, s);
}

hipError_t launch_fv2d_short_f32(const StageArgs<float>& a, int recon, int flux, int bc, int mode, hipStream_t s) {
  if (mode == MODE_STAGE1) return dispatch_scheme<float, FORM_DEV, MODE_STAGE1, 2, true>(a, recon, flux, bc, s);
  if (mode == MODE_STAGE) return dispatch_scheme<float, FORM_DEV, MODE_STAGE, 2, true>(a, recon, flux, bc, s);
  return hipErrorInvalidValue;
}

hipError_t launch_fv2d_batch_short_f64(const BatchArgs<double>& b, int blocks, int recon, int flux, int bc, int mode,
                                       hipStream_t s) {
  if (mode == MODE_STAGE1) return dispatch_batch<double, FORM_PLAIN, MODE_STAGE1, 2, true>(b, blocks, recon, flux, bc, s);
  if (mode == MODE_STAGE) return dispatch_batch<double, FORM_PLAIN, MODE_STAGE, 2, true>(b, blocks, recon, flux, bc, s);
  return hipErrorInvalidValue;
}

hipError_t launch_fv2d_batch_short_f32(const BatchArgs<float>& b, int blocks, int recon, int flux, int bc, int mode,
                                       hipStream_t s) {
  if (mode == MODE_STAGE1) return dispatch_batch<float, FORM_DEV, MODE_STAGE1, 2, true>(b, blocks, recon, flux, bc, s);
  if (mode == MODE_STAGE) return dispatch_batch<float, FORM_DEV, MODE_STAGE, 2, true>(b, blocks, recon, flux, bc, s);
  return hipErrorInvalidValue;
}

}  // namespace fvwb
