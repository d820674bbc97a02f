// What the two forms of the mask MLP forward share (mask_mlp.hip, mask_estimator.hip).
#pragma once

#include "common.h"

namespace pmsst {

// Mask application in the epilogue (stem s of S): est[b, s, c, f, t] = spec[b, f C + c, t] x the
// complex mask (out[m, 2 r], out[m, 2 r + 1]) of row m = b T + t, complex row r = f C + c, in the
// iSTFT layout [B * S * C, Fbins, T] (complex64); bin 0 zero when zero_dc.  The mask values are
// rounded to the storage dtype first, as the stored mask the stock product multiplies is.
struct MlpApply {
  const float2* spec;  // complex64 [B, Fbins * C, T]
  float2* est;         // complex64 [B * S * C, Fbins, T]; null: the mask itself is stored
  FastDiv frames;      // T
  int C, Fbins, S, s, zero_dc;
};

// One complex mask value (re, im), rounded to the storage dtype, times the spectrum value sv of row
// r and frame t of batch item b, into its place of the estimate.
template <typename T>
__device__ __forceinline__ void store_masked(const MlpApply& ap, uint32_t b, uint32_t t, int r, float2 sv, float re,
                                             float im) {
  const int f = r / ap.C, c = r - f * ap.C;
  const float mr = to_f32(from_f32<T>(re)), mi = to_f32(from_f32<T>(im));
  // explicit fused multiply-adds: every kernel rounds the product the same way
  float2 e = make_float2(fmaf(sv.x, mr, -(sv.y * mi)), fmaf(sv.x, mi, sv.y * mr));
  if (ap.zero_dc && f == 0) e = make_float2(0.f, 0.f);
  ap.est[((static_cast<int64_t>(b) * ap.S + ap.s) * ap.C + c) * static_cast<int64_t>(ap.Fbins) * ap.frames.d +
         static_cast<int64_t>(f) * ap.frames.d + t] = e;
}

// Whether launch_mask_final takes this shape (16-bit, band widths in whole fours, 16-byte aligned x and
// weight, 8-byte aligned bias, pre and out).
bool mask_final_supported(const int64_t* dim_inputs, int64_t band_count, int64_t H);

// The final layer and the GLU of the mask MLP from the stored hidden layer x[M, NB, H] (me_fwd_dma_kernel):
// pre, and out or, with ap.est, the masked spectrum.
template <typename T>
int launch_mask_final(const void* x, const void* weight, const void* bias, const int64_t* offsets,
                      const int64_t* dim_inputs, int64_t band_count, int64_t M, int64_t H, void* pre, void* out,
                      const MlpApply& ap, hipStream_t stream);

}  // namespace pmsst
