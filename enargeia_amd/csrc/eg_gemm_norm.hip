// The prefill GEMM over f32 rows of x, RMS-normalised on the way in, outputs stored with bias and residual.
#include "eg_gemm_kernel.hpp"

eg_gemm::KernelFn eg_gemm::pick_store_norm(int encoding, int bits, const Tile& t) {
  if (bits == 8) return encoding == EG_ENC_SIGNED ? pick_tile<EG_ENC_SIGNED, 8, kXNorm, kStore>(t)
                                                  : pick_tile<EG_ENC_OFFSET_ZEROS, 8, kXNorm, kStore>(t);
  return encoding == EG_ENC_SIGNED ? pick_tile<EG_ENC_SIGNED, 4, kXNorm, kStore>(t)
                                   : pick_tile<EG_ENC_OFFSET_ZEROS, 4, kXNorm, kStore>(t);
}
