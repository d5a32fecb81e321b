// The prefill GEMM over f32 rows of x, RMS-normalised on the way in, outputs stored with bias and residual
// (int4).
#include "eg_gemm_kernel.hpp"

eg_gemm::KernelFn eg_gemm::pick_store_norm(int encoding, const Tile& t) {
  return encoding == EG_ENC_SIGNED ? pick_tile<EG_ENC_SIGNED, 4, kXNorm, kStore>(t)
                                   : pick_tile<EG_ENC_OFFSET_ZEROS, 4, kXNorm, kStore>(t);
}
