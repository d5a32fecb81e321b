// The prefill GEMM over f32 rows of x, outputs stored with bias and residual.
#include "eg_gemm_kernel.hpp"

eg_gemm::KernelFn eg_gemm::pick_store_f32(int encoding, int bits, const Tile& t) {
  if (bits == 8) return encoding == EG_ENC_SIGNED ? pick_tile<EG_ENC_SIGNED, 8, kXF32, kStore>(t)
                                                  : pick_tile<EG_ENC_OFFSET_ZEROS, 8, kXF32, kStore>(t);
  return encoding == EG_ENC_SIGNED ? pick_tile<EG_ENC_SIGNED, 4, kXF32, kStore>(t)
                                   : pick_tile<EG_ENC_OFFSET_ZEROS, 4, kXF32, kStore>(t);
}
