// The prefill GEMM of q|k|v with RoPE and the cache append in the epilogue (int4).
#include "eg_gemm_kernel.hpp"

namespace {

template <int ENC>
eg_gemm::KernelFn pick(int xm, const eg_gemm::Tile& t) {
  using namespace eg_gemm;
  if (xm == kXBf16) return pick_tile<ENC, 4, kXBf16, kRope>(t);
  if (xm == kXF32) return pick_tile<ENC, 4, kXF32, kRope>(t);
  return pick_tile<ENC, 4, kXNorm, kRope>(t);
}

}  // namespace

eg_gemm::KernelFn eg_gemm::pick_rope(int encoding, int xm, const Tile& t) {
  return encoding == EG_ENC_SIGNED ? pick<EG_ENC_SIGNED>(xm, t) : pick<EG_ENC_OFFSET_ZEROS>(xm, t);
}
