// k_gemm_grp.hip -- the q4_0 GEMM's grouped variants (the expert-indexed MoE
// prefill): row tiles of up to 64 draws of one expert.
#include "gemm_variants.h"

namespace gemm {

// 64 draws x 64 outputs (GeGLU) or 128 columns (f32), 4 waves.  The GeGLU's
// rows are the hidden size, a multiple of 256; the down projection's, the
// expert FFN, may hold an odd number of blocks.
VariantSet variants_grp(bool glu, bool aligned) {
  static const Variant v[] = {
      GEMM_VARIANT(2, 2, 2, 2, 2, GEMM_F32, true, false, 170),
      GEMM_VARIANT(2, 2, 2, 2, 2, GEMM_F32, true, true, 170),
      GEMM_VARIANT(2, 2, 2, 2, 2, GEMM_GLU, true, true, 170),
  };
  if (glu) return {v + 2, aligned ? 1 : 0};
  return {v + (aligned ? 1 : 0), 1};
}

}  // namespace gemm
