// k_gemm_odd.hip -- the q4_0 GEMM for rows of an odd number of blocks, whose
// scales are not 4-byte aligned.  No matrix of the models has them, so there
// are fewer variants.
#include "gemm_variants.h"

namespace gemm {

VariantSet variants_f32_odd() {
  static Variant v[] = {
      GEMM_VARIANT(2, 2, 2, 2, 2, GEMM_F32, false), GEMM_VARIANT(2, 1, 2, 4, 2, GEMM_F32, false),
      GEMM_VARIANT(1, 1, 2, 4, 2, GEMM_F32, false),  GEMM_VARIANT(1, 1, 1, 8, 2, GEMM_F32, false),
  };
  return {v, (int)(sizeof(v) / sizeof(v[0]))};
}

VariantSet variants_glu_odd() {
  static Variant v[] = {
      GEMM_VARIANT(2, 2, 4, 2, 2, GEMM_GLU, false), GEMM_VARIANT(2, 2, 2, 2, 2, GEMM_GLU, false),
      GEMM_VARIANT(1, 2, 1, 4, 2, GEMM_GLU, false),
  };
  return {v, (int)(sizeof(v) / sizeof(v[0]))};
}

}  // namespace gemm
