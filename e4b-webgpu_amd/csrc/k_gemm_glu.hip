// k_gemm_glu.hip -- the q4_0 GEMM's GeGLU variants.
#include "gemm_variants.h"

namespace gemm {

// tokens x outputs of the tile, waves: 128 x 256, 8; 64 x 128, 8; 64 x 64, 8
// and 4; 32 x 32, 8 and 4
VariantSet variants_glu() {
  static Variant v[] = {
      GEMM_VARIANT(4, 2, 8, 1, 2, GEMM_GLU, true), GEMM_VARIANT(2, 2, 4, 2, 2, GEMM_GLU, true),
      GEMM_VARIANT(2, 2, 2, 4, 2, GEMM_GLU, true), GEMM_VARIANT(2, 2, 2, 2, 2, GEMM_GLU, true),
      GEMM_VARIANT(1, 2, 1, 4, 2, GEMM_GLU, true), GEMM_VARIANT(1, 2, 1, 8, 2, GEMM_GLU, true),
  };
  return {v, (int)(sizeof(v) / sizeof(v[0]))};
}

}  // namespace gemm
