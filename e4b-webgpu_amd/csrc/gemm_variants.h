// gemm_variants.h -- the q4_0 GEMM variants, by translation unit.
#pragma once
#include "gemm_kernel.h"

namespace gemm {
struct VariantSet {
  Variant* v;
  int n;
};
VariantSet variants_f32();      // rows of an even number of blocks
VariantSet variants_glu();
VariantSet variants_f32_odd();  // of an odd number
VariantSet variants_glu_odd();
}  // namespace gemm
