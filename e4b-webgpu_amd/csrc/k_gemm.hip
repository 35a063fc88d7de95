// k_gemm.hip -- choice and launch of the q4_0 GEMM variants (gemm_kernel.h).
#include <limits.h>

#include <algorithm>

#include "../../include/e4b.h"
#include "gemm_variants.h"
#include "kernels.h"
#include "util.h"

namespace gemm {

// tokens x rows of the tile, waves: 128 x 256, 4; 64 x 128, 4; 64 x 64, 8
// and 4; 32 x 64, 8 and 4; 32 x 32, 8 (of twelve measured, the seven without
// which some shape lost most)
VariantSet variants_f32() {
  static Variant v[] = {
      GEMM_VARIANT(4, 2, 4, 1, 2, GEMM_F32, true), GEMM_VARIANT(2, 2, 2, 2, 2, GEMM_F32, true),
      GEMM_VARIANT(2, 1, 2, 4, 2, GEMM_F32, true), GEMM_VARIANT(2, 1, 2, 2, 2, GEMM_F32, true),
      GEMM_VARIANT(1, 1, 2, 4, 2, GEMM_F32, true), GEMM_VARIANT(1, 1, 2, 2, 2, GEMM_F32, true),
      GEMM_VARIANT(1, 1, 1, 8, 2, GEMM_F32, true),
  };
  return {v, (int)(sizeof(v) / sizeof(v[0]))};
}

}  // namespace gemm

namespace {

using gemm::Variant;
using gemm::VariantSet;

VariantSet variants(int epi, bool aligned) {
  using namespace gemm;
  if (epi == GEMM_GLU) return aligned ? variants_glu() : variants_glu_odd();
  return aligned ? variants_f32() : variants_f32_odd();
}

// Estimated microseconds of a launch: which tile is best depends on how the
// workgroups fill 256 CUs (a tile twice as large halves the operand traffic
// and the nibble conversion, and leaves half the workgroups), so the variants
// are compared by this model instead of by thresholds.  A stage of one
// workgroup takes at least its latency (copies, barrier, the waves' chain of
// dependent matrix instructions); the workgroups that share a CU add up their
// work: 32 x 32 x 32 units at 107 / 81 / 65 ns of a SIMD for 1 / 2 / 4 token
// tiles a wave (the nibble conversion is shared by them).  Constants fitted
// on MI355X to the times of all variants over 3000 shapes (37..32768 rows,
// 64..16384 columns, 1..512 tokens), weights in cache and cold.  Over 2000
// other shapes it is 12 and 14 % rms off, and the variant it picks is 0.4 %
// slower than the best on average, 30 % at worst.
// Eight K groups count as one workgroup a CU also where two fit (rows of an
// odd number of blocks): two side by side take as long as one after the other
// (1.23 against 0.61 us a stage).
double gemm_cost_us(const Variant& v, int resident, int epi, int64_t units, int nb, int64_t M, int ks) {
  const int occ = v.KW == 8 ? 1 : resident;
  const int waves = v.RW * v.KW, sb = v.KW * v.KBL;
  const int uc = epi == GEMM_GLU ? 32 * v.RW : 32 * v.RW * v.NT;
  const double wgs = (double)((units + uc - 1) / uc) * (double)((M + 32 * v.T - 1) / (32 * v.T)) * ks;
  const double stages = (double)((nb + ks * sb - 1) / (ks * sb));
  const double unit = (v.T == 1 ? 0.107 : v.T == 2 ? 0.081 : 0.065) / 4;
  const double lat = 0.373 + 0.047 * v.T * v.NT * v.KBL * std::max(1.0, waves / 4.0);
  const double thr = v.T * v.NT * v.RW * v.KW * v.KBL * unit;
  const double per = (double)(int64_t)((wgs + 255) / 256);  // workgroups of the fullest CU
  const double full = (double)(int64_t)(per / occ), rem = per - full * occ;
  double t = full * std::max(lat, thr * occ) + (rem > 0 ? std::max(lat, thr * rem) : 0.0);
  t = 1.7 + stages * t + 0.3 * v.T * v.NT * (v.KW == 1 ? 1 : 2) * (full + (rem > 0 ? 1 : 0));
  return t;
}

// Workgroups of a variant that share a CU, as its kernel was compiled (LDS and
// registers); the runtime is asked once a variant.  0 and an error message if
// it does not know the kernel.
int occupancy(Variant& v) {
  int occ = v.occ.load(std::memory_order_relaxed);
  if (occ > 0) return occ;
  const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, v.kernel, 64 * v.RW * v.KW, 0);
  if (e != hipSuccess || occ < 1) {
    (void)e4b_fail(E4B_EHIP, "q4_0 GEMM: occupancy of a kernel -> %s", hipGetErrorString(e));
    return 0;
  }
  v.occ.store(occ, std::memory_order_relaxed);
  return occ;
}

// the variant of the least estimated time (its estimate in *us), or null
const Variant* choose(const VariantSet& s, int epi, int64_t units, int nb, int64_t M, int ks, double* us) {
  const Variant* best = nullptr;
  double tb = 0;
  for (int i = 0; i < s.n; ++i) {
    const int occ = occupancy(s.v[i]);
    if (!occ) return nullptr;
    const double t = gemm_cost_us(s.v[i], occ, epi, units, nb, M, ks);
    if (!best || t < tb) {
      best = &s.v[i];
      tb = t;
    }
  }
  if (us) *us = tb;
  return best;
}

// q4_0 blocks of a split-K slice: whole pairs of blocks, and the slices of
// every variant's stage alike
constexpr int kSliceBlocks = 4;
int slice_blocks(int nb, int ks) { return ((nb + ks - 1) / ks + kSliceBlocks - 1) / kSliceBlocks * kSliceBlocks; }

}  // namespace

int q40_gemm_kslices(int nb, int want) {
  for (int ks = want < 1 ? 1 : want; ks > 1; --ks) {
    const int nbs = slice_blocks(nb, ks);
    if ((nb + nbs - 1) / nbs == ks) return ks;
  }
  return 1;
}

int q40_gemm_best_kslices(int64_t rows, int nb, int M, int most) {
  const VariantSet s = variants(GEMM_F32, nb % 2 == 0);
  int best = 1;
  double tb = 0;
  for (int want = 1; want <= most; want *= 2) {
    const int ks = q40_gemm_kslices(nb, want);
    double t = 0;
    if (!choose(s, GEMM_F32, rows, nb, M, ks, &t)) return 1;  // (the launch says why)
    // each further slice is written once and read once by the consumer, at
    // about 4 MB a microsecond
    t += (double)(ks - 1) * (double)M * (double)rows * 8.0 / 4e6;
    if (want == 1 || t < tb) {
      best = ks;
      tb = t;
    }
  }
  return best;
}

int launch_q40_gemm(const GemmArgs& a, hipStream_t st) {
  const Q40Mat& W = a.W;
  const int K = W.nb * 32;
  if (a.M < 1 || K < 32) return e4b_fail(E4B_EINVAL, "q4_0 GEMM: empty operand (M=%d K=%d)", a.M, K);
  if ((uint64_t)W.rows * (uint64_t)W.nb * 16u > 0xffffffffull)
    return e4b_fail(E4B_EINVAL, "q4_0 GEMM: a %lld x %d-block matrix exceeds the 4 GiB plane limit",
                    (long long)W.rows, W.nb);
  if (a.ldx < K || a.ldx % 8) return e4b_fail(E4B_EINVAL, "q4_0 GEMM: x row stride %d (>= %d, multiple of 8)", a.ldx, K);
  const int ks = a.ks > 0 ? a.ks : 1;
  if (ks > 1 && a.epi != GEMM_F32) return e4b_fail(E4B_EINVAL, "q4_0 GEMM: split-K needs the f32 epilogue");
  if (ks > W.nb) return e4b_fail(E4B_EINVAL, "q4_0 GEMM: %d K slices for %d blocks", ks, W.nb);
  int64_t units = W.rows;
  switch (a.epi) {
    case GEMM_F32:
      if (!a.Y) return e4b_fail(E4B_EINVAL, "q4_0 GEMM: null output");
      break;
    case GEMM_GLU:
      if (!a.Yh || a.ff < 1 || 2 * a.ff != W.rows)
        return e4b_fail(E4B_EINVAL, "q4_0 GEMM: GeGLU needs 2*ff rows");
      units = a.ff;
      break;
    default: return e4b_fail(E4B_EINVAL, "q4_0 GEMM: epilogue %d", a.epi);
  }
  // blocks per split-K slice; the consumer sums exactly `ks` slices, so every
  // slice must hold blocks
  const int nbs = slice_blocks(W.nb, ks);
  const int kslices = (W.nb + nbs - 1) / nbs;
  if (kslices != ks)
    return e4b_fail(E4B_EINVAL, "q4_0 GEMM: %d blocks do not split into %d slices (use q40_gemm_kslices)", W.nb, ks);
  const VariantSet set = variants(a.epi, W.nb % 2 == 0);
  // the kernel addresses activations by 32-bit byte offsets and token tiles
  // by grid y: more tokens than those hold go in several launches
  const int64_t row_bytes = (int64_t)a.ldx * 2;
  int64_t most = (int64_t)0xffffffffll / row_bytes;
  most = std::min<int64_t>(most, 65535 * 32);
  if (most >= 128) most = most / 128 * 128;  // whole tiles (rows of 32 MiB and more: as many as fit)
  if (a.M <= most) {
    const Variant* v = choose(set, a.epi, units, W.nb, a.M, ks, nullptr);
    if (!v) return E4B_EHIP;
    v->go(a, nbs, (unsigned)((a.M + 32 * v->T - 1) / (32 * v->T)), (unsigned)ks, st);
  } else {
    if (ks > 1) return e4b_fail(E4B_EINVAL, "q4_0 GEMM: %d rows of %d in %d K slices", a.M, a.ldx, ks);
    for (int64_t m0 = 0; m0 < a.M; m0 += most) {
      GemmArgs c = a;
      c.M = (int)std::min<int64_t>(most, a.M - m0);
      c.X = a.X + m0 * a.ldx;
      if (a.Y) c.Y = a.Y + m0 * units;
      if (a.Yh) c.Yh = a.Yh + m0 * units;
      const Variant* v = choose(set, c.epi, units, W.nb, c.M, 1, nullptr);
      if (!v) return E4B_EHIP;
      v->go(c, nbs, (unsigned)((c.M + 32 * v->T - 1) / (32 * v->T)), 1, st);
    }
  }
  E4B_HIP(hipGetLastError());
  return E4B_OK;
}

int launch_q40_gemm(const Q40Mat& W, const uint16_t* X, int M, float* Y, uint16_t* Yh, int64_t ff, hipStream_t st) {
  GemmArgs a{};
  a.W = W;
  a.X = X;
  a.M = M;
  a.ldx = W.nb * 32;
  a.epi = Yh ? GEMM_GLU : GEMM_F32;
  a.Y = Y;
  a.Yh = Yh;
  a.ff = ff;
  a.ks = 1;
  return launch_q40_gemm(a, st);
}

// For the tests of every tile: the one that e4b_k_q40_gemm (geglu 0; units
// rows) or e4b_k_q40_gemm_geglu (geglu 1; units = ff) takes.  tile: token
// rows, outputs and waves of a workgroup, K groups, blocks a K stage,
// workgroups that share a CU.
extern "C" int e4b_q40_gemm_tile(int64_t units, int64_t cols, int m, int geglu, int32_t* tile) {
  if (units < 1 || cols < 32 || cols % 32 || cols > INT_MAX || m < 1 || !tile)
    return e4b_fail(E4B_EINVAL, "e4b_q40_gemm_tile: bad arguments");
  const int epi = geglu ? GEMM_GLU : GEMM_F32, nb = (int)(cols / 32);
  const Variant* v = choose(variants(epi, nb % 2 == 0), epi, units, nb, m, 1, nullptr);
  if (!v) return E4B_EHIP;
  tile[0] = 32 * v->T;
  tile[1] = 32 * v->RW * (geglu ? 1 : v->NT);
  tile[2] = v->RW * v->KW;
  tile[3] = v->KW;
  tile[4] = v->KW * v->KBL;
  tile[5] = v->occ.load(std::memory_order_relaxed);
  return E4B_OK;
}
