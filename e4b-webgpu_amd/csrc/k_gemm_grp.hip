// k_gemm_grp.hip -- the q4_0 GEMM's grouped launch (the expert-indexed MoE
// prefill): row tiles of up to 64 draws of one expert, and beside them the
// tiles of an ordinary product over all token rows (the dense branch).
#include "../../include/e4b.h"
#include "gemm_variants.h"
#include "util.h"

namespace gemm {

// 64 draws x 64 outputs (GeGLU) or 128 columns (f32), 4 waves.  A matrix whose
// rows have an odd number of blocks loads its scales singly, the other not.
template <int EPI, bool GALN, bool DALN>
void go_grp(const GemmArgs& g, const GemmArgs& d, hipStream_t st) {
  constexpr int T = 2, NT = 2, RW = 2, KW = 2, KBL = 2;
  constexpr int UC = EPI == GEMM_GLU ? 32 * RW : 32 * RW * NT, TOK = 32 * T;
  static_assert(TOK == kGroupTileRows, "a group's row tile");
  const int64_t gu = EPI == GEMM_GLU ? g.ff : g.group_rows, du = EPI == GEMM_GLU ? d.ff : d.W.rows;
  const int gbx = (int)((gu + UC - 1) / UC), dbx = (int)((du + UC - 1) / UC);
  // Up to 64 tokens the dense product's serial K loop can outlast the experts'
  // tiles, and in tiles of 32 tokens a stage of it takes 3/4 of the time.  A
  // half-layer of 1 token 57 -> 48 us (hidden 2816, 128 experts of 704, dense
  // 2112), of 37 tokens 49 -> 42 (hidden 1024, 16 experts of 160, dense 2112),
  // where launches of its own took 56 and 45.  At 128 tokens tiles of 32 were
  // 10 % faster at the second shape and 2 % slower at the first with dense 2080.
  const int dtok = d.M <= 64 ? 32 : TOK;
  const int ndense = dbx * ((d.M + dtok - 1) / dtok);
  hipLaunchKernelGGL((k_q40_gemm_grp<T, NT, RW, KW, KBL, EPI, GALN, DALN>), dim3((unsigned)(ndense + gbx * g.max_tiles)),
                     dim3(64 * RW * KW), 0, st, g, d, ndense, dbx, dtok, gbx);
}

}  // namespace gemm

int launch_q40_gemm_grouped(const GemmArgs& g, const GemmArgs& d, hipStream_t st) {
  for (const GemmArgs* a : {&g, &d}) {
    const int K = a->W.nb * 32;
    if (a->M < 1 || K < 32) return e4b_fail(E4B_EINVAL, "grouped q4_0 GEMM: empty operand (M=%d K=%d)", a->M, K);
    if ((uint64_t)a->W.rows * (uint64_t)a->W.nb * 16u > 0xffffffffull)
      return e4b_fail(E4B_EINVAL, "q4_0 GEMM: a %lld x %d-block matrix exceeds the 4 GiB plane limit",
                      (long long)a->W.rows, a->W.nb);
    if (a->ldx < K || a->ldx % 8 || a->M > 0xffffffffll / (2 * (int64_t)a->ldx))
      return e4b_fail(E4B_EINVAL, "grouped q4_0 GEMM: %d rows, stride %d", a->M, a->ldx);
    if (a->epi != g.epi || (a->epi != GEMM_F32 && a->epi != GEMM_GLU) || a->ks > 1)
      return e4b_fail(E4B_EINVAL, "grouped q4_0 GEMM: epilogues %d and %d, %d slices", g.epi, d.epi, a->ks);
    if (a->epi == GEMM_F32 ? !a->Y : (!a->Yh || a->ff < 1 || 2 * a->ff != (a == &g ? g.group_rows : d.W.rows)))
      return e4b_fail(E4B_EINVAL, "grouped q4_0 GEMM: outputs");
  }
  if (!g.tiles || !g.ntiles || g.max_tiles < 1 || g.group_rows < 1 || g.W.rows % g.group_rows ||
      (g.gather && g.gather_div < 1))
    return e4b_fail(E4B_EINVAL, "q4_0 GEMM: bad grouped-mode arguments");
  const bool ga = g.W.nb % 2 == 0, da = d.W.nb % 2 == 0;
  if (g.epi == GEMM_GLU) {
    if (!ga || !da) return e4b_fail(E4B_EINVAL, "q4_0 GEMM: no grouped GeGLU over rows of %d and %d blocks", g.W.nb,
                               d.W.nb);
    gemm::go_grp<GEMM_GLU, true, true>(g, d, st);
  } else {
    (ga ? da ? gemm::go_grp<GEMM_F32, true, true> : gemm::go_grp<GEMM_F32, true, false>
        : da ? gemm::go_grp<GEMM_F32, false, true> : gemm::go_grp<GEMM_F32, false, false>)(g, d, st);
  }
  E4B_HIP(hipGetLastError());
  return E4B_OK;
}
