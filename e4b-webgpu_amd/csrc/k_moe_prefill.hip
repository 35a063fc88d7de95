// k_moe_prefill.hip -- the MoE FFN half-layer over M prompt tokens (the
// batched prefill of the A4B engine, src/engine-a4b.js:478-549 routerTopB /
// expGroup / guGsg32 / downGsg32 / waccB, kernels/expgroup.wgsl:15-50,
// kernels/q40gugrp.wgsl:47-103), with the per-token arithmetic of the decode
// half-layer (k_moe.hip):
//
//   router + top-8      the decode kernels over token rows (bit-identical picks)
//   k_moe_group         counting sort of the M*8 (token, slot) draws by expert
//                       into contiguous runs, cut into tiles of <= 64 rows
//   grouped GEMMs       expert gate/up + GeGLU and expert down on the matrix
//                       cores (k_gemm_grp.hip): each tile reads its expert's
//                       rows once for up to 64 draws; the dense branch's two
//                       products over all M tokens are tiles of the same
//                       launches
//   k_moe_combine_tail  moe[m] = sum_k w_k down_sorted[pos(m, k)], in k order,
//                       and the decode tail
#include <algorithm>

#include "../../include/e4b.h"
#include "kernels.h"
#include "moe.h"
#include "util.h"

namespace {

constexpr int K = kMoeTopK;
constexpr int kMoePfMaxTokens = 1024;
constexpr int kTileRows = kGroupTileRows;

// one workgroup: histogram of the draws' experts in LDS, exclusive scan,
// placement (list[slot] = draw, pos[draw] = slot) and the tile table.  The
// order of draws inside an expert's run depends on LDS atomics; every output
// row is computed from its own input row only, so results do not.
//
// All latency.  A thread keeps its draws (at most 8) and the rank that the
// histogram's atomic returned for each, so the picks are read once and one
// round of atomics places them; rows and tiles are scanned together (16 bits
// each) by lane shifts.
// (One thread scanning 128 experts, the picks read twice: 8.8 us over 512
// tokens; now 5.4.)
__global__ __launch_bounds__(1024) void k_moe_group(const uint32_t* __restrict__ topk_idx, int npairs, int E,
                                                    uint32_t* __restrict__ list, uint32_t* __restrict__ pos,
                                                    int4* __restrict__ tiles, int* __restrict__ ntiles) {
  constexpr int D = kMoePfMaxTokens * K / 1024;  // draws per thread
  __shared__ int cnt[256];
  __shared__ uint32_t off[256];  // rows before the expert, tiles before it << 16
  __shared__ uint32_t wtot[4];
  const int t = threadIdx.x, lane = t & 63;
  int e[D], rank[D];
#pragma unroll
  for (int i = 0; i < D; ++i) e[i] = t + 1024 * i < npairs ? min((int)topk_idx[t + 1024 * i], E - 1) : -1;
  if (t < 256) cnt[t] = 0;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < D; ++i) rank[i] = e[i] >= 0 ? atomicAdd(&cnt[e[i]], 1) : 0;
  __syncthreads();
  uint32_t own = 0, sum = 0;
  if (t < 256) {
    const int n = cnt[t];
    own = (uint32_t)n | (uint32_t)((n + kTileRows - 1) / kTileRows) << 16;
    sum = own;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t o = __shfl_up(sum, d, 64);
      sum += lane >= d ? o : 0u;
    }
    if (lane == 63) wtot[t >> 6] = sum;
  }
  __syncthreads();
  if (t < 256) {
    for (int w = 0; w < t >> 6; ++w) sum += wtot[w];
    const uint32_t ex = sum - own;
    off[t] = ex;
    const int n = (int)(own & 0xffffu), row = (int)(ex & 0xffffu), tile = (int)(ex >> 16);
    for (int j = 0; j * kTileRows < n; ++j)
      tiles[tile + j] = make_int4(t, row + j * kTileRows, min(kTileRows, n - j * kTileRows), 0);
    if (t == 255) *ntiles = (int)(sum >> 16);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < D; ++i)
    if (e[i] >= 0) {
      const int p = t + 1024 * i, s = (int)(off[e[i]] & 0xffffu) + rank[i];
      list[s] = (uint32_t)p;
      pos[p] = (uint32_t)s;
    }
}

// One workgroup per token row m: moe[m] = sum_k w[m][k] down[pos[m K + k]], in
// slot order, and the decode tail (k_moe_tail) of it and the dense branch's
// output.  Bounded by the reads of the K sorted rows: a thread owns four
// adjacent elements, so that all its loads are in flight at once (12 single
// elements a thread, in a loop, took 22 us over 512 rows).
// Measured over 512 rows of 2816: 13.4 us, in two kernels 9.9 + 6.6 and the
// launch between them (the layer, with the grouping above, 260 -> 247).
constexpr int kCtThreads = 768;  // 4 elements each: H <= 3072
DEV float4 ld4(const float* p) {  // 4-byte aligned
  float4 v;
  __builtin_memcpy(&v, p, 16);
  return v;
}
DEV float4 fma4(float s, float4 a, float4 b) {
  return make_float4(fmaf(s, a.x, b.x), fmaf(s, a.y, b.y), fmaf(s, a.z, b.z), fmaf(s, a.w, b.w));
}
DEV float dot4(float4 a) { return fmaf(a.x, a.x, fmaf(a.y, a.y, fmaf(a.z, a.z, a.w * a.w))); }
DEV float ct_sum(float v, float* red) {  // over the workgroup; red: one float a wave
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  lds_sync();
  float s = 0.f;
#pragma unroll
  for (int w = 0; w < kCtThreads / 64; ++w) s += red[w];
  return s;
}
__global__ __launch_bounds__(kCtThreads) void k_moe_combine_tail(MoeArgs A, const float* __restrict__ down,
                                                                 const uint32_t* __restrict__ pos) {
  __shared__ float red[3][kCtThreads / 64];
  const int H = A.H, m = blockIdx.x;
  const bool in = 4 * (int)threadIdx.x < H;
  const int i = min(4 * (int)threadIdx.x, H - 4);
  const int64_t o = (int64_t)m * H + i;
  float4 r[K];
#pragma unroll
  for (int k = 0; k < K; ++k) r[k] = ld4(down + (int64_t)pos[m * K + k] * H + i);
  const float4 d = ld4(A.dense_out + o);
  const float4 w1 = ld4(A.post_ffw1 + i), w2 = ld4(A.post_ffw2 + i), wp = ld4(A.post_ffw + i), h = ld4(A.h + o);
  float4 mo = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int k = 0; k < K; ++k) mo = fma4(A.topk_w[m * K + k], r[k], mo);
  if (in) *reinterpret_cast<float4*>(A.moe_out + o) = mo;
  const float s1 = wave_sum(in ? dot4(d) : 0.f), s2 = wave_sum(in ? dot4(mo) : 0.f);
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = s1;
    red[1][threadIdx.x >> 6] = s2;
  }
  lds_sync();
  float t1 = 0.f, t2 = 0.f;
#pragma unroll
  for (int w = 0; w < kCtThreads / 64; ++w) {
    t1 += red[0][w];
    t2 += red[1][w];
  }
  const float i1 = rms_inv(t1, H, A.eps), i2 = rms_inv(t2, H, A.eps);
  const float4 c = make_float4(d.x * i1 * w1.x + mo.x * i2 * w2.x, d.y * i1 * w1.y + mo.y * i2 * w2.y,
                               d.z * i1 * w1.z + mo.z * i2 * w2.z, d.w * i1 * w1.w + mo.w * i2 * w2.w);
  const float i3 = rms_inv(ct_sum(in ? dot4(c) : 0.f, red[2]), H, A.eps);
  if (in) {
    const float4 y = make_float4((h.x + c.x * i3 * wp.x) * A.layer_scale, (h.y + c.y * i3 * wp.y) * A.layer_scale,
                                 (h.z + c.z * i3 * wp.z) * A.layer_scale, (h.w + c.w * i3 * wp.w) * A.layer_scale);
    __builtin_memcpy(A.h_out + o, &y, 16);
  }
}

}  // namespace

size_t moe_prefill_scratch(const MoeArgs& a, int M, MoePrefillBufs* b, uint8_t* base) {
  const int H = a.H, E = a.E, FF = a.FF, FF2 = a.FF2;
  const size_t P = (size_t)M * K;
  // the most tiles: every expert that P draws can reach ends in a part-empty one
  const int max_tiles = (int)((P + (kTileRows - 1) * std::min<size_t>(E, P)) / kTileRows);
  size_t cur = 0;
  auto take = [&](size_t bytes) {
    uint8_t* p = base ? base + cur : nullptr;
    cur += E4B_ALIGN256(bytes);
    return p;
  };
  uint8_t* p_scores = take((size_t)M * E * 4);
  uint8_t* p_xd = take((size_t)M * H * 2);
  uint8_t* p_xm = take((size_t)M * H * 2);
  uint8_t* p_idx = take(P * 4);
  uint8_t* p_w = take(P * 4);
  uint8_t* p_list = take(P * 4);
  uint8_t* p_pos = take(P * 4);
  uint8_t* p_tiles = take((size_t)max_tiles * 16);
  uint8_t* p_nt = take(16);
  uint8_t* p_g = take(P * FF * 2);
  uint8_t* p_d = take(P * H * 4);
  uint8_t* p_gd = take((size_t)M * FF2 * 2);
  uint8_t* p_dense = take((size_t)M * H * 4);
  uint8_t* p_moe = take((size_t)M * H * 4);
  if (b) {
    b->scores = (float*)p_scores;
    b->xd = (uint16_t*)p_xd;
    b->xm = (uint16_t*)p_xm;
    b->topk_idx = (uint32_t*)p_idx;
    b->topk_w = (float*)p_w;
    b->list = (uint32_t*)p_list;
    b->pos = (uint32_t*)p_pos;
    b->tiles = (int4*)p_tiles;
    b->ntiles = (int*)p_nt;
    b->max_tiles = max_tiles;
    b->g_sorted = (uint16_t*)p_g;
    b->d_sorted = (float*)p_d;
    b->g_dense = (uint16_t*)p_gd;
    b->dense_out = (float*)p_dense;
    b->moe_out = (float*)p_moe;
  }
  return cur;
}

int launch_moe_prefill(const MoeArgs& base, int M, const MoePrefillBufs& b, hipStream_t st) {
  const int H = base.H, E = base.E, FF = base.FF, FF2 = base.FF2;
  if (M < 1 || M > kMoePfMaxTokens)
    return e4b_fail(E4B_EINVAL, "MoE prefill: %d tokens (1..1024 per call)", M);
  if (E < K || E > 256 || H % 256 || H > 4 * kCtThreads || FF % 32 || FF2 % 32)
    return e4b_fail(E4B_EINVAL, "MoE prefill: bad shape (H=%d E=%d FF=%d FF2=%d)", H, E, FF, FF2);
  MoeArgs a = base;
  a.scores = b.scores;
  a.xd = b.xd;
  a.xm = b.xm;
  a.topk_idx = b.topk_idx;
  a.topk_w = b.topk_w;
  a.dense_out = b.dense_out;
  a.moe_out = b.moe_out;
  int rc;
  if ((rc = launch_moe_router_rows(a, M, st)) || (rc = launch_moe_topk_rows(a, M, st))) return rc;
  hipLaunchKernelGGL(k_moe_group, dim3(1), dim3(1024), 0, st, b.topk_idx, M * K, E, b.list, b.pos, b.tiles, b.ntiles);
  E4B_HIP(hipGetLastError());
  // expert gate/up + GeGLU over the sorted draws and the dense branch's over
  // all tokens in one launch, then both down projections in another
  GemmArgs g{}, d{};
  g.W = a.exp_gu;
  g.X = b.xm;
  g.M = M * K;
  g.ldx = H;
  g.epi = GEMM_GLU;
  g.Yh = b.g_sorted;
  g.ff = FF;
  g.ks = 1;
  g.tiles = b.tiles;
  g.ntiles = b.ntiles;
  g.max_tiles = b.max_tiles;
  g.group_rows = 2 * (int64_t)FF;
  g.gather = b.list;
  g.gather_div = K;
  d.W = a.dense_gu;
  d.X = b.xd;
  d.M = M;
  d.ldx = H;
  d.epi = GEMM_GLU;
  d.Yh = b.g_dense;
  d.ff = FF2;
  d.ks = 1;
  if ((rc = launch_q40_gemm_grouped(g, d, st))) return rc;
  g.W = a.exp_down;
  g.X = b.g_sorted;
  g.ldx = FF;
  g.epi = GEMM_F32;
  g.Y = b.d_sorted;
  g.Yh = nullptr;
  g.ff = 0;
  g.group_rows = H;
  g.gather = nullptr;
  g.gather_div = 1;
  d.W = a.dense_down;
  d.X = b.g_dense;
  d.ldx = FF2;
  d.epi = GEMM_F32;
  d.Y = a.dense_out;
  d.Yh = nullptr;
  d.ff = 0;
  if ((rc = launch_q40_gemm_grouped(g, d, st))) return rc;
  hipLaunchKernelGGL(k_moe_combine_tail, dim3(M), dim3(kCtThreads), 0, st, a, b.d_sorted, b.pos);
  E4B_HIP(hipGetLastError());
  return E4B_OK;
}
