// gemm_kernel.h -- q4_0 weight x f16 activation GEMM on the gfx950 matrix
// cores, the batched-prefill counterpart of the decode GEMV
// (src/engine-a4b.js:465-585 runs its prefill as multi-column GEMVs,
// kernels/q40mm.wgsl / kernels/q40sg.wgsl; here it is an MFMA GEMM).  Device
// code; k_gemm.hip chooses and launches the variants.
//
//   Y[m][n] = sum_k X[m][k] W[n][k],  W q4_0 [N][K] (repacked planes),
//   X f16 [M][K] row-major (row stride ldx), Y f32 [M][N]; epilogues: split-K
//   partial slices (Y + z M N, summed by the consumer), or the GeGLU over
//   W = [gate; up] to f16 [M][FF] = gelu(gate) * up.
//
// v_mfma_f32_32x32x16_f16 with A = a 32-token x 16-k slice of X and B = the
// 16-k x 32-row slice of W^T: lane l holds A[l % 32][8 (l / 32) + t] (t < 8),
// B[8 (l / 32) + t][l % 32] and D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32]
// (r < 16), so every lane owns one weight row n = l % 32 of the tile.  The 32
// k of a q4_0 block go to its two instructions as (0-7, 16-23) and (8-15,
// 24-31), which makes both operands of a lane contiguous: two nibble words
// and 32 bytes of activations.  The nibbles become the exact f16 values n - 8;
// each block is accumulated from zero and then scaled by the row's block
// scale in f32, as the decode GEMV does, so the products are exact and only
// the f32 summation order differs from it.
//
// What bounds it: per 32 x 32 tile and block, two matrix instructions (64
// cycles of a SIMD's matrix core) and 16 scale multiply-adds plus the nibble
// conversion (9 instructions a nibble word, two words a lane and row tile,
// shared by the T token tiles) on the vector unit, 4 cycles each.  The two
// units run side by side only if the instructions are interleaved: a
// register-only loop takes 32.6 ns a tile and SIMD with the matrix
// instructions alone, 37.3 with the multiply-adds alone, 43.6 with both (two
// waves per SIMD), i.e. 1.5 PFLOP/s, while this card's library f16 product
// reaches 1.1-1.2.  So the loop below is written as a software pipeline
// (multiply-adds of one tile between the matrix instructions of the next).
//
// A workgroup is RW x KW waves: RW groups of NT row tiles of 32, KW groups
// that share the K loop (each takes KBL of every KW KBL blocks; their sums
// meet in LDS at the end).  Splitting K inside the workgroup instead of over
// the grid needs no partial sums in memory, so also a call that has no
// scratch can fill the chip: a 2048 x 16384 matrix over 512 tokens 148 -> 55
// us, 3072 x 2048 over 37 tokens 17.7 -> 5 us (MI355X; before: 4 waves, one
// K group, operands staged through registers).
#pragma once
#include <atomic>
#include <type_traits>

#include "kernels.h"

namespace gemm {

typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) const void glb_void;

// 8 exact f16 values (n - 8) of one repacked nibble word, in element order.
// A pair of nibbles at bits 0-3 / 16-19 under the pattern 0x6400 is 1024 + n;
// at bits 4-7 / 20-23 it is 1024 + 16 n, and (1024 + 16 n) / 16 - 72 = n - 8:
// one shift, four and-ors, two packed adds and two packed fmas per 8 values.
// `mag` is 0x64006400 in a vector register (and-or takes one scalar operand).
DEV h8 nib_word_f16(uint32_t w, uint32_t mag) {
  const uint32_t M = 0x000F000Fu, M4 = 0x00F000F0u;
  const uint32_t v = w >> 8;
  const h2v p0 = __builtin_bit_cast(h2v, (w & M) | mag), p1 = __builtin_bit_cast(h2v, (v & M) | mag);
  const h2v p2 = __builtin_bit_cast(h2v, (w & M4) | mag), p3 = __builtin_bit_cast(h2v, (v & M4) | mag);
  const h2v off = {(_Float16)-1032.0f, (_Float16)-1032.0f}, six = {(_Float16)0.0625f, (_Float16)0.0625f};
  const h2v o16 = {(_Float16)-72.0f, (_Float16)-72.0f};
  const h2v a = p0 + off, b = p1 + off;
  const h2v c = __builtin_elementwise_fma(p2, six, o16), d = __builtin_elementwise_fma(p3, six, o16);
  return h8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// gelu_tanh (common.h) as g / (1 + e^-2t): 1 + tanh(t) = 2 / (1 + e^-2t), a
// dozen instructions instead of tanhf's fifty, and no cancellation for t < 0.
// At the clamp, t <= -20, it is 0 as there (tanhf(-20) is -1): e^-40 g would
// grow with a large gate again.
DEV float gelu_sigmoid(float g) {
  const float t = 0.7978845608028654f * (g + 0.044715f * g * g * g);
  const float e = t > -20.f ? __expf(-2.f * fminf(t, 20.f)) : __builtin_inff();
  return g / (1.f + e);
}

__device__ const uint4 kZeros[8] = {};
constexpr int kRsrcWord3 = 0x00020000;  // raw buffer resource, 32-bit data format

// 16-byte piece p of staged row r sits in slot p ^ swz(r): rows 256 bytes or
// a power-of-two fraction apart would put one piece of 16 rows in the same
// banks; the xor spreads them over all 16 columns (P = pieces per row)
template <int P>
DEV int swz(int r) {
  return P >= 16 ? (r & 15) : (r / (P >= 16 ? 1 : 16 / P)) & (P - 1);
}

// keeps the multiply-adds before it where they are written (the compiler
// would sink them past the stage's barrier to the next use of the sums)
DEV void pin8(float* v) {
  asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]));
}

template <int T, int NT, int RW, int KW, int KBL>
struct Shape {
  static constexpr int TOK = 32 * T;            // token rows per workgroup
  static constexpr int COLS = 32 * RW * (NT);   // staged weight rows per workgroup
  static constexpr int SB = KW * KBL;           // q4_0 blocks per stage
  static constexpr int NTHR = 64 * RW * KW;
  static constexpr int WPC = COLS * SB;         // 16-byte pieces of a weight stage
  static constexpr int XPC = TOK * SB * 4;      // and of an activation stage
  static constexpr int BUF = WPC + XPC;
};

// EPI GEMM_GLU: NT = 2, tile 0 a gate tile, tile 1 the up tile of the same
// outputs.  Other epilogues: NT tiles of 32 adjacent row groups.
// bx: row tile; by: first token row (GRP: entry of the tile table); bufa,
// bufb: two separate LDS arrays of Shape::BUF pieces (the compiler then knows
// that the copies into one do not alias the reads of the other), scb: the
// scales of two stages.
template <int T, int NT, int RW, int KW, int KBL, int EPI, bool GRP, bool ALN>
DEV void gemm_tile(const GemmArgs& a, int nb, int nbs, int bx, int by, u32x4* bufa, u32x4* bufb, uint32_t* scb) {
  using S = Shape<T, NT, RW, KW, KBL>;
  constexpr int SB = S::SB, NTHR = S::NTHR, TOK = S::TOK;
  constexpr int WJ = S::WPC / NTHR, XJ = S::XPC / NTHR;  // pieces per thread
  static_assert(WJ >= 1 && XJ >= 1 && S::WPC % NTHR == 0 && S::XPC % NTHR == 0, "whole pieces per thread");
  static_assert((SB & (SB - 1)) == 0 && SB <= 16, "power-of-two stage");
  static_assert(EPI != GEMM_GLU || NT == 2, "a gate and an up tile");
  static_assert(KW == 1 || S::BUF * 16 >= KW * RW * NT * 2048, "reduction fits a stage buffer");
  const Q40Mat& W = a.W;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hi = lane >> 5;
  const int rw = wave % RW, kg = wave / RW;
  const int64_t units = EPI == GEMM_GLU ? a.ff : (GRP ? a.group_rows : W.rows);
  constexpr int UC = EPI == GEMM_GLU ? 32 * RW : 32 * RW * NT;  // output columns per workgroup
  int tok0, nrows;
  int64_t wbase = 0;
  if constexpr (GRP) {
    const int4 tl = a.tiles[by];
    wbase = (int64_t)tl.x * a.group_rows;
    tok0 = tl.y;
    nrows = tl.z;
  } else {
    tok0 = by;
    nrows = min(TOK, a.M - tok0);
  }
  const int64_t c0 = (int64_t)bx * UC;
  const int kz = blockIdx.z;
  const int kbeg = kz * nbs, kend = min(nb, kbeg + nbs);
  // global row of staged weight row r (rows past the end repeat the last one
  // and are never stored)
  auto grow = [&](int r) -> int64_t {
    if constexpr (EPI == GEMM_GLU)
      return wbase + (r >= 32 * RW ? a.ff : 0) + min(c0 + (r & (32 * RW - 1)), units - 1);
    else
      return wbase + min(c0 + r, units - 1);
  };
  // Staging.  Weights: [row][SB blocks], a row's blocks contiguous in memory
  // and xor-swizzled in LDS.  Activations: [BP blocks][token][pieces], so
  // that a fragment's block is an immediate offset and a thread's copies of
  // all blocks share one address register.  Every copy is a scalar offset
  // that advances with the stage plus a fixed per-thread offset.  Blocks past
  // the K range (the last stage only) meet zeros: their activations are
  // copied from a page of zeros, while a weight copy runs at most SB - 1
  // blocks on, into the next row or the scale plane behind the nibbles (at
  // least 256 bytes).  (Buffer loads: the compiler counts a global load into
  // LDS as a flat access, and then waits for all LDS reads at once.)
  const auto wrs = __builtin_amdgcn_make_buffer_rsrc((void*)W.nib, 0, 0xffffffffu, kRsrcWord3);
  const auto xrs = __builtin_amdgcn_make_buffer_rsrc((void*)a.X, 0, 0xffffffffu, kRsrcWord3);
  const auto zrs = __builtin_amdgcn_make_buffer_rsrc((void*)kZeros, 0, sizeof(kZeros), kRsrcWord3);
  uint32_t woff[WJ];
#pragma unroll
  for (int j = 0; j < WJ; ++j) {
    const int i = j * NTHR + tid, r = i / SB;
    woff[j] = ((uint32_t)grow(r) * (uint32_t)nb + (uint32_t)((i % SB) ^ swz<SB>(r))) * 16u;
  }
  constexpr int BP = ALN ? 2 : 1, PB = 4 * BP;  // blocks, and 16-byte pieces, of a row side by side
  static_assert(KBL % BP == 0, "whole block pairs per K group");
  constexpr int XR = TOK * PB > NTHR ? TOK * PB / NTHR : 1;  // token rows of a thread's copies
  static_assert(TOK * PB % NTHR == 0 || NTHR % (TOK * PB) == 0, "whole token rows");
  uint32_t xoff[XR];  // (the host keeps the token rows of a launch under 4 GiB)
#pragma unroll
  for (int j = 0; j < XR; ++j) {
    const int r = ((j * NTHR + wave * 64) % (TOK * PB) + lane) / PB;
    int64_t row = tok0 + min(r, nrows - 1);
    if constexpr (GRP) row = a.gather ? (int64_t)(a.gather[row] / (uint32_t)a.gather_div) : row;
    xoff[j] = (uint32_t)row * (uint32_t)a.ldx * 2u + (uint32_t)((lane % PB) ^ swz<PB>(r)) * 16u;
  }
  auto issue = [&](u32x4* buf, int kb0) {
#pragma unroll
    for (int j = 0; j < WJ; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, (lds_void*)(buf + j * NTHR + wave * 64), 16, (int)woff[j],
                                               kb0 * 16, 0, 0);
#pragma unroll
    for (int j = 0; j < XJ; ++j) {
      lds_void* dst = (lds_void*)(buf + S::WPC + j * NTHR + wave * 64);
      const int blk = kb0 + (j * NTHR + wave * 64) / (TOK * PB) * BP;  // uniform per wave
      if (blk < kend)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xrs, dst, 16, (int)xoff[j % XR], blk * 64, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(zrs, dst, 16, (lane % PB) * 16, 0, 0, 0);
    }
  };
  // block scales.  ALN (an even number of blocks a row): the scales of two
  // stages are copied to LDS in 4-byte pieces -- a row's scales of one stage
  // are a few bytes of a 128-byte line, so loading them stage by stage in
  // every lane moved more lines than the weights do -- and read from there
  // once, into registers.  Else single loads, one stage ahead, kept apart
  // (packing them would wait for each).
  int lrow[NT];
#pragma unroll
  for (int u = 0; u < NT; ++u) lrow[u] = (u * RW + rw) * 32 + l32;
  typedef uint16_t sv __attribute__((ext_vector_type(KBL)));
  struct Scales {
    std::conditional_t<ALN, sv, uint16_t[KBL]> v[NT];
  };
  const auto srs = __builtin_amdgcn_make_buffer_rsrc((void*)W.sc, 0, 0xffffffffu, kRsrcWord3);
  auto issue_scales_lds = [&](int kb0) {
    if constexpr (ALN) {
      constexpr int SJ = (S::COLS * SB + NTHR - 1) / NTHR;
#pragma unroll
      for (int j = 0; j < SJ; ++j) {
        const int i = j * NTHR + tid;
        if (S::COLS * SB % NTHR == 0 || j * NTHR + wave * 64 < S::COLS * SB) {
          const uint32_t e = (uint32_t)grow(i / SB) * (uint32_t)nb + (uint32_t)min(kb0 + 2 * (i % SB), nb - 2);
          __builtin_amdgcn_raw_ptr_buffer_load_lds(srs, (lds_void*)(scb + j * NTHR + wave * 64), 4, (int)(e * 2u), 0, 0,
                                                   0);
        }
      }
    }
  };
  auto read_scales = [&](Scales& s, int half) {
    if constexpr (ALN) {
#pragma unroll
      for (int u = 0; u < NT; ++u)
        s.v[u] = *reinterpret_cast<const sv*>(reinterpret_cast<const uint16_t*>(scb) + lrow[u] * (2 * SB) + half * SB +
                                              kg * KBL);
    }
  };
  auto issue_scales = [&](Scales& s, int kb0) {
    if constexpr (!ALN) {
#pragma unroll
      for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int j = 0; j < KBL; ++j)
          s.v[u][j] = W.sc[(uint32_t)grow(lrow[u]) * (uint32_t)nb + (uint32_t)min(kb0 + kg * KBL + j, nb - 1)];
    }
  };
  // LDS byte addresses of this lane's fragments: block 0 of weight row
  // 32 rw + l32 (block j at the same address xor 16 j), and the two 16-byte
  // halves of its 32 bytes of an activation block
  const int b0 = kg * KBL;
  const int wl0 = ((rw * 32 + l32) * SB + (b0 ^ swz<SB>(l32))) * 16 + hi * 8;
  const int xl0 = (S::WPC + b0 / BP * (TOK * PB) + l32 * PB + ((2 * hi) ^ swz<PB>(l32))) * 16;
  uint32_t mag = 0x64006400u;
  asm("" : "+v"(mag));

  float acc[NT][T][16];
#pragma unroll
  for (int u = 0; u < NT; ++u)
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[u][t][r] = 0.f;

  auto ldw = [&](const u32x4* buf, int j, int u) {
    return *reinterpret_cast<const u32x2*>(reinterpret_cast<const char*>(buf) + (wl0 ^ (16 * j)) +
                                           u * (RW * 32 * SB * 16));
  };
  auto ldx = [&](const u32x4* buf, int j, int s, int t) {
    return __builtin_bit_cast(h8, *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(buf) +
                                                                  (xl0 ^ (16 * s + 64 * (j % BP))) +
                                                                  (j / BP * TOK + 32 * t) * (PB * 16)));
  };
  // one stage, software pipelined over its KBL x T x NT tiles: while a tile's
  // two matrix instructions run, the vector unit does the scale
  // multiply-adds of the tile before it
  auto compute = [&](const u32x4* buf, const Scales& sc) {
    constexpr int N = KBL * T * NT;
    f16v d[2];
    h8 bw[NT][2];
    float ds[KBL][NT];
    h8 xa[2][2];
    u32x2 wn[NT];
#pragma unroll
    for (int u = 0; u < NT; ++u) wn[u] = ldw(buf, 0, u);
    xa[0][0] = ldx(buf, 0, 0, 0);
    xa[0][1] = ldx(buf, 0, 1, 0);
#pragma unroll
    for (int k = 0; k < N + 1; ++k) {
      const int j = k / (T * NT), t = k / NT % T, u = k % NT;
      if (k < N) {
        const int i = k / NT;
        if (t == 0) {
          bw[u][0] = nib_word_f16(wn[u].x, mag);
          bw[u][1] = nib_word_f16(wn[u].y, mag);
          ds[j][u] = h2f(sc.v[u][j]);
          asm("" : "+v"(ds[j][u]));  // converted once, not folded into every multiply-add
          if (j + 1 < KBL) wn[u] = ldw(buf, j + 1, u);
        }
        if (u == 0 && i + 1 < KBL * T) {
          xa[(i + 1) & 1][0] = ldx(buf, (i + 1) / T, 0, (i + 1) % T);
          xa[(i + 1) & 1][1] = ldx(buf, (i + 1) / T, 1, (i + 1) % T);
        }
        f16v z = {};
        z = __builtin_amdgcn_mfma_f32_32x32x16_f16(xa[i & 1][0], bw[u][0], z, 0, 0, 0);
        d[k & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xa[i & 1][1], bw[u][1], z, 0, 0, 0);
      }
      if (k >= 1) {
        const int q = k - 1, qj = q / (T * NT), qt = q / NT % T, qu = q % NT;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[qu][qt][r] = fmaf(ds[qj][qu], d[q & 1][r], acc[qu][qt][r]);
        pin8(acc[qu][qt]);
        pin8(acc[qu][qt] + 8);
      }
      if (k < N) {
        __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
        if (t == 0) __builtin_amdgcn_sched_group_barrier(0x002, 19, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // every wave's copies of the stage have landed, and every wave is done
  // with the buffer the next copies overwrite
  auto stage_sync = [&]() {
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    lds_sync();
  };
  Scales sa, sb;
  issue(bufa, kbeg);
  issue_scales_lds(kbeg);
  issue_scales(sa, kbeg);
  for (int kb0 = kbeg;;) {
    stage_sync();
    read_scales(sa, 0);
    read_scales(sb, 1);
    const bool odd = kb0 + SB < kend, more = kb0 + 2 * SB < kend;
    if (odd) {
      issue(bufb, kb0 + SB);
      issue_scales(sb, kb0 + SB);
    }
    compute(bufa, sa);
    if (!odd) break;
    stage_sync();
    kb0 += 2 * SB;
    if (more) {
      issue(bufa, kb0);
      issue_scales_lds(kb0);
      issue_scales(sa, kb0);
    }
    compute(bufb, sb);
    if (!more) break;
  }

  // output: lane owns column l32 of its tile, tokens 32 t + 8 (r / 4) + 4 hi + r % 4
  auto put = [&](int t, int r, const float (&v)[NT]) {
    const int ml = 32 * t + 8 * (r / 4) + 4 * hi + (r % 4);
    if (ml >= nrows) return;
    const int64_t m = tok0 + ml;
    if constexpr (EPI == GEMM_GLU) {
      const int64_t n = c0 + rw * 32 + l32;
      if (n < units) a.Yh[m * a.ff + n] = f2h(gelu_sigmoid(v[0]) * v[1]);
    } else {
#pragma unroll
      for (int u = 0; u < NT; ++u) {
        const int64_t n = c0 + (u * RW + rw) * 32 + l32;
        if (n >= units) continue;
        a.Y[((int64_t)kz * a.M + m) * units + n] = v[u];
      }
    }
  };
  if constexpr (KW == 1) {
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float v[NT];
#pragma unroll
        for (int u = 0; u < NT; ++u) v[u] = acc[u][t][r];
        put(t, r, v);
      }
  } else {
    // the K groups' sums meet in LDS, 8 of a tile's 16 rows at a time; each
    // group adds and stores 8 / KW of them, in group order
    static_assert(8 % KW == 0, "rows per group");
    float* red = reinterpret_cast<float*>(bufa);
#pragma unroll
    for (int c = 0; c < 2 * T; ++c) {
      const int t = c / 2, r0 = 8 * (c % 2);
      lds_sync();
#pragma unroll
      for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int r = 0; r < 8; ++r) red[(((kg * RW + rw) * NT + u) * 8 + r) * 64 + lane] = acc[u][t][r0 + r];
      lds_sync();
#pragma unroll
      for (int i = 0; i < 8 / KW; ++i) {
        const int r = kg * (8 / KW) + i;
        float v[NT];
#pragma unroll
        for (int u = 0; u < NT; ++u) {
          float x = red[((rw * NT + u) * 8 + r) * 64 + lane];
#pragma unroll
          for (int g = 1; g < KW; ++g) x += red[(((g * RW + rw) * NT + u) * 8 + r) * 64 + lane];
          v[u] = x;
        }
        put(t, r0 + r, v);
      }
    }
  }
}

template <int T, int NT, int RW, int KW, int KBL, int EPI, bool ALN>
__global__ __launch_bounds__(64 * RW * KW, 2) void k_q40_gemm(GemmArgs a, int nb, int nbs) {
  using S = Shape<T, NT, RW, KW, KBL>;
  __shared__ __align__(16) u32x4 bufa[S::BUF];
  __shared__ __align__(16) u32x4 bufb[S::BUF];
  __shared__ __align__(16) uint32_t scb[ALN ? S::COLS * S::SB : 4];
  gemm_tile<T, NT, RW, KW, KBL, EPI, false, ALN>(a, nb, nbs, blockIdx.x, blockIdx.y * S::TOK, bufa, bufb, scb);
}

// A grouped product and an ordinary one in one launch: the first ndense
// workgroups are tiles of d (dbx of them side by side, dtok token rows each),
// the rest of g.  The dense branch of an MoE layer alone leaves most of the
// chip idle; in front of the experts' tiles it fills the workgroup slots that
// their last, part-empty wave leaves: a half-layer over 512 tokens 247 -> 239
// us (MI355X; the dense branch in launches of its own: 30 + 17 us).
//
// Tiles of at most 32 live rows (an expert's last draws, the dense branch's
// few or last tokens) are one token tile a wave, half the work of two; K is
// summed in the same order, so a token's result does not depend on its tile.
// GALN, DALN: whether g's and d's rows have an even number of blocks, each for
// its own tiles: a dense width of an odd number must not put the experts'
// product, the far larger one, on the kernel that loads scales singly.
template <int T, int NT, int RW, int KW, int KBL, int EPI, bool GALN, bool DALN>
__global__ __launch_bounds__(64 * RW * KW, 2) void k_q40_gemm_grp(GemmArgs g, GemmArgs d, int ndense, int dbx,
                                                                  int dtok, int gbx) {
  using S = Shape<T, NT, RW, KW, KBL>;
  __shared__ __align__(16) u32x4 bufa[S::BUF];
  __shared__ __align__(16) u32x4 bufb[S::BUF];
  __shared__ __align__(16) uint32_t scb[GALN || DALN ? S::COLS * S::SB : 4];
  int id = blockIdx.x;
  if (id < ndense) {
    const int tok0 = id / dbx * dtok, bx = id % dbx;
    if (T == 2 && (dtok <= 32 || d.M - tok0 <= 32))
      gemm_tile<1, NT, RW, KW, KBL, EPI, false, DALN>(d, d.W.nb, d.W.nb, bx, tok0, bufa, bufb, scb);
    else
      gemm_tile<T, NT, RW, KW, KBL, EPI, false, DALN>(d, d.W.nb, d.W.nb, bx, tok0, bufa, bufb, scb);
    return;
  }
  id -= ndense;
  const int by = id / gbx, bx = id % gbx;
  if (by >= *g.ntiles) return;  // the grid is sized for the most tiles
  if (T == 2 && g.tiles[by].z <= 32)
    gemm_tile<1, NT, RW, KW, KBL, EPI, true, GALN>(g, g.W.nb, g.W.nb, bx, by, bufa, bufb, scb);
  else
    gemm_tile<T, NT, RW, KW, KBL, EPI, true, GALN>(g, g.W.nb, g.W.nb, bx, by, bufa, bufb, scb);
}

// The variants k_gemm.hip chooses from; each translation unit instantiates
// its own.  A variant's kernel and launcher, and how many of its workgroups
// share a CU (0: not asked for yet).
struct Variant {
  int T, NT, RW, KW, KBL;
  const void* kernel;
  void (*go)(const GemmArgs& a, int ks_blocks, unsigned gy, unsigned gz, hipStream_t st);
  std::atomic<int> occ{0};
};

template <int T, int NT, int RW, int KW, int KBL, int EPI, bool ALN>
void launch_variant(const GemmArgs& a, int nbs, unsigned gy, unsigned gz, hipStream_t st) {
  using S = Shape<T, NT, RW, KW, KBL>;
  constexpr int UC = EPI == GEMM_GLU ? 32 * RW : 32 * RW * NT;
  const int64_t units = EPI == GEMM_GLU ? a.ff : a.W.rows;
  hipLaunchKernelGGL((k_q40_gemm<T, NT, RW, KW, KBL, EPI, ALN>), dim3((unsigned)((units + UC - 1) / UC), gy, gz),
                     dim3(S::NTHR), 0, st, a, a.W.nb, nbs);
}

#define GEMM_VARIANT(T, NT, RW, KW, KBL, EPI, ALN)                                                   \
  {                                                                                                  \
    T, NT, RW, KW, KBL, reinterpret_cast<const void*>(k_q40_gemm<T, NT, RW, KW, KBL, EPI, ALN>),     \
        launch_variant<T, NT, RW, KW, KBL, EPI, ALN>                                                 \
  }

}  // namespace gemm
