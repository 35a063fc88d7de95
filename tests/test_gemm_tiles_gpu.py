"""GPU parity of every tile variant of the batched q4_0 GEMM, at the edges of
its tiles, against float64 products of the same f16 activations and the
oracle's dequantised weights.

The variant follows from the shape (rows, columns, tokens).  The lists hold,
for each, a shape that is ragged in rows and in tokens and ends in a K stage
that is not full (a stage of two blocks over rows of an even number always
is); test_lists_hold_every_tile asks the library for the choices and checks
that.  Products are exact and sums are f32, so outputs lie within
1e-5 of max|Y| (2048 columns: f32 rounding of partial sums, 64 blocks x 2^-24,
is 4e-6 at worst); the GeGLU adds one f16 rounding (2^-11) of the output.
"""
import ctypes

import numpy as np
import pytest

import oracle as orc
from e4b import formats
from e4b._lib import check, lib
from e4b.kernels import MoeLayer, Q40Matrix
from tests.util import max_rel_err

pytestmark = pytest.mark.gpu


def _dense(w, rows, cols):
    return orc.q40_dequant(w).astype(np.float64).reshape(rows, cols)


def _gelu(g):
    return 0.5 * g * (1 + np.tanh(np.clip(0.7978845608028654 * (g + 0.044715 * g ** 3), -20, 20)))


# rows of an even number of blocks (64 x 1 .. 2048), then of an odd number
F32 = [(9176, 192, 639), (14280, 704, 217), (8591, 2048, 35), (14338, 384, 161), (102, 192, 3), (17554, 384, 1),
       (18046, 64, 294), (10890, 448, 260), (5833, 1600, 67), (12647, 448, 99), (8234, 192, 1), (16425, 64, 1),
       (33, 320, 1),
       (61, 384, 5), (5306, 224, 689), (5696, 2016, 65), (151, 224, 2), (312, 288, 1), (33, 64, 33), (1, 32, 1),
       (16947, 96, 162), (12724, 96, 98), (8206, 96, 1), (33, 288, 1)]
GLU = [(6717, 192, 326), (6946, 192, 165), (6714, 192, 105), (6569, 384, 97), (76, 192, 2), (152, 384, 1),
       (17266, 64, 130), (16388, 320, 129), (6281, 192, 104), (6382, 64, 99), (33, 64, 1), (33, 320, 1),
       (8744, 224, 139), (6557, 224, 100), (19, 224, 8), (33, 64, 33),
       (19705, 160, 136), (6176, 96, 97), (33, 96, 1)]
# token rows, outputs, waves and K groups of the tiles, for rows of an even
# and of an odd number of blocks
TILES = {(False, False): {(128, 256, 4, 1), (64, 128, 4, 2), (64, 64, 8, 4), (64, 64, 4, 2), (32, 64, 8, 4),
                          (32, 64, 4, 2), (32, 32, 8, 8)},
         (False, True): {(64, 128, 4, 2), (64, 64, 8, 4), (32, 64, 8, 4), (32, 32, 8, 8)},
         (True, False): {(128, 256, 8, 1), (64, 128, 8, 2), (64, 64, 8, 4), (64, 64, 4, 2), (32, 32, 4, 4),
                         (32, 32, 8, 8)},
         (True, True): {(64, 128, 8, 2), (64, 64, 4, 2), (32, 32, 4, 4)}}


def _tile(outputs, cols, m, geglu):
    t = (ctypes.c_int32 * 6)()
    check(lib.e4b_q40_gemm_tile(ctypes.c_int64(outputs), ctypes.c_int64(cols), m, int(geglu), t), "e4b_q40_gemm_tile")
    return list(t)


@pytest.mark.parametrize("geglu", [False, True])
def test_lists_hold_every_tile(geglu):
    seen = {False: set(), True: set()}
    for outputs, cols, m in GLU if geglu else F32:
        nb = cols // 32
        tok, out, waves, kg, stage, _ = _tile(outputs, cols, m, geglu)
        if outputs % out and m % tok and (nb % stage or (stage == 2 and nb % 2 == 0)):
            seen[nb % 2 == 1].add((tok, out, waves, kg))
    for odd in (False, True):
        assert seen[odd] == TILES[geglu, odd], f"rows of an {'odd' if odd else 'even'} number of blocks"


def test_workgroups_per_cu():
    # as the kernels were compiled: 160 KB of LDS hold three tiles of 64 x 128
    # (50 KB; 162 registers allow three waves a SIMD), and of the tile of
    # eight K groups two where rows have an odd number of blocks (no staged
    # scales: 80 KB), else one
    assert _tile(10890, 448, 260, False)[:1] + _tile(10890, 448, 260, False)[5:] == [64, 3]
    assert _tile(33, 288, 1, False)[3:] == [8, 16, 2]
    assert _tile(33, 320, 1, False)[3:] == [8, 16, 1]


@pytest.mark.parametrize("rows,cols,m", F32)
def test_f32_tiles(rows, cols, m):
    w = formats.synth_q40(rows + cols + m, rows, cols, 0.02)
    x = formats.synth_normal(rows + m, m * cols).reshape(m, cols).astype(np.float16)
    got = Q40Matrix(w, rows, cols).gemm(x)
    assert max_rel_err(got, x.astype(np.float64) @ _dense(w, rows, cols).T) < 1e-5


@pytest.mark.parametrize("ff,cols,m", GLU)
def test_geglu_tiles(ff, cols, m):
    w = formats.synth_q40(ff + cols + m, 2 * ff, cols, 0.02)
    x = formats.synth_normal(ff + m, m * cols).reshape(m, cols).astype(np.float16)
    got = Q40Matrix(w, 2 * ff, cols).gemm_geglu(x).astype(np.float64)
    y = x.astype(np.float64) @ _dense(w, 2 * ff, cols).T
    want = _gelu(y[:, :ff]) * y[:, ff:]
    assert np.max(np.abs(got - want) - (2.0 ** -11 * np.abs(want) + 1e-5 * np.abs(want).max())) <= 0


def test_non_finite_token_stays_in_its_row():
    # the last K stage of 7 blocks is completed with zeros, not with another
    # block's activations: an infinity there reaches its own token only, and
    # as the sum it is (weights of one sign: +inf, not NaN)
    rows, cols, m = 70, 224, 40
    w = formats.synth_q40(5, rows, cols, 0.02).reshape(-1, 18)
    w[:, 2:] = (w[:, 2:] & 0x77) | 0x88
    w[:, 2:] |= 0x11  # nibbles 9..15: every weight positive
    x = formats.synth_normal(6, m * cols).reshape(m, cols).astype(np.float16)
    x[17, cols - 1] = np.inf
    got = Q40Matrix(w.reshape(-1), rows, cols).gemm(x)
    assert np.all(got[17] == np.inf)
    x[17, cols - 1] = 0
    rest = np.delete(np.arange(m), 17)
    ref = x.astype(np.float64) @ _dense(w.reshape(-1), rows, cols).T
    assert max_rel_err(got[rest], ref[rest]) < 1e-5


@pytest.mark.parametrize("m", [31, 65, 130, 300])
def test_grouped_tiles(m):
    # 9 experts, top 8: nearly every token reaches every expert, so a run of
    # draws is cut into tiles of 64 with a remainder above and below 32 rows;
    # expert FFN 96 = 3 blocks (odd), dense FFN 160
    H, E, FF, FF2 = 512, 9, 96, 160
    rng = np.random.default_rng(m)
    q = lambda r, c, s: formats.synth_q40(s, r, c, 0.02)  # noqa: E731
    vec = lambda: (1 + 0.1 * rng.standard_normal(H)).astype(np.float32)  # noqa: E731
    t = {"ffn_norm": vec(), "router_scale": vec(), "pre_ffw2": vec(), "post_ffw1": vec(), "post_ffw2": vec(),
         "post_ffw": vec(), "pes": (1 + 0.2 * rng.standard_normal(E)).astype(np.float32),
         "router_w": formats.synth_normal(3, E * H, 0.0, 0.02).reshape(E, H), "dense_gate": q(FF2, H, 1),
         "dense_up": q(FF2, H, 2), "dense_down": q(H, FF2, 3), "exp_gate_up": q(E * 2 * FF, H, 4),
         "exp_down": q(E * H, FF, 5)}
    h = formats.synth_normal(m, m * H).reshape(m, H)
    got = MoeLayer(H, E, FF, FF2, t).prefill(h)
    ref = dict(t, hidden=H, n_experts=E, top_k=8, expert_ffn=FF, dense_ffn=FF2)
    for i in sorted({0, 1, m // 2, m - 2, m - 1}):
        idx, wts, dense, moe, hout = orc.moe_ffn(ref, h[i])
        np.testing.assert_array_equal(got["topk_idx"][i], idx)
        # f16 branch inputs and GeGLU outputs, as the half-layer stores them
        assert max_rel_err(got["dense_out"][i], dense) < 2e-3
        assert max_rel_err(got["moe_out"][i], moe) < 2e-3
        assert max_rel_err(got["h_out"][i], hout) < 1e-3
