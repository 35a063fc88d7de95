"""The batched GeGLU (e4b_k_q40_gemm_geglu) over the whole range of its gate.

gelu_tanh clamps the tanh argument t to +-20 and tanh(-20) is -1 in f32, so
from there on the result is zero whatever the gate and the up value are, as
the decode kernel gives it; above, the result is g u / (1 + e^-2t).  One block
of equal weights a row and equal activations make gate and up exact powers of
two times small numbers.

Tolerance: t = 0.798 (g + 0.0447 g^3) carries a few f32 roundings, at most 4 x
2^-24 x 20 = 5e-6, which e^-2t doubles and the exponential's own error (an ulp
and 2^-24 x 40 of its argument) adds to: 2e-5 of the value covers them.  The
f16 result rounds by 2^-11 of it, or by 2^-25 where it is subnormal.
"""
import numpy as np
import pytest

from e4b import formats
from e4b.kernels import Q40Matrix

pytestmark = pytest.mark.gpu


def _rows(scales, nibble):
    """one q4_0 block a row: every weight (nibble - 8) * scale"""
    b = np.full((len(scales), 18), nibble * 17, np.uint8)
    b[:, :2] = np.asarray(scales, np.float16).reshape(-1, 1).view(np.uint8)
    return b


@pytest.mark.parametrize("m", [1, 40, 130])  # tiles of one, two and four tokens a wave
@pytest.mark.parametrize("up", [2.0 ** -20, 1.0, 2.0 ** 15])
def test_negative_gates(m, up):
    ff, cols = 416, 32
    gate = np.float16(np.geomspace(2.0 ** -16, 60000.0, ff))
    w = np.concatenate([_rows(gate, 7), _rows(np.full(ff, up), 9)])
    amp = 2.0 ** np.arange(-4, 6)[np.arange(m) % 10]  # of a token's activations
    x = np.repeat(amp[:, None], cols, 1).astype(np.float16)
    got = Q40Matrix(w.reshape(-1), 2 * ff, cols).gemm_geglu(x).astype(np.float64)
    g = -32.0 * amp[:, None] * gate.astype(np.float64)
    u = 32.0 * amp[:, None] * up
    t = 0.7978845608028654 * (g + 0.044715 * g ** 3)
    want = np.where(t > -20, g * u / (1 + np.exp(-2 * np.maximum(t, -20))), 0.0)
    assert (t < -20).sum() > ff // 4 and (t > -9).sum() > ff // 4
    sure = np.abs(t + 20) > 1e-4  # on either side of the clamp
    lim = 65504.0
    far = np.abs(want) > lim  # overflows to an infinity
    assert np.all(np.isinf(got[far & (np.abs(want) > 65520)]))
    err = np.abs(got - want) - ((2.0 ** -11 + 2e-5) * np.abs(want) + 2.0 ** -25)
    assert err[sure & ~far].max() <= 0
    assert np.all(got[t < -20.001] == 0)


def test_infinite_and_nan_tokens_stay_in_their_rows():
    ff, cols, m = 96, 64, 37
    w = formats.synth_q40(3, 2 * ff, cols, 0.02)
    x = formats.synth_normal(4, m * cols).reshape(m, cols).astype(np.float16)
    M = Q40Matrix(w, 2 * ff, cols)
    want = M.gemm_geglu(x)
    x[5], x[33, 7] = np.inf, np.nan
    got = M.gemm_geglu(x)
    rest = np.delete(np.arange(m), [5, 33])
    np.testing.assert_array_equal(got[rest].view(np.uint16), want[rest].view(np.uint16))
    assert np.all(np.isnan(got[33]))
    assert not np.any(np.isfinite(got[5]) & (got[5] != 0))
