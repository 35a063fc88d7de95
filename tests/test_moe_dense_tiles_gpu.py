"""The MoE half-layer over m tokens: a row does not depend on the others.

Expert runs and the dense branch are cut into tiles of 64 or 32 rows by how
many tokens there are, and either matrix may have rows of an odd number of
blocks; every tile sums K in the same order, so each row's results are, bit
for bit, those of a call with another number of tokens.  Row counts lie
around the tiles' edges, block counts are even and odd in either matrix.
The rows themselves are compared with the decode layer (2e-3 of the largest
result: four flipped 16-bit roundings of the GeGLU outputs, 2^-11 each).
"""
import numpy as np
import pytest

from e4b import formats
from e4b.kernels import MoeLayer

pytestmark = pytest.mark.gpu

H, E = 512, 9  # 9 experts, top 8: nearly every token reaches every expert


def _layer(FF, FF2):
    q = lambda r, c, s: formats.synth_q40(s, r, c, 0.02)  # noqa: E731
    v = lambda s, n=H: 1 + 0.1 * formats.synth_normal(s, n)  # noqa: E731
    t = {"ffn_norm": v(1), "router_scale": v(2), "pre_ffw2": v(3), "post_ffw1": v(4), "post_ffw2": v(5),
         "post_ffw": v(6), "pes": v(13, E), "router_w": formats.synth_normal(7, E * H).reshape(E, H),
         "dense_gate": q(FF2, H, 8), "dense_up": q(FF2, H, 9), "dense_down": q(H, FF2, 10),
         "exp_gate_up": q(E * 2 * FF, H, 11), "exp_down": q(E * H, FF, 12)}
    return MoeLayer(H, E, FF, FF2, t)


@pytest.mark.parametrize("ff,ff2", [(128, 160), (96, 192), (96, 160), (64, 192)])
def test_rows_do_not_depend_on_their_number(ff, ff2):
    layer = _layer(ff, ff2)
    h = formats.synth_normal(21, 200 * H).reshape(200, H)
    want = layer.prefill(h)
    for m in (1, 31, 32, 33, 63, 64, 65, 96, 97, 128, 129):
        got = layer.prefill(h[:m])
        for n in ("topk_idx", "topk_w", "dense_out", "moe_out", "h_out"):
            np.testing.assert_array_equal(got[n], want[n][:m], err_msg=f"{n} of {m} tokens")
    for r in (0, 31, 32, 63, 64, 128, 199):
        one = layer.forward(h[r])
        for n in ("dense_out", "moe_out", "h_out"):
            assert np.abs(want[n][r].astype(np.float64) - one[n]).max() < 2e-3 * np.abs(one[n]).max(), f"row {r} {n}"
