"""The MoE half-layer over token rows at the edges of its kernels: row counts
around the router's 2 rows a block and the grouped product's 64-row tiles,
expert counts around its 16 experts a block, hidden sizes from one piece of a
row to all twelve, odd block counts in either down projection, and draws that
all go to the same 8 experts.

Picks and weights equal the decode router's bit for bit (the same operations
in the same order).  The branch results are compared with the decode layer's:
both hold the GeGLU output in 16 bits, so a sum that differs in its last f32
bit can flip a rounding (2^-11 of one element of the down projection's input);
2e-3 of the largest result is above four such flips in a row of FF >= 32.
"""
import numpy as np
import pytest

from e4b import formats
from e4b.kernels import MoeLayer

pytestmark = pytest.mark.gpu


def _layer(H, E, FF, FF2, same):
    q = lambda r, c, s: formats.synth_q40(s, r, c, 0.02)  # noqa: E731
    v = lambda s, n=H: 1 + 0.1 * formats.synth_normal(s, n)  # noqa: E731
    w = formats.synth_normal(7, E * H).reshape(E, H) / np.sqrt(H)
    if same:  # element 0 of a row decides: the same 8 experts for every token
        w *= 1e-3
        w[:, 0] += np.linspace(-4, 4, E)
    t = {"ffn_norm": v(1), "router_scale": v(2), "pre_ffw2": v(3), "post_ffw1": v(4), "post_ffw2": v(5),
         "post_ffw": v(6), "pes": v(13, E), "router_w": w.astype(np.float32) * np.float32(np.sqrt(H)),
         "dense_gate": q(FF2, H, 8), "dense_up": q(FF2, H, 9), "dense_down": q(H, FF2, 10),
         "exp_gate_up": q(E * 2 * FF, H, 11), "exp_down": q(E * H, FF, 12)}
    return MoeLayer(H, E, FF, FF2, t)


@pytest.mark.parametrize("H,E,FF,FF2,m,same", [
    (256, 8, 32, 32, 1, False),      # one piece a row, the fewest experts, one block a down row
    (256, 17, 64, 96, 9, False),     # an expert and a token row past the block; odd dense down rows
    (512, 16, 96, 64, 8, False),     # odd expert down rows
    (1024, 61, 160, 512, 65, True),  # 65 rows of each of 8 experts: a tile and one row
    (2816, 128, 704, 2112, 7, False),
    (3072, 255, 64, 128, 33, False),  # all twelve pieces of a row
    (256, 256, 64, 2112, 1024, False),  # the most draws and experts
    (256, 128, 64, 64, 1024, True),  # 16 full tiles of each of 8 experts
])
def test_rows_match_decode(H, E, FF, FF2, m, same):
    L = _layer(H, E, FF, FF2, same)
    h = formats.synth_normal(31, m * H).reshape(m, H)
    if same:
        h[:, 0] = 3.0 + 0.01 * np.arange(m)
    got = L.prefill(h)
    if same:
        assert len(np.unique(got["topk_idx"])) == 8
    rows = range(m) if m <= 65 else [0, 1, 7, 8, 63, 64, 500, m - 9, m - 1]
    for r in rows:
        want = L.forward(h[r])
        np.testing.assert_array_equal(got["topk_idx"][r], want["topk_idx"], err_msg=f"row {r}")
        np.testing.assert_array_equal(got["topk_w"][r], L.router_top8(h[r])[1], err_msg=f"row {r}")
        for n in ("dense_out", "moe_out", "h_out"):
            err = np.abs(got[n][r].astype(np.float64) - want[n]).max() / np.abs(want[n]).max()
            assert err < 2e-3, f"row {r} {n}: {err:.2e}"
