"""Prefill attention where the end of the KV ring falls inside a 32-key tile.

A tile of the kernel ends at the ring's end and the next one starts at slot 0,
so tiles are cut short there: at every offset within a tile, with rings that
are no multiple of the tile, inside a key split and in its last tile, with
one, two and four q heads per KV head.

Tolerance: the output is f16 (half an ulp of a value at most max |want|:
2^-11 = 4.9e-4 of it); K, V are f16 and the products are formed to ~2^-22, so
twice the rounding of the output bounds the rest (the oracle rounds to f16 too).
"""
import numpy as np
import pytest

import oracle as orc
from e4b.kernels import attn_prefill

pytestmark = pytest.mark.gpu
HD = 256


@pytest.mark.parametrize("gqa,kvh,slots,window,p0,m", [
    (4, 1, 45, 29, 45 * 3 - 1, 17),    # one slot before the end; one split
    (4, 1, 45, 29, 45 * 3 + 30, 16),   # 17 queries' worth of ring, cut in its middle
    (2, 2, 77, 40, 77 + 5, 38),        # 32-query tiles, the smallest ring of the chunk
    (1, 2, 101, 33, 101 * 2 - 31, 69),  # 64-query tiles, two of them
    (4, 2, 549, 513, 549 * 2 + 200, 37),  # several key splits, the end inside one
    (4, 2, 549, 513, 549 * 2 + 127, 2),   # and one key before a split's last tile
])
def test_ring_end_inside_a_tile(gqa, kvh, slots, window, p0, m):
    qh = gqa * kvh
    rng = np.random.default_rng(slots + p0)
    q = rng.standard_normal((m, qh, HD)).astype(np.float32)
    k = (0.25 * rng.standard_normal((kvh, slots, HD))).astype(np.float16)
    v = rng.standard_normal((kvh, slots, HD)).astype(np.float16)
    got = attn_prefill(q, k, v, window, p0).astype(np.float64)
    ko = np.ascontiguousarray(k.transpose(1, 0, 2)).view(np.uint16)  # the oracle's layout: [slot][kvh][HD]
    vo = np.ascontiguousarray(v.transpose(1, 0, 2)).view(np.uint16)
    for i in range(m):
        want = orc.attn_ring(q[i].ravel(), ko, vo, qh, kvh, HD, slots, window, p0 + i)
        want = want.view(np.float16).astype(np.float64)
        err = np.abs(got[i].ravel() - want.ravel()).max() / np.abs(want).max()
        assert err < 2 * 2.0 ** -11, f"query {i} (pos {p0 + i}): rel err {err:.3e}"
