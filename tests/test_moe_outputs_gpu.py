"""e4b_k_moe_prefill writes its optional results straight into the caller's
buffers or, where those cannot stand in for its scratch, copies them: both
give the same bits, in buffers at any 4-byte offset and in overlapping ones
(the later result of the argument order stays, as with copies in that order).
"""
import ctypes as C

import numpy as np
import pytest

from e4b import formats
from e4b._lib import check, lib
from e4b.device import DeviceBuffer
from e4b.kernels import MoeLayer

pytestmark = pytest.mark.gpu

H, E, FF, FF2, M = 256, 16, 64, 96, 7


def _layer():
    q = lambda r, c, s: formats.synth_q40(s, r, c, 0.02)  # noqa: E731
    v = lambda s: 1 + 0.1 * formats.synth_normal(s, H)  # noqa: E731
    t = {"ffn_norm": v(1), "router_scale": v(2), "pre_ffw2": v(3), "post_ffw1": v(4), "post_ffw2": v(5),
         "post_ffw": v(6), "pes": np.ones(E, np.float32), "router_w": formats.synth_normal(7, E * H).reshape(E, H),
         "dense_gate": q(FF2, H, 8), "dense_up": q(FF2, H, 9), "dense_down": q(H, FF2, 10),
         "exp_gate_up": q(E * 2 * FF, H, 11), "exp_down": q(E * H, FF, 12)}
    return MoeLayer(H, E, FF, FF2, t)


def _run(layer, h, ptrs):
    hd, ho = DeviceBuffer.from_array(h), DeviceBuffer(h.nbytes)
    check(lib.e4b_k_moe_prefill(C.byref(layer.w), C.c_void_p(hd.ptr), M, C.c_void_p(ho.ptr),
                                *[C.c_void_p(p) for p in ptrs], None), "e4b_k_moe_prefill")
    return ho.download(np.float32, h.size)


@pytest.mark.parametrize("off", [0, 4, 12])
def test_outputs_at_offsets(off):
    layer, h = _layer(), formats.synth_normal(20, M * H).reshape(M, H)
    want = layer.prefill(h)
    n = [M * 32, M * 32, M * H * 4, M * H * 4]
    bufs = [DeviceBuffer(k + 16) for k in n]
    hout = _run(layer, h, [b.ptr + off for b in bufs])
    got = [b.download(np.uint8, k, off) for b, k in zip(bufs, n)]
    names = ("topk_idx", "topk_w", "dense_out", "moe_out")
    np.testing.assert_array_equal(hout, want["h_out"].reshape(-1))
    for g, name in zip(got, names):
        np.testing.assert_array_equal(g, want[name].reshape(-1).view(np.uint8), err_msg=name)


def test_overlapping_outputs():
    layer, h = _layer(), formats.synth_normal(21, M * H).reshape(M, H)
    want = layer.prefill(h)
    both = DeviceBuffer(M * H * 4)
    hout = _run(layer, h, [0, 0, both.ptr, both.ptr])
    np.testing.assert_array_equal(hout, want["h_out"].reshape(-1))
    np.testing.assert_array_equal(both.download(np.float32, M * H), want["moe_out"].reshape(-1))
