"""The batched q4_0 GEMM beyond one launch and with rows of 32 MiB and more.

A launch addresses its activations by 32-bit byte offsets and its token tiles
by a 16-bit grid coordinate; more tokens go in several launches.  The counts
here pass either limit, with the last launch a ragged remainder.

Block scales of one and small whole activations: every partial sum is a whole
number below 2^24 (random signs; the widest row's sums stay near 2^14), so
results are exact in any order.
"""
import numpy as np
import pytest

from e4b.device import DeviceBuffer
from e4b.kernels import Q40Matrix

pytestmark = pytest.mark.gpu


def _weights(rng, rows, cols):
    """ggml q4_0 bytes of random nibbles under a scale of 1, and their values"""
    n = rng.integers(0, 16, (rows, cols // 32, 32), dtype=np.uint8)
    b = np.empty((rows, cols // 32, 18), np.uint8)
    b[..., :2] = np.frombuffer(np.float16(1).tobytes(), np.uint8)
    b[..., 2:] = n[..., :16] | n[..., 16:] << 4  # elements 0-15 in the low nibbles
    return b.reshape(-1), n.reshape(rows, cols).astype(np.float32) - 8


def test_tokens_past_the_grid():
    # 65535 tiles of 32 tokens and a ragged rest
    rows, cols, m = 3, 32, 65535 * 32 + 77
    rng = np.random.default_rng(1)
    w, d = _weights(rng, rows, cols)
    x = rng.integers(-8, 9, (m, cols), dtype=np.int8).astype(np.float16)
    got = Q40Matrix(w, rows, cols).gemm(x)
    np.testing.assert_array_equal(got, x.astype(np.float32) @ d.T)


@pytest.mark.parametrize("m", [
    1,
    3,
    130,  # past 4 GiB of activations: 127 rows and 3
])
def test_rows_of_32_mib(m):
    # 2^24 + 64 columns; token t is one row times -(t % 4)
    rows, cols = 2, (1 << 24) + 64
    rng = np.random.default_rng(2)
    w, d = _weights(rng, rows, cols)
    x = rng.integers(-1, 2, cols, dtype=np.int8)
    want = d.astype(np.float64) @ x
    xd, yd = DeviceBuffer(m * cols * 2), DeviceBuffer(m * rows * 4)
    for t in range(m):
        xd.upload((x * np.int8(-(t % 4))).astype(np.float16), t * cols * 2)
    Q40Matrix(w, rows, cols).gemm_dev(xd, m, yd)
    got = yd.download(np.float32, m * rows).reshape(m, rows)
    np.testing.assert_array_equal(got, -(np.arange(m) % 4)[:, None] * want[None])
    assert np.abs(want).max() > 1000
