"""Prefill attention of the A4B full layers (head dim 512, 8 q heads a KV
head) at the edges of its tiles: prompts around 16 queries, around the splits
of 128 keys, over several chunks, and long enough for splits of more than 128
keys, against the same prompts through the decode step.

Two full layers, so that the second layer's K/V rows of every token hold the
first layer's attention; 8 experts, so that rounding cannot change the picks.
Tolerance: that of the engine's cache comparisons (f16 rounding points carried
through a layer): 1e-2 of the largest and 1e-3 of the mean value.
"""
import numpy as np
import pytest

from e4b._lib import FLAG_STEP_PREFILL
from e4b.engine import Engine
from e4b.model import a4b_config, norm_weights_random, synth_tensors

pytestmark = pytest.mark.gpu

SHAPE = dict(layers=2, vocab=1000, max_seq=1536, layer_global=[1, 1], layer_kv_heads=[2, 2], n_experts=8,
             expert_ffn=64, ffn=256)


@pytest.fixture(scope="module")
def engines():
    cfg = a4b_config(**SHAPE)
    tensors = norm_weights_random(synth_tensors(cfg, 15), 16)
    return Engine(cfg, tensors), Engine(a4b_config(flags=FLAG_STEP_PREFILL, **SHAPE), tensors)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 127, 129, 257, 530, 1100])
def test_prompt_lengths(engines, n):
    ids = np.random.default_rng(n).integers(0, SHAPE["vocab"], n)
    kv = []
    for eng in engines:
        eng.reset()
        eng.prefill(ids)
        kv.append([x.view(np.float16).astype(np.float64)[:, :n] for x in eng.read_kv(1)])
    for x, y, name in zip(*kv, "kv"):
        d = np.abs(x - y)
        assert d.max() <= 1e-2 * np.abs(y).max(), f"{n} tokens: {name} (max)"
        assert d.mean() <= 1e-3 * np.abs(y).mean(), f"{n} tokens: {name} (mean)"
