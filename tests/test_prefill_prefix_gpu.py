"""What a prompt's rows have in common with those of a longer prompt that
begins alike.

The batched prefill shapes its products by the number of tokens, and with it
the order of their f32 sums: the same call repeated gives the same bits, while
rows of a common prefix agree up to that rounding, carried through the layers
(the tolerances of the engine's cache comparisons: 1e-2 of the largest and
1e-3 of the mean value).  Through the decode step
(E4B_FLAG_STEP_PREFILL) a row depends on nothing behind it, bit for bit.
"""
import numpy as np
import pytest

from e4b._lib import FLAG_STEP_PREFILL
from e4b.engine import Engine
from e4b.model import E4BConfig, a4b_config, norm_weights_random, synth_tensors

pytestmark = pytest.mark.gpu


def _e4b(**kw):
    return E4BConfig(layers=3, vocab=1000, max_seq=512, layer_global=[0, 1, 0], **kw)


def _a4b(**kw):
    # 8 experts, so that rounding cannot change the picks
    return a4b_config(layers=2, vocab=1000, max_seq=512, layer_global=[0, 1], n_experts=8, **kw)


@pytest.mark.parametrize("config", [_e4b, _a4b])
@pytest.mark.parametrize("step", [False, True])
def test_common_prefix(config, step):
    cfg = config(flags=FLAG_STEP_PREFILL) if step else config()
    eng = Engine(cfg, norm_weights_random(synth_tensors(cfg, 5), 6))
    ids = np.random.default_rng(7).integers(0, cfg.vocab, 300)

    def rows(n, keep):
        eng.reset()
        eng.prefill(ids[:n])
        return [[x[:, :keep] for x in eng.read_kv(layer)] for layer in range(cfg.layers)], eng.read_logits()

    for short, long in ((1, 37), (37, 300), (64, 65)):
        a, la = rows(short, short)
        again, lb = rows(short, short)
        b, _ = rows(long, short)
        np.testing.assert_array_equal(la, lb)
        for layer in range(cfg.layers):
            for x, y, z in zip(a[layer], again[layer], b[layer]):
                np.testing.assert_array_equal(x, y)
                if step:
                    np.testing.assert_array_equal(x, z, err_msg=f"{short} of {long} tokens, layer {layer}")
                    continue
                fx, fz = x.view(np.float16).astype(np.float64), z.view(np.float16).astype(np.float64)
                d = np.abs(fx - fz)
                assert d.max() <= 1e-2 * np.abs(fx).max(), f"{short} of {long} tokens, layer {layer} (max)"
                assert d.mean() <= 1e-3 * np.abs(fx).mean(), f"{short} of {long} tokens, layer {layer} (mean)"
