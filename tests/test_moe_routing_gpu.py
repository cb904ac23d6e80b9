"""Routing of rows that hold no numbers: every place of a token's list of experts is filled, whatever its scores are (common.h score_key), so that
such a row harms no other.  Each form of routing, prompts and decode steps."""
import numpy as np
import pytest

import bolinex_models as BM
import medulorn_models as MM
from layered_helpers import build

pytestmark = pytest.mark.gpu
BAD, GOOD = 5, 6          # tokens: the first one's embedding is infinite


def both(run):
    """The clean sequence's logits beside a bad and beside a good one (the same calls): the same bit for bit, rows being independent."""
    bad, good = run(BAD), run(GOOD)
    for b, g in zip(bad, good):
        assert not np.isfinite(b[0]).any() and np.isfinite(g).all()
        assert np.array_equal(b[1], g[1])


@pytest.mark.parametrize("precision", ["f32", "bf16"])
@pytest.mark.parametrize("n", [3, 40])                                   # 6 and 80 rows of a prompt
@pytest.mark.parametrize("settings", [{}, {31: 2}, {31: 0}, {22: 0}, {22: 0, 8: 0}])     # routing in the router's launch, apart, planned in one launch, sorted
def test_plain_models(gpu, precision, n, settings):
    cfg = gpu.synth.tiny_config("granite_moe", tied_embedding=False)
    w = gpu.synth.make_weights(cfg, seed=9, scale=0.05)
    w["tok_emb", 0][BAD] = np.inf
    r = np.random.default_rng(n)
    a, b = (r.integers(10, cfg["vocab_size"], n).tolist() for _ in range(2))

    def run(token):
        m = gpu.HipTransformerModel(cfg, w, precision=precision, max_seqs=2, max_batch_tokens=128)
        m.seq_reset(0), m.seq_reset(1)
        out = [m.forward_batch([0, 1], [a[:-1] + [token], b], [0, 0])[0], m.forward_batch([0, 1], [[token], [11]], [n, n])[0]]
        m.close()
        return out

    old = [(k, gpu.lib().nvl_set_tuning(k, v)) for k, v in settings.items()]
    try:
        both(run)
    finally:
        for k, v in old:
            gpu.lib().nvl_set_tuning(k, v)


@pytest.mark.parametrize("precision", ["f32", "bf16"])
@pytest.mark.parametrize("n", [3, 40])
@pytest.mark.parametrize("models,cfg", [(BM, BM.config([BM.attention(mlp=BM.moe())], width=96)), (BM, BM.config([BM.attention(mlp=BM.moe(72, 5, (9, 4), 12, None))], width=64)),
                                        (MM, MM.config([MM.attention(mlp=MM.moe())], width=64))], ids=["groups", "72-experts", "softmax"])
def test_lists_of_layers(gpu, tmp_path, precision, n, models, cfg):
    w = models.weights(cfg, 13)
    w["embed"][BAD] = np.inf
    r = np.random.default_rng(n)
    a, b = (r.integers(10, cfg["vocab"], n).tolist() for _ in range(2))

    def run(token):
        m = build(gpu, tmp_path, cfg, w, precision)
        m.seq_open(0), m.seq_open(1)
        out = [m.forward_batch([0, 1], [a[:-1] + [token], b], [0, 0])[0], m.forward_batch([0, 1], [[token], [11]], [n, n])[0]]
        m.close()
        return out

    both(run)
