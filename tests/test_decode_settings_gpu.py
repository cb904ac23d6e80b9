"""Decode steps under the documented settings that change which projections a deferred norm rides on (nvl_set_tuning keys 2, 3, 27): the same
numbers as the fp32 mode whatever the form."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu
TOL = 1.5e-2

CONFIGS = {
    "llama": ("llama", dict(num_layers=3)),
    "moe": ("granite_moe", dict(num_layers=3, embedding_multiplier=1.0, residual_multiplier=1.0, num_experts_per_tok=8)),      # all eight: no near tie between experts
    "hybrid": ("granite_hybrid", dict(hidden=256, mamba_num_heads=16, mamba_head_dim=32, embedding_multiplier=1.0, residual_multiplier=1.0)),      # 16 heads: the one-launch Mamba-2 step
}


@pytest.mark.parametrize("name", list(CONFIGS))
@pytest.mark.parametrize("n", [1, 16, 17, 40])                  # half tiles of 8 columns up to 16 rows, whole tiles above
def test_settings_keep_the_numbers(gpu, name, n):
    family, over = CONFIGS[name]
    cfg = gpu.synth.tiny_config(family, **over)
    w = gpu.synth.make_weights(cfg, seed=31, scale=0.05)
    r = np.random.default_rng(n)
    prompts = [r.integers(0, cfg["vocab_size"], 2 + i % 3).tolist() for i in range(n)]
    steps = r.integers(0, cfg["vocab_size"], (2, n)).tolist()
    ids = list(range(n))

    def logits(m):
        for i in ids:
            m.seq_reset(i)
        m.forward_batch(ids, prompts, [0] * n, want_logits=False)
        return np.stack([m.forward_batch(ids, [[t] for t in s], [len(p) + j for p in prompts])[0] for j, s in enumerate(steps)])

    m = gpu.HipTransformerModel(cfg, w, precision="f32", max_seqs=n, max_batch_tokens=256)
    want = logits(m)
    m.close()
    m = gpu.HipTransformerModel(cfg, w, precision="bf16", max_seqs=n, max_batch_tokens=256)
    errs = {}
    for key, value in ((3, 1), (3, 0), (3, 2), (3, 3), (2, 1), (2, 2), (2, 4), (27, 0)):
        old = gpu.lib().nvl_set_tuning(key, value)
        try:
            errs[key, value] = rel_err(logits(m), want)
        finally:
            gpu.lib().nvl_set_tuning(key, old)
    m.close()
    assert max(errs.values()) <= TOL, errs


@pytest.mark.parametrize("n,ffn", [(8, 4096), (8, 8256), (40, 2048), (40, 4160)])      # up to and beyond 32 blocks of an expert's k-steps a wave
def test_wide_experts(gpu, n, ffn):
    """The experts' down projection of a decode batch, an expert of any width a wave, against experts sorted into grouped products (key 22 = 0)."""
    cfg = gpu.synth.tiny_config("granite_moe", ffn_dim=ffn, num_experts=4, num_layers=2)
    m = gpu.HipTransformerModel(cfg, gpu.synth.make_weights(cfg, seed=7, scale=0.05), precision="bf16", max_seqs=n, max_batch_tokens=128)
    ids, got = list(range(n)), []
    for dense in (1, 0):
        old = gpu.lib().nvl_set_tuning(22, dense)
        try:
            for i in ids:
                m.seq_reset(i)
            m.forward_batch(ids, [[3 + i] for i in ids], [0] * n, want_logits=False)
            got.append(m.forward_batch(ids, [[9 + i] for i in ids], [1] * n)[0])
        finally:
            gpu.lib().nvl_set_tuning(22, old)
    m.close()
    assert rel_err(got[0], got[1]) <= TOL
