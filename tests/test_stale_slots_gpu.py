"""What a sequence left in the cache is nothing to the next one: a sequence whose keys, values and states are all NaN goes, the same slot or blocks serve
another, and that one's logits are bit for bit what they were before.  Every attention kernel of every family; lengths at which the last tile of 64 keys holds
one key, is full, and lies in between; decode steps whole and dealt over workgroups.  And a sequence of NaN beside another in one call."""
import numpy as np
import pytest

import lufazen_models as LM
import medulorn_models as MM
import potuzen_models as PM
from layered_helpers import build

pytestmark = pytest.mark.gpu
NAN = 7                    # the token whose embedding is NaN
LENGTHS = [1, 33, 64, 65, 130, 300]


def run(m, tokens, steps, reset):
    """Logits of a prompt and of single tokens behind it, without the NaN token's column (tied heads)."""
    reset(0)
    n = len(tokens) - steps
    out = [m.forward_batch([0], [tokens[:n]], [0])[0]] + [m.forward_batch([0], [[t]], [n + i])[0] for i, t in enumerate(tokens[n:])]
    return np.delete(np.concatenate([np.array(x) for x in out]), NAN, axis=1)


def check(m, vocab, reset, settings=((),)):
    r = np.random.default_rng(5)
    lib = m.lib
    for n in LENGTHS:
        tokens = r.integers(NAN + 1, vocab, n + 2).tolist()
        for setting in settings:
            old = [(k, lib.nvl_set_tuning(k, v)) for k, v in setting]
            try:
                want = run(m, tokens, 2, reset)
                assert np.isfinite(want).all(), (n, setting)
                reset(0)
                left = m.forward_batch([0], [[NAN] * (min(n + 70, 370))], [0])[0]
                assert np.isnan(left).all()
                assert np.array_equal(run(m, tokens, 2, reset), want), (n, setting)
            finally:
                for k, v in old:
                    lib.nvl_set_tuning(k, v)
        if n > 1:                                          # beside one of NaN
            reset(0); reset(1)
            pair = m.forward_batch([0, 1], [tokens, [NAN] * 3], [0, 0])[0][0]
            again = m.forward_batch([0, 1], [[9], [NAN]], [n + 2, 3])[0][0]
            reset(0); reset(1)
            other = m.forward_batch([0, 1], [tokens, [11] * 3], [0, 0])[0][0]
            step = m.forward_batch([0, 1], [[9], [11]], [n + 2, 3])[0][0]
            for a, b in ((pair, other), (again, step)):
                a, b = np.delete(a, NAN), np.delete(b, NAN)
                assert np.isfinite(a).all() and np.abs(a - b).max() <= 1e-2 * np.abs(b).max(), n
    m.close()


@pytest.mark.parametrize("precision", ["f32", "bf16"])
@pytest.mark.parametrize("family,over", [("gpt2", {}), ("llama", {}), ("llama", dict(head_dim=128, hidden=512)), ("falcon", {}), ("granite_moe", {}), ("granite_hybrid", {})])
def test_plain_models(gpu, family, over, precision):
    cfg = gpu.synth.tiny_config(family, max_seq_len=512, **over)
    w = gpu.synth.make_weights(cfg, seed=7, scale=0.05)
    w["tok_emb", 0] = w["tok_emb", 0].copy()
    w["tok_emb", 0][NAN] = np.nan
    m = gpu.HipTransformerModel(cfg, w, precision=precision, max_seqs=2, max_batch_tokens=512)
    # keys 10: rows of a prefill workgroup, 15 and 25: waves of a decode workgroup and rounds of tiles each of several has, 18: short prompts' query / key / value form
    check(m, cfg["vocab_size"], m.seq_reset, ((),) if precision == "f32" else ((), ((10, 0), (15, 2), (25, 2)), ((10, 2), (15, 4), (25, 0)), ((10, 3), (15, 8), (25, 2), (18, 64))))


LAYERS = {
    "latent-64": lambda: LM.config([LM.latent(heads=6, dim=64, rot=64, vdim=64, q_rank=96, kv_rank=64)], width=128, vocab=90), "latent-128+64": lambda: LM.config([LM.latent(heads=4, dim=128, rot=64, vdim=128, q_rank=192, kv_rank=512)], width=256, vocab=90),
    "latent-wide": lambda: LM.config([LM.latent(heads=2, dim=100, rot=60, vdim=200)], width=64, vocab=90), "latent-big-heads": lambda: LM.config([LM.latent(heads=2, dim=272, rot=64, vdim=264, scale=0.04)], width=64, vocab=90),
    "delta": lambda: LM.config([LM.delta(heads=4, kv_heads=2, dim=64, vdim=64)], width=128, vocab=90), "delta-odd": lambda: LM.config([LM.delta()], width=96, vocab=90),
    "attention": lambda: MM.config([MM.attention(chunk=None)], width=96, vocab=90), "attention-128": lambda: MM.config([MM.attention(heads=4, kv_heads=2, dim=128, vdim=128, chunk=None, turn=MM.rot(64))], width=128, vocab=90),
    "chunks": lambda: MM.config([MM.attention(chunk=50)], width=96, vocab=90), "windows": lambda: MM.config([MM.parallel()], width=96, vocab=90), "many-heads": lambda: MM.config([MM.attention(heads=34, kv_heads=1, dim=16, vdim=8, chunk=None, turn=MM.rot(8))], width=96, vocab=90),
    "big-heads": lambda: MM.config([MM.attention(heads=2, kv_heads=1, dim=272, vdim=264, scale=0.05, chunk=None, turn=MM.rot(136))], width=64, vocab=90),
}


@pytest.mark.parametrize("precision", ["f32", "bf16"])
@pytest.mark.parametrize("name", list(LAYERS))
def test_layers(gpu, tmp_path, name, precision):
    cfg = LAYERS[name]()
    w = (LM if cfg["architecture"] == "Lufazen" else MM).weights(cfg, 7)
    w["embed"] = w["embed"].copy()
    w["embed"][NAN] = np.nan
    m = build(gpu, tmp_path, cfg, w, precision, max_seqs=2, kv_num_blocks=8)
    check(m, 90, m.seq_reset, ((), ((37, 3),)))
