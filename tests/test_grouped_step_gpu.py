"""Decode steps of the grouped attention whose launch norms and rotates queries and keys, appends the key and carries a second mixer's gated
norm (grouped.h grouped_short_kernel, QK), against the plain restatement of the model and against launches of their own."""
import pytest

import medulorn_models as MM
from layered_helpers import build, err, feed

pytestmark = pytest.mark.gpu
BF16_LAYER = 0.03       # a single bf16 layer against the fp32 restatement, as in the other tests of these models
att, par, rot = MM.attention, MM.parallel, MM.rot

LAYERS = {
    "64-group-4": att(heads=4, kv_heads=1, dim=64, vdim=64, chunk=None, turn=rot(64)),
    "128-chunk": att(heads=6, kv_heads=2, dim=128, vdim=128, chunk=100, turn=rot(128)),
    "no-turn": att(heads=4, kv_heads=4, dim=64, vdim=32, chunk=None, turn=None),
    "group-17": att(heads=17, kv_heads=1, dim=64, vdim=32, chunk=None, turn=rot(64)),                        # a second tile of one row
    "norm-of-all": par(heads=6, kv_heads=2, dim=64, vdim=64, window=70, keep=66, turn=rot(64)),
    "norm-of-2560": par(heads=20, kv_heads=4, dim=128, vdim=40, window=None, turn=rot(128)),                 # more columns than the threads hold
    "carried-norm": par(heads=4, kv_heads=2, dim=128, vdim=128, window=65, keep=0, turn=rot(128), heads2=9, dim2=16, vdim2=128),
    "carried-odd": par(heads=4, kv_heads=2, dim=64, vdim=64, turn=rot(64), heads2=3, dim2=20, vdim2=30),     # 90 columns: a launch of its own
}


@pytest.mark.parametrize("name", list(LAYERS))
def test_steps(gpu, tmp_path, name):
    """Steps across the borders of key tiles, alone and in splits of the keys; captured passes come with the repetition."""
    cfg = MM.config([LAYERS[name]], width=128, vocab=90)
    w = MM.weights(cfg, 21)
    tok, want, _ = MM.clear_tokens(cfg, w, 190, 3)
    m = build(gpu, tmp_path, cfg, w, "bf16")
    lib, got = gpu.lib(), {}
    for i, (own, split) in enumerate(((1, 0), (0, 0), (0, 1), (0, 2), (0, 5))):
        old = [(key, lib.nvl_set_tuning(key, v)) for key, v in ((42, 1 - own), (37, split))]
        got[own, split] = feed(m, i, tok, [60] + [1] * 10 + [55] + [1] * 65)
        for key, v in old:
            lib.nvl_set_tuning(key, v)
        m.seq_close(i)
    m.close()
    for k, v in got.items():
        assert err(v, want, "bf16") < BF16_LAYER, k
