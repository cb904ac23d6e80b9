"""Decode steps whose attention launch also takes a second mixer's recurrence and, by the last of a sequence's workgroups, its gated norm (grouped.h
grouped_short_kernel): the bits of the launches of their own."""
import numpy as np
import pytest

import medulorn_models as MM
from layered_helpers import build, err

pytestmark = pytest.mark.gpu
rot = MM.rot
LAYERS = {      # key and value widths of the recurrence: what a thread's eight rows hold at most, ragged rows and columns, one head, more heads than attention
    "128x128": dict(heads=4, kv_heads=2, dim=128, vdim=128, window=65, keep=3, turn=rot(128), heads2=5, dim2=128, vdim2=128),
    "20x32": dict(heads=4, kv_heads=2, dim=64, vdim=64, window=None, turn=rot(64), heads2=3, dim2=20, vdim2=32),
    "one-head": dict(heads=4, kv_heads=4, dim=64, vdim=32, window=70, turn=rot(64), heads2=1, dim2=64, vdim2=52),
    "many-heads": dict(heads=2, kv_heads=1, dim=64, vdim=128, window=None, turn=rot(64), heads2=24, dim2=16, vdim2=16),
    "256x64": dict(heads=4, kv_heads=2, dim=128, vdim=64, window=None, turn=rot(128), heads2=2, dim2=256, vdim2=64),
    "256x128": dict(heads=4, kv_heads=2, dim=128, vdim=128, window=None, turn=rot(128), heads2=2, dim2=256, vdim2=128),      # sixteen rows a thread: a launch of its own
}


@pytest.mark.parametrize("split", [0, 3])
@pytest.mark.parametrize("n", [1, 5, 40])
@pytest.mark.parametrize("name", list(LAYERS))
def test_same_bits(gpu, tmp_path, name, n, split):
    cfg = MM.config([MM.parallel(**LAYERS[name]), MM.parallel(**LAYERS[name])], width=128, vocab=90)
    m = build(gpu, tmp_path, cfg, MM.weights(cfg, 4), "bf16", max_seqs=40, kv_num_blocks=160)
    r = np.random.default_rng(n)
    ids, lens = list(range(n)), [1 + (37 * i) % 90 for i in range(n)]
    prompts = [r.integers(0, 90, k).tolist() for k in lens]
    lib, got = gpu.lib(), []
    for rides in (0, 2):
        old = [(key, lib.nvl_set_tuning(key, v)) for key, v in ((44, rides), (37, split))]
        for i in ids:
            m.seq_open(i)
        for a in range(0, n, 8):
            m.forward_batch(ids[a:a + 8], prompts[a:a + 8], [0] * len(ids[a:a + 8]), want_logits=False)
        got.append(np.stack([m.forward_batch(ids, [[(5 * i + j) % 90] for i in ids], [k + j for k in lens])[0] for j in range(6)]))      # (replays from the third)
        for i in ids:
            m.seq_close(i)
        for key, v in old:
            lib.nvl_set_tuning(key, v)
    m.close()
    assert np.isfinite(got[0]).all() and np.array_equal(got[0], got[1])


@pytest.mark.parametrize("wide", [dict(dim=64, vdim=272, turn=rot(64)), dict(dim=320, vdim=64, turn=rot(64))], ids=["values-272", "keys-320"])
@pytest.mark.parametrize("at", [0, 1])                      # the wide layer in front and behind
def test_beside_a_wider_layer(gpu, tmp_path, wide, at):
    """Another layer's heads fit no instance: this one's recurrence rides all the same (tickets of its own), and the keys of a long context are split (2100 keys: two
    parts).  Steps against the fp32 mode, and the same bits as the launches of their own."""
    layers = [MM.parallel(**LAYERS["128x128"] | dict(window=None))]
    layers.insert(at, MM.attention(heads=2, kv_heads=1, chunk=None, **wide))
    cfg = MM.config(layers, width=128, vocab=90)
    w = MM.weights(cfg, 4)
    r, got = np.random.default_rng(at), {}
    prompts = [r.integers(0, 90, k).tolist() for k in (2100, 40)]
    for mode, rides in (("f32", 1), ("bf16", 1), ("bf16", 0)):
        old = gpu.lib().nvl_set_tuning(44, rides)
        m = build(gpu, tmp_path, cfg, w, mode, max_seqs=2, max_seq_len=2112, max_batch_tokens=2144, kv_num_blocks=72)
        for i in (0, 1):
            m.seq_open(i)
        m.forward_batch([0, 1], prompts, [0, 0], want_logits=False)
        got[mode, rides] = np.stack([m.forward_batch([0, 1], [[7 + j], [3 + j]], [2100 + j, 40 + j])[0] for j in range(4)])
        m.close()
        gpu.lib().nvl_set_tuning(44, old)
    assert np.array_equal(got["bf16", 1], got["bf16", 0])
    assert err(got["bf16", 1], got["f32", 1]) < 0.06            # two bf16 layers, the worst row (0.03 a layer in the other tests of these models)


def test_profile_counts_the_recurrence(gpu, tmp_path):
    """Work and traffic of a step's launches are the same whether the recurrence rides or not."""
    cfg = MM.config([MM.parallel(**LAYERS["128x128"])], width=128, vocab=90)
    m = build(gpu, tmp_path, cfg, MM.weights(cfg, 4), "bf16", max_seqs=3)
    for i in range(3):
        m.seq_open(i)
    m.forward_batch([0, 1, 2], [[3, 4, 5]] * 3, [0, 0, 0], want_logits=False)
    total = []
    for rides in (0, 2):
        old = gpu.lib().nvl_set_tuning(44, rides)
        m.reset_stats()
        m.set_profile(True)
        m.forward_batch([0, 1, 2], [[7]] * 3, [3 + len(total)] * 3, want_logits=False)
        m.set_profile(False)
        gpu.lib().nvl_set_tuning(44, old)
        ks = [k for k in m.kernel_stats() if k["site"] in ("attention", "lightning_scan") and k["launches"]]
        assert len(ks) == (1 if rides else 2)
        total.append((sum(k["flops"] for k in ks), sum(k["bytes"] for k in ks)))
    m.close()
    state = 2 * 3 * 5 * 128 * 128 * 4                           # every sequence's five states, in and out
    assert total[0][1] > state and abs(total[1][0] / total[0][0] - 1) < 0.05 and abs(total[1][1] / total[0][1] - 1) < 0.05      # (a key more in the second step)
