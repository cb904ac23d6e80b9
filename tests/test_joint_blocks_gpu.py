"""Parallel blocks whose projections of one operand, and into one sum, are one matrix each, against the fp32 mode, which keeps them apart."""
import ctypes as C

import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu
TOL = 1.5e-2


@pytest.mark.parametrize("at,mult,joint", [("mqa", 0.0, True), ("mha", 0.0, True), ("mha", 0.25, True), ("gqa", 0.5, False)])      # biases with mha; joint False: two multipliers
# steps on the narrow decode form and, of 70 sequences, in 64-row groups (the wide form, the ring kernel and tiles: below); prompts of 40 and 100 rows leave
# fp32 rows of queries and keys, those of 146 .. 199 place them
@pytest.mark.parametrize("n", [1, 5, 17, 40, 70])
def test_against_fp32(gpu, at, mult, joint, n):
    kv = dict(mqa=1, mha=4, gqa=2)[at]
    cfg = gpu.synth.tiny_config("falcon", hidden=256, num_heads=4, num_kv_heads=kv, ffn_dim=4096, attention_type=at, num_layers=2, max_seq_len=256, attention_multiplier=mult,
                                residual_multiplier=mult if joint else 0.75)
    w = gpu.synth.make_weights(cfg, seed=8, scale=0.05)
    r = np.random.default_rng(n)
    ids = list(range(n))
    prompts = [r.integers(0, cfg["vocab_size"], {1: 40, 5: 96}.get(n, 130) if i == 0 else 1).tolist() for i in ids]
    steps = r.integers(0, cfg["vocab_size"], (2, n)).tolist()

    def logits(m):
        for i in ids:
            m.seq_reset(i)
        out, at_ = [m.forward_batch(ids, prompts, [0] * n)[0]], [len(p) for p in prompts]
        for s in steps:
            out.append(m.forward_batch(ids, [[t] for t in s], at_)[0])
            at_ = [a + 1 for a in at_]
        return np.stack(out)

    got = []
    for precision in ("f32", "bf16"):
        m = gpu.HipTransformerModel(cfg, w, precision=precision, max_seqs=n, max_batch_tokens=256)
        got.append(logits(m))
        if precision == "bf16":          # what stays readable behind finalize
            for slot, n_in in (("wo", 256), ("w2", 4096)):
                back = np.empty((n_in, 256), np.float32)
                gpu._lib.check(m.lib.nvl_get_weight(m.h, gpu._lib.SLOT_ID[slot], 1, back.ctypes.data_as(C.c_void_p), n_in, 256), m.h)
                assert np.array_equal(back, gpu.synth.round_bf16(w[slot, 1]))
        m.close()
    assert rel_err(got[1], got[0]) <= TOL


@pytest.fixture(scope="module")
def wide(gpu):
    """Falcon-7B's widths, one layer: [QKV | W1] is 22848 = 178.5 x 128 rows of 4544."""
    cfg = dict(gpu.synth.FULL_CONFIGS["falcon-7b"], num_layers=1, vocab_size=1000, max_seq_len=64)
    w = gpu.synth.make_weights(cfg, seed=9, scale=0.02)
    models = [gpu.HipTransformerModel(cfg, w, precision=p, max_seqs=450, max_batch_tokens=450) for p in ("f32", "bf16")]
    yield cfg, models
    for m in models:
        m.close()


@pytest.mark.parametrize("n", [5, 24, 100, 140, 450])          # steps: narrow and wide decode form, ring kernel, 128x128 and 256x256 tiles
def test_last_tiles_of_the_joint_matrix(wide, n):
    """Whole tiles reach past the matrix's last rows; the first sequence's prompt of 40 tokens leaves fp32 rows of queries and keys too."""
    cfg, models = wide
    r = np.random.default_rng(n)
    ids, first = list(range(n)), r.integers(0, cfg["vocab_size"], 40).tolist()
    tokens, steps = r.integers(0, cfg["vocab_size"], n).tolist(), r.integers(0, cfg["vocab_size"], n).tolist()
    got = []
    for m in models:
        for i in ids:
            m.seq_reset(i)
        out = [m.forward_batch([0], [first], [0])[0], m.forward_batch(ids, [[t] for t in tokens], [40] + [0] * (n - 1))[0], m.forward_batch(ids, [[t] for t in steps], [41] + [1] * (n - 1))[0]]
        got.append(np.concatenate(out))
    assert rel_err(got[1], got[0]) <= TOL


def test_workspace_holds_attention_once(gpu):
    """Attention writes beside the feed-forward's columns: as much memory as blocks whose projections are apart (two multipliers) take, not 64 MiB more."""
    import torch
    used = []
    for residual in (0.25, 0.75, 0.25):          # (the first one is where the library's own first allocations go)
        cfg = gpu.synth.tiny_config("falcon", hidden=256, num_heads=8, num_kv_heads=2, head_dim=64, ffn_dim=2048, attention_type="gqa", num_layers=1, attention_multiplier=0.25, residual_multiplier=residual)
        w = gpu.synth.make_weights(cfg, seed=8, scale=0.05)
        free = torch.cuda.mem_get_info()[0]
        m = gpu.HipTransformerModel(cfg, w, precision="bf16", max_seqs=1, max_batch_tokens=65536)
        used.append(free - torch.cuda.mem_get_info()[0])
        m.close()
    assert used[2] - used[1] < 32 << 20, used
