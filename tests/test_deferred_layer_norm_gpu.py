"""Layer norms that the projection in front of them carries (batches of up to 64 rows; nvl_set_tuning key 3 = 0: norm launches), against the fp32 mode."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu
TOL = 1.5e-2


@pytest.mark.parametrize("hidden", [256, 768, 1280])      # 16, 48 and 80 tiles of 16 columns: one and two groups of sums a lane
@pytest.mark.parametrize("n", [1, 3, 16, 17, 33, 64])     # half tiles up to 16 rows; one to four row tiles
@pytest.mark.parametrize("offset", [0.0, 12.0])           # rows whose mean is far from zero, some 12 deviations
def test_carried_norms(gpu, hidden, n, offset):
    cfg = gpu.synth.tiny_config("gpt2", hidden=hidden, num_heads=hidden // 64, num_kv_heads=hidden // 64, head_dim=64, ffn_dim=2 * hidden + 64, num_layers=3, max_seq_len=64)
    w = gpu.synth.make_weights(cfg, seed=5, scale=0.05)
    r = np.random.default_rng(n)
    if offset:
        w["pos_emb", 0] = gpu.synth.round_bf16((w["pos_emb", 0] + offset * np.std(w["tok_emb", 0])).astype(np.float32))
    ids = list(range(n))
    prompts = [r.integers(0, cfg["vocab_size"], 1 + (i == 0) * min(5, 65 - n)).tolist() for i in ids]
    steps = r.integers(0, cfg["vocab_size"], (2, n)).tolist()

    def logits(m):
        for i in ids:
            m.seq_reset(i)
        out = [m.forward_batch(ids, prompts, [0] * n)[0]]
        at = [len(p) for p in prompts]
        for s in steps:
            out.append(m.forward_batch(ids, [[t] for t in s], at)[0])
            at = [a + 1 for a in at]
        return np.stack(out)

    m = gpu.HipTransformerModel(cfg, w, precision="f32", max_seqs=n, max_batch_tokens=128)
    want = logits(m)
    m.close()
    m = gpu.HipTransformerModel(cfg, w, precision="bf16", max_seqs=n, max_batch_tokens=128)
    got = logits(m)
    assert np.array_equal(got, logits(m))
    old = gpu.lib().nvl_set_tuning(3, 0)
    try:
        launches = logits(m)
    finally:
        gpu.lib().nvl_set_tuning(3, old)
    m.close()
    carried, plain = rel_err(got, want), rel_err(launches, want)
    print(f"hidden {hidden} rows {n} offset {offset}: carried {carried:.2e} launches {plain:.2e}", flush=True)
    assert carried <= TOL and plain <= TOL


def test_fused_steps(gpu):
    """Steps on the device (their first norm is the seam's) choose the tokens that single calls choose."""
    cfg = gpu.synth.tiny_config("gpt2", hidden=256, num_heads=4, num_kv_heads=4, head_dim=64, ffn_dim=512, num_layers=3, max_seq_len=64)
    w = gpu.synth.make_weights(cfg, seed=6, scale=0.05)
    m = gpu.HipTransformerModel(cfg, w, precision="bf16", max_seqs=3, max_batch_tokens=64)
    ids = [0, 1, 2]

    def prompts():
        for i in ids:
            m.seq_reset(i)
        return m.forward_batch(ids, [[3], [9, 8], [4]], [0] * 3)[1]

    fused = m.decode_greedy(ids, prompts(), 8)
    toks, single = prompts(), []
    for j in range(8):
        toks = m.forward_batch(ids, [[int(t)] for t in toks], [1 + j, 2 + j, 1 + j])[1]
        single.append(toks)
    m.close()
    assert np.array_equal(fused, np.stack(single))


@pytest.mark.parametrize("n", [1, 16, 33])              # half tiles, whole ones, several row tiles
@pytest.mark.parametrize("by", ["bias", "weights"])     # what a projection adds to its rows' means: the same for all rows, or each row's own
def test_means_that_move(gpu, by, n):
    """Every residual projection moves the means of its rows by some ten deviations.  Norm launches round the normed row to bf16 and carried norms the row
    without its mean, so both lose the same; a mean that is off by d deviations would cost sqrt(1 + d^2) times that."""
    cfg = gpu.synth.tiny_config("gpt2", hidden=768, num_heads=12, num_kv_heads=12, head_dim=64, ffn_dim=1600, num_layers=3, max_seq_len=64)
    w = gpu.synth.make_weights(cfg, seed=5, scale=0.05)
    for i in range(3):
        # (behind the first projection rows have deviations of 2 .. 5; the feed-forward's 1600 inputs sum to some 900, attention's 768 to +- 40)
        for slot, add in (("bo", 30.0), ("b2", 30.0)) if by == "bias" else (("wo", 0.75), ("w2", 0.04)):
            w[slot, i] = gpu.synth.round_bf16((w.get((slot, i), np.zeros(768)) + add).astype(np.float32))
    r = np.random.default_rng(n)
    ids, prompts = list(range(n)), [[int(t)] for t in r.integers(0, cfg["vocab_size"], n)]
    steps = r.integers(0, cfg["vocab_size"], (3, n)).tolist()

    def logits(m):
        for i in ids:
            m.seq_reset(i)
        return np.stack([m.forward_batch(ids, prompts, [0] * n)[0]] + [m.forward_batch(ids, [[t] for t in s], [at + 1] * n)[0] for at, s in enumerate(steps)])

    m = gpu.HipTransformerModel(cfg, w, precision="f32", max_seqs=n, max_batch_tokens=128)
    want = logits(m).astype(np.float64)
    m.close()
    m = gpu.HipTransformerModel(cfg, w, precision="bf16", max_seqs=n, max_batch_tokens=128)
    err = [float(np.linalg.norm(logits(m) - want) / np.linalg.norm(want))]
    old = gpu.lib().nvl_set_tuning(3, 0)
    try:
        err.append(float(np.linalg.norm(logits(m) - want) / np.linalg.norm(want)))
    finally:
        gpu.lib().nvl_set_tuning(3, old)
    m.close()
    print(f"{by} {n} rows: carried {err[0]:.2e} launches {err[1]:.2e}", flush=True)
    assert err[0] <= 1.3 * err[1]          # (the two differ by chance where they round: 1.0 +- 0.1)
