"""128x128 tiles with a ring of K tiles of 32: fewer of them than the ring holds, even and odd numbers, ragged rows and columns."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu
TOL = 1.5e-2


@pytest.mark.parametrize("k", [64, 128, 192, 256, 320, 2048])          # 2, 4, 6, 8, 10 and 64 K tiles; the ring holds 4
@pytest.mark.parametrize("m,n", [(65, 130), (128, 128), (129, 384), (700, 96), (1000, 1000),      # 64x128 tiles
                                 (1500, 1601), (2049, 1030)])                                       # 312 and 297 of those: 128x128, on eight waves
def test_products_are_exact(gpu, m, n, k):
    """Small whole numbers: every sum is exact in fp32, whatever its order."""
    r = np.random.default_rng(m + n + k)
    a, b = (r.integers(-4, 5, s).astype(np.float32) for s in ((m, k), (k, n)))
    old = gpu.lib().nvl_set_tuning(0, 1)
    try:
        got = gpu.ops.mat_mul(a, b, precision="bf16")
    finally:
        gpu.lib().nvl_set_tuning(0, old)
    assert np.array_equal(got, (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32))


@pytest.mark.parametrize("hidden", [64, 128, 192, 256, 320])           # 2 .. 10 K tiles
def test_few_tiles_of_k_on_four_waves(gpu, hidden):
    """Gate | up columns of a prompt on 660 tiles of 128x128, whose gated results are bf16: four waves, against the fp32 mode."""
    cfg = gpu.synth.tiny_config("llama", hidden=hidden, num_heads=hidden // 64, num_kv_heads=hidden // 64, head_dim=64, ffn_dim=8448, num_layers=2, max_seq_len=640)
    w = gpu.synth.make_weights(cfg, seed=4, scale=0.03)
    tokens = np.random.default_rng(hidden).integers(0, cfg["vocab_size"], 601).tolist()
    got = []
    old = gpu.lib().nvl_set_tuning(0, 1)
    try:
        for precision in ("f32", "bf16"):
            m = gpu.HipTransformerModel(cfg, w, precision=precision, max_seqs=1, max_batch_tokens=640)
            m.seq_reset(0)
            got.append(m.forward_batch([0], [tokens], [0], all_logits=True)[0])
            m.close()
    finally:
        gpu.lib().nvl_set_tuning(0, old)
    assert rel_err(got[1], got[0]) <= TOL


# 2048 columns: two slices of 33 K tiles of FFN-down's 66, up to 200 rows the LDS-ring kernel instead; 512: four of 17, 17, 16 and 16
@pytest.mark.parametrize("hidden,rows", [(2048, 70), (2048, 200), (2048, 513), (2048, 900), (512, 513), (512, 900)])
def test_slices_of_odd_numbers_of_tiles(gpu, hidden, rows):
    """A prompt whose residual projections run in slices that the norm behind them sums, against the fp32 mode."""
    cfg = gpu.synth.tiny_config("llama", hidden=hidden, num_heads=8, num_kv_heads=8, head_dim=64, ffn_dim=2112, num_layers=2, max_seq_len=1024)
    w = gpu.synth.make_weights(cfg, seed=4, scale=0.03)
    tokens = np.random.default_rng(rows).integers(0, cfg["vocab_size"], rows).tolist()
    got = []
    for precision in ("f32", "bf16"):
        m = gpu.HipTransformerModel(cfg, w, precision=precision, max_seqs=1, max_batch_tokens=1024)
        m.seq_reset(0)
        got.append(m.forward_batch([0], [tokens], [0], all_logits=True)[0])
        if precision == "bf16":
            m.seq_reset(0)
            assert np.array_equal(got[1], m.forward_batch([0], [tokens], [0], all_logits=True)[0])
        m.close()
    assert rel_err(got[1], got[0]) <= TOL


@pytest.mark.parametrize("n", [1, 100, 256, 257])          # 256 tokens x 8 of 32 experts: 64 rows an expert, the last prompt that takes 128-row tiles
def test_experts_of_few_rows(gpu, n):
    """The experts' products of a short prompt against forced 256-row tiles (key 17), which add up in the same order."""
    import torch
    from bench import gen_weights_on_device
    cfg = dict(gpu.synth.FULL_CONFIGS["granite-3.0-1b-a400m"], num_layers=2, vocab_size=1000)
    m = gpu.HipTransformerModel(cfg, None, precision="bf16", max_seqs=2, max_batch_tokens=320)
    gen_weights_on_device(gpu, cfg, m, torch, torch.device("cuda", 0), keep_host=False)
    m.finalize()
    prompts = [np.random.default_rng(n).integers(0, 1000, k).tolist() for k in (n, 66)][: 2 if n < 200 else 1]
    ids, got = list(range(len(prompts))), []
    for rows in (0, 256):
        old = gpu.lib().nvl_set_tuning(17, rows)
        try:
            for i in ids:
                m.seq_reset(i)
            got.append(m.forward_batch(ids, prompts, [0] * len(ids))[0])
        finally:
            gpu.lib().nvl_set_tuning(17, old)
    m.close()
    assert rel_err(got[0], got[1]) <= TOL


@pytest.mark.parametrize("tile", [1, 2, 3, 5])          # the ring, 256x128, lock-step 256x256, ping-pong
@pytest.mark.parametrize("family,hd", [("llama", 64), ("llama", 128), ("gpt2", 64)])      # angles; biases
@pytest.mark.parametrize("rows", [129, 300, 515])
def test_epilogues_of_ragged_rows(gpu, tile, family, hd, rows):
    """Residuals whose old values and query / key tiles whose angles are fetched ahead of the stores before them: last tiles of 1, 44 and 3 rows, against the fp32 mode; a second
    sequence's keys in the blocks of a pool."""
    cfg = gpu.synth.tiny_config(family, hidden=576, num_heads=8, num_kv_heads=8 if family == "gpt2" else 4, head_dim=hd, ffn_dim=1152, num_layers=2, max_seq_len=640)
    w = gpu.synth.make_weights(cfg, seed=4, scale=0.03)
    g = np.random.default_rng(rows)
    tokens = [g.integers(0, cfg["vocab_size"], n).tolist() for n in (rows - 70, 70)]
    got = []
    old = gpu.lib().nvl_set_tuning(0, tile)
    try:
        for precision in ("f32", "bf16"):
            m = gpu.HipTransformerModel(cfg, w, precision=precision, max_seqs=2, max_batch_tokens=640)
            for i in (0, 1):
                m.seq_reset(i)
            out = list(m.forward_batch([0, 1], tokens, [0, 0], all_logits=True)[0])
            out.append(np.asarray(m.forward_batch([0, 1], [[3], [5]], [len(t) for t in tokens])[0]))
            got.append(np.concatenate([np.asarray(o).reshape(-1, cfg["vocab_size"]) for o in out]))
            m.close()
    finally:
        gpu.lib().nvl_set_tuning(0, old)
    assert rel_err(got[1], got[0]) <= TOL
