"""The ring of K tiles of 32 in its other forms: 256x128 tiles with six K tiles in flight, 128x128 tiles on four and on eight waves."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu
TOL = 1.5e-2            # bf16 operands, 2^-8 relative, over two layers; sums in another order


def product(gpu, tile, m, n, k):
    r = np.random.default_rng(m + n + k)
    a, b = (r.integers(-4, 5, s).astype(np.float32) for s in ((m, k), (k, n)))
    old = gpu.lib().nvl_set_tuning(0, tile)
    try:
        return gpu.ops.mat_mul(a, b, precision="bf16"), (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32)
    finally:
        gpu.lib().nvl_set_tuning(0, old)


@pytest.mark.parametrize("k", [64, 128, 192, 256, 320, 384, 448, 512, 2048])          # 2 .. 16 and 64 K tiles around the six of the ring
@pytest.mark.parametrize("m,n", [(65, 130), (256, 128), (257, 384), (700, 96), (513, 1000)])
def test_wide_tiles_are_exact(gpu, m, n, k):
    """Small whole numbers: every sum is exact in fp32, whatever its order."""
    got, want = product(gpu, 2, m, n, k)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("m,n,k", [(2200, 2176, 2112), (4100, 1100, 64), (2049, 2049, 320)])      # more than 256 tiles: of a long K on four waves, else on eight
def test_many_tiles_are_exact(gpu, m, n, k):
    got, want = product(gpu, 1, m, n, k)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("family,ffn", [("llama", 4224), ("gpt2", 8448), ("falcon", 8448)])      # 66 tiles of 128 gate | up or GELU columns (and falcon's joint ones)
@pytest.mark.parametrize("rows", [385, 512, 513])                                               # the first and last that take 256x128 tiles, and one past it
def test_prompts(gpu, family, ffn, rows):
    """A prompt whose up projection is wide, against the fp32 mode, and again bit for bit."""
    cfg = gpu.synth.tiny_config(family, hidden=256, num_heads=4, num_kv_heads=2 if family == "llama" else 4, head_dim=64, ffn_dim=ffn, num_layers=2, max_seq_len=1024)
    w = gpu.synth.make_weights(cfg, seed=4, scale=0.03)
    tokens = np.random.default_rng(rows).integers(0, cfg["vocab_size"], rows).tolist()
    got = []
    for precision in ("f32", "bf16"):
        m = gpu.HipTransformerModel(cfg, w, precision=precision, max_seqs=1, max_batch_tokens=1024)
        for _ in range(2 if precision == "bf16" else 1):
            m.seq_reset(0)
            got.append(m.forward_batch([0], [tokens], [0], all_logits=True)[0])
        m.close()
    assert np.array_equal(got[1], got[2])
    assert rel_err(got[1], got[0]) <= TOL


@pytest.mark.parametrize("rows,tile,hidden,heads,kv", [(513, 2, 256, 4, 2), (769, 2, 320, 5, 5),       # every projection on 256x128 tiles: rotated heads and residuals too
                                                       (1537, 0, 1024, 32, 8), (2560, 0, 1024, 32, 8)])      # 312 and 480 tiles of 3072 columns: they are chosen for queries, keys and values
def test_wide_tiles_of_heads_and_residuals(gpu, rows, tile, hidden, heads, kv):
    cfg = gpu.synth.tiny_config("llama", hidden=hidden, num_heads=heads, num_kv_heads=kv, head_dim=64, ffn_dim=512, num_layers=2, max_seq_len=2560)
    w = gpu.synth.make_weights(cfg, seed=5, scale=0.03)
    tokens = np.random.default_rng(rows).integers(0, cfg["vocab_size"], rows).tolist()
    got = []
    old = gpu.lib().nvl_set_tuning(0, tile)
    try:
        for precision in ("f32", "bf16"):
            m = gpu.HipTransformerModel(cfg, w, precision=precision, max_seqs=1, max_batch_tokens=2560)
            for _ in range(2 if precision == "bf16" else 1):
                m.seq_reset(0)
                got.append(m.forward_batch([0], [tokens], [0], all_logits=True)[0])
            m.close()
    finally:
        gpu.lib().nvl_set_tuning(0, old)
    assert np.array_equal(got[1], got[2])
    assert rel_err(got[1], got[0]) <= TOL
