"""64x128 tiles of the K ring (at most one a CU), four and six K tiles deep: edges of tiles and of the ring, and slices of K in a prompt."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu
TOL = 1.5e-2            # bf16 operands, 2^-8 relative, over two layers; sums in another order


@pytest.mark.parametrize("k", [64, 128, 192, 256, 320, 2048, 4096, 4224])          # from 4096 on the ring is six deep
@pytest.mark.parametrize("m,n", [(65, 130), (64, 128), (129, 384), (700, 96), (1000, 1000), (2048, 1024)])
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


@pytest.mark.parametrize("hidden,ffn,rows", [(1024, 1024, 130), (1024, 4096, 513), (1024, 4096, 900), (2048, 2048, 300), (2048, 2048, 487), (2048, 2048, 1024)])
@pytest.mark.parametrize("family", ["llama", "gpt2"])
def test_prompts(gpu, family, hidden, ffn, rows):
    """Rotated heads, residuals whole and in slices, GELUs and gates: against the fp32 mode, and again bit for bit."""
    cfg = gpu.synth.tiny_config(family, hidden=hidden, num_heads=hidden // 64, num_kv_heads=hidden // 64, head_dim=64, ffn_dim=ffn, num_layers=2, max_seq_len=1024)
    w = gpu.synth.make_weights(cfg, seed=4, scale=0.02)
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
