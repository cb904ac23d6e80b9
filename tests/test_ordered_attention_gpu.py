"""Decode attention that takes ragged contexts from the longest down: the same bits as in the batch's order, for single steps and the greedy loop
(captured graphs replayed), and contexts that cross key tiles and rounds."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,nh,nkv,n", [(64, 8, 8, 33), (64, 16, 4, 66), (128, 8, 4, 70), (64, 40, 1, 90)])      # (40 heads of one group: three query tiles)
@pytest.mark.parametrize("waves", [0, 2, 4, 8])
def test_order_changes_no_bit(gpu, hd, nh, nkv, n, waves):
    """waves 0: the launcher's choice, which may take another number of waves with the order than without: then only as close as any order of sums
    (bf16 activations, 2^-8 relative each, a few layers)."""
    L = gpu.lib()
    cfg = gpu.synth.tiny_config("llama", hidden=256, num_heads=nh, num_kv_heads=nkv, head_dim=hd, ffn_dim=256, max_seq_len=1088, num_layers=2)
    w = gpu.synth.make_weights(cfg, seed=6, scale=0.05)
    r = np.random.default_rng(n + waves)
    lens = [int(x) for x in np.exp(r.uniform(np.log(3), np.log(300), n))]
    lens[n // 2], lens[-1], lens[0] = 1050, 64, 63              # the longest in the middle; tile edges
    prompts = [r.integers(0, cfg["vocab_size"], k).tolist() for k in lens]
    old, got = L.nvl_set_tuning(15, waves), {}
    ids = list(range(n))
    try:
        for order in (0, 2, 1):
            L.nvl_set_tuning(43, order)
            m = gpu.HipTransformerModel(cfg, w, precision="bf16", max_seqs=n, max_batch_tokens=sum(lens))
            for i in ids:
                m.seq_reset(i)
            _, am = m.forward_batch(ids, prompts, [0] * n, want_logits=False)
            steps = []
            for j in range(4):                                  # (the third step of a configuration is a replay)
                lg, am = m.forward_batch(ids, [[int(t)] for t in am], [k + j for k in lens])
                steps.append(lg)
            got[order] = np.stack(steps), m.decode_greedy(ids, am, 6)
            m.close()
    finally:
        L.nvl_set_tuning(43, 1)
        L.nvl_set_tuning(15, old)
    for order in (2, 1) if waves else (2,):
        assert np.array_equal(got[order][0], got[0][0]) and np.array_equal(got[order][1], got[0][1])
    assert rel_err(got[1][0][0], got[0][0][0]) <= 1.5e-2
