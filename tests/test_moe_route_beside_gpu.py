"""Decode steps whose experts' up projection routes in its first workgroups, against routing as a launch of its own (nvl_set_tuning key 31 = 2): one to
four expert tiles over one to sixteen waves, one and several row tiles, the narrow and the wide form, 16 waves of four row tiles in the down projection."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("experts,top,ffn", [(8, 2, 64), (33, 5, 64), (48, 12, 64), (64, 3, 128)])      # 64 x 2 x 128 rows: the wide form above 16 rows
@pytest.mark.parametrize("n", [1, 15, 16, 17, 33, 64])
def test_routing_beside_the_up_projection(gpu, experts, top, ffn, n):
    cfg = gpu.synth.tiny_config("granite_moe", num_experts=experts, num_experts_per_tok=top, ffn_dim=ffn, num_layers=2)
    m = gpu.HipTransformerModel(cfg, gpu.synth.make_weights(cfg, seed=17, scale=0.05), precision="bf16", max_seqs=n, max_batch_tokens=256)
    r = np.random.default_rng(n)
    prompts = [r.integers(0, cfg["vocab_size"], 2 + i % 3).tolist() for i in range(n)]
    tokens, ids, got = r.integers(0, cfg["vocab_size"], n).tolist(), list(range(n)), {}
    for key in (1, 2):
        old = gpu.lib().nvl_set_tuning(31, key)
        try:
            for i in ids:
                m.seq_reset(i)
            m.forward_batch(ids, prompts, [0] * n, want_logits=False)
            got[key] = m.forward_batch(ids, [[t] for t in tokens], [len(p) for p in prompts])[0]
        finally:
            gpu.lib().nvl_set_tuning(31, old)
    m.close()
    assert np.array_equal(got[1], got[2])          # (the router's K slices are summed in one order, whatever the launch)
