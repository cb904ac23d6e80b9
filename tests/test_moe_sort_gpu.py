"""The sort of (token, expert) pairs for prompts and large decode batches (elem.h moe_place_kernel): counted alone or over counters, experts' rows from their
places, the combine under the next norm.  Rows are independent, so each size is checked against the same sequences inside a batch that takes other forms."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu
TOL = 1.5e-2            # bf16 operands, 2^-8 relative, over two layers; sums in another order


@pytest.mark.parametrize("experts,top_k,ffn", [(8, 2, 256), (40, 8, 256), (64, 4, 128)])
def test_sizes_agree(gpu, experts, top_k, ffn):
    """Rows at both sides of what a workgroup takes (1024 pairs), what counts alone (4096), a row-major copy of the operand (512 rows) and the
    combine's own launch (1024 rows); every call twice: the counters are zero again, and nothing depends on the order of a segment's rows."""
    cfg = gpu.synth.tiny_config("granite_moe", hidden=256, num_heads=4, num_kv_heads=2, head_dim=64, ffn_dim=ffn, num_experts=experts, num_experts_per_tok=top_k,
                                num_layers=2, max_seq_len=64, tied_embedding=False)
    w = gpu.synth.make_weights(cfg, seed=5, scale=0.05)
    r = np.random.default_rng(top_k)
    lens = [int(x) for x in r.integers(3, 40, 80)]
    prompts = [r.integers(0, cfg["vocab_size"], k).tolist() for k in lens]
    m = gpu.HipTransformerModel(cfg, w, precision="bf16", max_seqs=80, max_batch_tokens=4096)

    def run(n):
        for i in range(n):
            m.seq_reset(i)
        return m.forward_batch(list(range(n)), prompts[:n], [0] * n)[0]

    whole = run(80)
    rows = np.cumsum(lens)
    assert rows[-1] > 1200
    sizes = {int(np.searchsorted(rows, at, side)) + (side == "right") for at in (128, 256, 512, 1024) for side in ("left", "right")} | {5, 79}
    for n in sorted(sizes):
        got = run(n)
        assert np.array_equal(got, run(n)), n
        assert rel_err(got, whole[:n]) <= TOL, (n, rows[n - 1])
    assert np.array_equal(run(80), whole)
    run(66)                                                     # decode batches of more than 64 rows: captured and replayed
    steps = [m.forward_batch(list(range(66)), [[7]] * 66, [k + j for k in lens[:66]])[0] for j in range(4)]
    run(80)
    for j in range(4):
        assert rel_err(m.forward_batch(list(range(80)), [[7]] * 80, [k + j for k in lens])[0][:66], steps[j]) <= TOL
    m.close()
