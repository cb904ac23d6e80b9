"""forward_rows of a decode batch: the logits of the rows that were named, not of the first ones."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu
TOL = 1.5e-2


@pytest.mark.parametrize("family", ["llama", "gpt2", "granite_moe", "granite_hybrid"])
@pytest.mark.parametrize("rows", [[1], [0, 2], [2]])
def test_rows_of_a_step(gpu, family, rows):
    cfg = gpu.synth.tiny_config(family, num_layers=2, **(dict(hidden=256, mamba_num_heads=16, mamba_head_dim=32) if family == "granite_hybrid" else dict(hidden=256)))
    m = gpu.HipTransformerModel(cfg, gpu.synth.make_weights(cfg, seed=3, scale=0.05), precision="bf16", max_seqs=3, max_batch_tokens=64)
    out = []
    for named in (None, rows):
        for i in range(3):
            m.seq_reset(i)
        m.forward_batch([0, 1, 2], [[5, 6], [7], [8, 9, 2]], [0, 0, 0], want_logits=False)
        step = ([0, 1, 2], [[11], [12], [13]], [2, 1, 3])
        out.append(m.forward_batch(*step)[0] if named is None else m.forward_rows(*step, named)[0])
    m.close()
    # (the final norm in a launch of its own: another rounding of its operand to bf16, 2^-9 of a value at most, on each side)
    assert rel_err(out[1], out[0][rows]) <= TOL
