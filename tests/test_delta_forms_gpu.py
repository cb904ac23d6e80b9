"""The state scan of delta-rule layers in one, two and four parts of the key channels (delta_inst.hip scan_shape: by the longest sequence and
the work of all), at the sizes where the choice changes."""
import numpy as np
import pytest

import lufazen_models as LM
import lufazen_oracle as O
from layered_helpers import build, err

pytestmark = pytest.mark.gpu
F32_LAYER = 1e-4        # a single fp32 layer against the plain restatement, as in the other tests of these models


@pytest.mark.parametrize("heads,dim,vdim", [(2, 40, 24), (4, 100, 72), (16, 128, 128), (3, 200, 72), (40, 128, 40), (20, 250, 130)])
def test_scan_parts(gpu, tmp_path, heads, dim, vdim):
    """One long sequence alone (most parts), beside a shorter one, and in a crowd (whole channels): the same logits."""
    cfg = LM.config([LM.delta(heads=heads, kv_heads=heads, dim=dim, vdim=vdim, ff=None)], width=64, vocab=60)
    w = LM.weights(cfg, 17)
    g = np.random.default_rng(heads)
    tok = [g.integers(0, 60, n).tolist() for n in (330, 97) + (40,) * 30]
    want = O.forward(cfg, w, tok[0])
    m = build(gpu, tmp_path, cfg, w, "f32", max_seqs=32, max_batch_tokens=2048)
    for n in (1, 2, 32):
        ids = list(range(n))
        for i in ids:
            m.seq_reset(i)
        got = m.forward_batch(ids, tok[:n], [0] * n, all_logits=True)[0]
        assert err(np.asarray(got)[:330], want, "f32") < F32_LAYER, n
    m.close()
