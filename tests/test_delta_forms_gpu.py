"""The state scan of delta-rule layers with all key channels a wave and in parts of them (delta_inst.hip scan_shape: by the longest sequence and
the work of all), at the sizes where the choice changes."""
import numpy as np
import pytest

import lufazen_models as LM
import lufazen_oracle as O
from layered_helpers import build, err

pytestmark = pytest.mark.gpu
F32_LAYER = 1e-4        # a single fp32 layer against the plain restatement, as in the other tests of these models
BF16_LAYER = 0.03       # a single bf16 layer, as there


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


@pytest.mark.parametrize("dim,vdim", [(32, 32), (64, 64), (66, 64), (66, 66), (100, 72), (128, 130), (128, 136), (256, 256)])
@pytest.mark.parametrize("lens", [[32], [33], [1, 31, 65, 96], [300] * 24])
def test_scan_forms(gpu, tmp_path, dim, vdim, lens):
    """Chunks that end with the sequence or a token behind or before it, an odd and an even number of them; 24 equal sequences are more than the chip takes at once (all channels a wave).
    Every sequence against the restatement, and the same bits in every run."""
    cfg = LM.config([LM.delta(heads=16, kv_heads=16, dim=dim, vdim=vdim, ff=None)], width=64, vocab=60)
    w = LM.weights(cfg, 17)
    g = np.random.default_rng(dim)
    tok = [g.integers(0, 60, n).tolist() for n in lens]
    m = build(gpu, tmp_path, cfg, w, "f32", max_seqs=len(lens), max_batch_tokens=sum(lens), kv_num_blocks=512)
    ids = list(range(len(lens)))
    runs = []
    for _ in range(4):
        for i in ids:
            m.seq_reset(i)
        runs.append(np.array(m.forward_batch(ids, tok, [0] * len(ids), all_logits=True)[0]))
    m.close()
    got = runs[0]
    at = 0
    for i, t in enumerate(tok):
        assert err(got[at:at + len(t)], O.forward(cfg, w, t), "f32") < F32_LAYER, (i, len(t))
        at += len(t)
    assert all(np.array_equal(got, r) for r in runs[1:])


@pytest.mark.parametrize("lens", [[40, 97], [97, 40, 40], [17, 130, 3, 97, 64], [33, 1, 160, 160, 9, 34], list(range(20, 83)) + [200], [20] * 3 + list(range(80, 19, -1)) + [100]])
def test_scan_order(gpu, tmp_path, lens):
    """The scan takes up to 64 sequences by their lengths (64 and 65 at the end): ties, sequences that another kernel serves, every sequence against the restatement."""
    cfg = LM.config([LM.delta(heads=2, kv_heads=2, dim=40, vdim=72, ff=None)], width=64, vocab=60)
    w = LM.weights(cfg, 17)
    g = np.random.default_rng(len(lens))
    tok = [g.integers(0, 60, n).tolist() for n in lens]
    m = build(gpu, tmp_path, cfg, w, "f32", max_seqs=len(lens), max_batch_tokens=4096, kv_num_blocks=192)
    ids = list(range(len(lens)))
    for i in ids:
        m.seq_reset(i)
    got = np.asarray(m.forward_batch(ids, tok, [0] * len(ids), all_logits=True)[0])
    m.close()
    at = 0
    for t in tok:
        assert err(got[at:at + len(t)], O.forward(cfg, w, t), "f32") < F32_LAYER, len(t)
        at += len(t)


@pytest.mark.parametrize("width", [64, 1056, 2080, 4096])             # 4 / 8 / 16 chunks of a row per lane
@pytest.mark.parametrize("lens", [[513], [519, 9], [1025], [1031, 9]])  # a row per workgroup; 1025 and 1040 rows: tiles of eight, one row over and whole tiles
def test_sandwich_tiles(gpu, tmp_path, width, lens):
    """The prompt's sandwich norms, above 1024 rows in tiles of eight, against portions of up to 300 rows, a row per workgroup: two bf16 runs
    whose operands may round apart, each within the bf16 bound of a layer."""
    cfg = LM.config([LM.delta(heads=2, kv_heads=2, dim=32, vdim=32)], width=width, vocab=60)
    w = LM.weights(cfg, 17)
    g = np.random.default_rng(width)
    tok = [g.integers(0, 60, n).tolist() for n in lens]
    m = build(gpu, tmp_path, cfg, w, "bf16", max_seqs=4, max_seq_len=1088, max_batch_tokens=1088, kv_num_blocks=80)
    ids = list(range(len(lens)))
    for i in range(4):
        m.seq_reset(i)
    whole = np.asarray(m.forward_batch(ids, tok, [0] * len(ids), all_logits=True)[0])
    parts = []
    for i, t in enumerate(tok):
        for a in range(0, len(t), 300):
            parts.append(np.asarray(m.forward_batch([2 + i], [t[a:a + 300]], [a], all_logits=True)[0]))
    m.close()
    assert err(whole, np.concatenate(parts), "bf16") < 2 * BF16_LAYER
