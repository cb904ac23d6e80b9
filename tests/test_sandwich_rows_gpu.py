"""Sandwich norms of 513 .. 1024 rows, a workgroup per row with a row-major copy for experts and K slices to add up, and of more rows, tiles of eight.
Experts of whole 256-wide tiles (experts-in-place) read their rows from that copy, in 256-row segments that end anywhere."""
import numpy as np
import pytest

import medulorn_models as MM
from layered_helpers import build, err, feed

pytestmark = pytest.mark.gpu
BF16_LAYER = 0.03       # a single bf16 layer, as in the other tests of these models


def against_fp32(gpu, tmp_path, cfg, w, tok):
    got = {}
    for precision in ("bf16", "f32"):
        m = build(gpu, tmp_path, cfg, w, precision, max_seqs=2, max_seq_len=1088, max_batch_tokens=1088)
        m.seq_reset(0)
        got[precision] = np.asarray(m.forward_batch([0], [tok], [0], all_logits=True)[0])
        m.close()
    assert err(got["bf16"], got["f32"], "bf16") < BF16_LAYER


@pytest.mark.parametrize("n", [513, 768, 769, 1024, 1025, 1031])      # queries and keys normed and turned head by head up to 768 rows (heads of 64 in registers: 512), in tiles of 16 tokens above
@pytest.mark.parametrize("layer,width", [(MM.attention(mlp=MM.moe()), 96), (MM.attention(mlp=MM.moe()), 1056), (MM.attention(mlp=MM.moe()), 2080), (MM.parallel(mlp=MM.dense(48)), 96),
                                         (MM.attention(mlp=MM.moe(experts=6, top=2, ff=256)), 256), (MM.attention(mlp=MM.moe(experts=6, top=2, ff=256)), 512),
                                         (MM.attention(heads=16, kv_heads=4, dim=64, vdim=64, turn=MM.rot(64), mlp=MM.dense(2048)), 1024),      # 64 and more slices of both residual projections
                                         (MM.attention(heads=4, kv_heads=2, dim=128, vdim=128, turn=MM.rot(128), mlp=MM.dense(48)), 128)],
                         ids=["experts-96", "experts-1056", "experts-2080", "parallel", "experts-in-place-256", "experts-in-place-512", "slices", "heads-128"])
def test_rows_and_tiles(gpu, tmp_path, layer, width, n):
    cfg = MM.config([layer], width=width, vocab=130)
    w = MM.weights(cfg, 11)
    tok = np.random.default_rng(n).integers(0, 130, n).tolist()
    if "experts" in str(layer):
        tok = MM.clear_tokens(cfg, w, n, 1)[0]          # (no near tie between experts)
    against_fp32(gpu, tmp_path, cfg, w, list(tok))


@pytest.mark.parametrize("layer,width", [(MM.attention(mlp=MM.moe(experts=96)), 96), (MM.attention(mlp=MM.moe(experts=80)), 2080), (MM.attention(mlp=MM.dense(48)), 4128)],
                         ids=["six-parts", "five-parts", "wide"])
def test_one_row_a_workgroup(gpu, tmp_path, layer, width):
    """Single rows: more than four partial sums of the experts, and rows too wide for the weights of both norms to be fetched ahead."""
    cfg = MM.config([layer, layer], width=width, vocab=130)
    w = MM.weights(cfg, 11)
    tok = MM.clear_tokens(cfg, w, 7, 1, margin=0.01)[0]          # (no near tie between experts)
    got = {}
    for precision in ("bf16", "f32"):
        m = build(gpu, tmp_path, cfg, w, precision, max_seqs=2, max_seq_len=64, max_batch_tokens=64)
        got[precision] = feed(m, 0, tok, [1] * len(tok))
        m.close()
    assert err(got["bf16"], got["f32"], "bf16") < 2 * BF16_LAYER          # (two layers)


@pytest.mark.parametrize("experts,top,ff,width", [(8, 2, 1100, 2080), (33, 3, 448, 1056), (48, 3, 330, 992), (64, 2, 256, 1024)])      # one to four expert tiles, one to four chunks of a row a thread
def test_routing_with_the_norm(gpu, tmp_path, experts, top, ff, width):
    """Single rows whose experts' routing is in the launch of the norm that makes their input, against one of its own (nvl_set_tuning key 31 = 2)."""
    cfg = MM.config([MM.attention(mlp=MM.moe(experts=experts, top=top, ff=ff)), MM.attention(mlp=MM.moe(experts=experts, top=top, ff=ff, shared=None))], width=width, vocab=130)
    m = build(gpu, tmp_path, cfg, MM.weights(cfg, 11), "bf16", max_seqs=20, max_seq_len=64, max_batch_tokens=64)
    m.set_profile(True)
    g = np.random.default_rng(1)
    for n in (1, 5, 17):
        tok, got, launches, ids = g.integers(0, 130, (3, n)).tolist(), {}, {}, list(range(n))
        for key in (1, 2):
            old = gpu.lib().nvl_set_tuning(31, key)
            try:
                for i in ids:
                    m.seq_reset(i)
                m.reset_stats()
                got[key] = [np.asarray(m.forward_batch(ids, [[t] for t in row], [p] * n)[0]) for p, row in enumerate(tok)]
                launches[key] = sum(k["launches"] for k in m.kernel_stats() if k["site"] == "moe_router")
            finally:
                gpu.lib().nvl_set_tuning(31, old)
        assert all(np.array_equal(a, b) for a, b in zip(got[1], got[2]))          # (the router's K slices and their sums are the same)
        assert launches[1] == 0 and launches[2] > 0
    m.close()
