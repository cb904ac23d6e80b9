"""Decode attention with its keys dealt over workgroups: 1, 2, 3, 5 and 8 parts of one sequence (up to three are combined with fewer loads than up to eight), two,
four and eight waves (of which some have no output block to combine), heads of 64 and 128, groups of heads that fill a row tile and groups that don't."""
import numpy as np
import pytest

from test_model_gpu import build, rel_err

pytestmark = pytest.mark.gpu
BF16_STEP = 1.5e-2        # logits of a bf16 model, as in the tests against the oracle: the forms round the attention's fp32 sums apart by at most one bf16 step


@pytest.mark.parametrize("family,hd", [("llama", 64), ("llama", 128), ("falcon", 64)])
def test_parts_against_whole(gpu, oracle, family, hd):
    over = dict(max_seq_len=1280)
    if hd == 128:
        over.update(head_dim=128, hidden=512)
    cfg, _, _ = build(gpu, oracle, family, "bf16", **over)
    hm = gpu.HipTransformerModel(cfg, gpu.synth.make_weights(cfg, seed=7, scale=0.05), precision="bf16", max_seqs=6, max_batch_tokens=2304, kv_num_blocks=15, kv_block_size=256)
    r = np.random.default_rng(31)
    lens = [1100, 513, 260, 130, 64, 1]
    prompts = [r.integers(0, cfg["vocab_size"], n).tolist() for n in lens]
    ids, tables, at = list(range(len(lens))), [], 0
    for n in lens:
        tables.append(np.arange(at, at + n // 256 + 1, dtype=np.int32))
        at += n // 256 + 1
    tok = [[int(t)] for t in r.integers(0, cfg["vocab_size"], len(lens))]
    hm.forward_paged(prompts, [0] * len(lens), tables, want_logits=False)

    def step(waves, split):
        old = [(k, gpu.lib().nvl_set_tuning(k, v)) for k, v in ((15, waves), (25, split))]
        try:
            out, _ = hm.forward_paged(tok, lens, tables)          # (the step's own keys are written again at the same places)
            again, _ = hm.forward_paged(tok, lens, tables)
            assert np.array_equal(out, again), (waves, split)  # whichever workgroup comes last
            return out.copy()
        finally:
            for k, v in old:
                gpu.lib().nvl_set_tuning(k, v)

    seen = set()
    for waves in (2, 4, 8):
        whole = step(waves, 0)
        for split in (2, 3, 4):                                # 1, 2 and 3 rounds of tiles a part: 18 tiles of 64 keys in up to 8 parts
            got = step(waves, split)
            tiles = (split - 1) * waves * (2 if hd == 64 else 1)
            for i in ids:
                parts = min(8, -(-(lens[i] // 64 + 1) // tiles))
                assert rel_err(got[i], whole[i]) <= BF16_STEP, (waves, split, lens[i])
                if parts == 1:
                    assert np.array_equal(got[i], whole[i]), (waves, split, lens[i])
                elif lens[i] > 500:                            # (sums of hundreds of keys in another order: some of the bits differ)
                    assert not np.array_equal(got[i], whole[i]), (waves, split, lens[i])
                    seen.add(parts)
    assert seen >= ({2, 3, 5} if hd == 64 else {2, 3, 5, 8})
    hm.close()
