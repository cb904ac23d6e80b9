"""Projections of up to 512 rows (gemm.h gemm_mid_bf16_kernel: K split over workgroups, split_finish) and the single-launch Mamba-2 decode
step (mamba.h mamba_step_kernel), at the sizes where they can go wrong."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu
TOL = 1.5e-2


@pytest.mark.parametrize("parts", [0, 1, 2, 5, 8])                 # K split over workgroups; 0: the launcher's choice
@pytest.mark.parametrize("m,k,n", [(65, 2048, 64), (66, 2112, 200), (96, 2048, 130), (97, 4160, 2048), (128, 2048, 1003), (129, 2048, 256),
                                   (255, 2176, 320), (257, 2048, 2049), (512, 2048, 192), (1, 4096, 64), (33, 1984, 2049), (64, 64, 33)])
def test_matmul_is_exact_on_integers(gpu, parts, m, k, n):
    """Ragged rows, columns and K (a last stage of 64, K parts of unequal length), the kernel forced (by cost it would take few of these); the
    sums are exact in fp32 in any order."""
    a = (np.arange(m * k).reshape(m, k) % 7).astype(np.float32) - 1.0
    b = (np.arange(k * n).reshape(k, n) % 5).astype(np.float32) - 2.0        # |sums| < 2^24
    old = [(key, gpu.lib().nvl_set_tuning(key, v)) for key, v in ((39, parts), (38, 2))]
    try:
        got = gpu.ops.mat_mul(a, b, precision="bf16")
    finally:
        for key, v in old:
            gpu.lib().nvl_set_tuning(key, v)
    want = (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("m,k,n", [(97, 4160, 2048), (129, 2048, 256), (70, 2048, 1024)])
def test_a_forced_kernel_is_taken(gpu, m, k, n):
    """Keys 38 and 39 go before the form that has all of K in a workgroup, which would take these sizes: K in one part, in three and in five are sums in three orders."""
    r = np.random.default_rng(m)
    a, b, got = r.standard_normal((m, k)).astype(np.float32), r.standard_normal((k, n)).astype(np.float32), {}
    for mid, parts in ((2, 1), (2, 3), (2, 5), (1, 3)):
        old = [(key, gpu.lib().nvl_set_tuning(key, v)) for key, v in ((38, mid), (39, parts))]
        try:
            got[mid, parts] = gpu.ops.mat_mul(a, b, precision="bf16")
        finally:
            for key, v in old:
                gpu.lib().nvl_set_tuning(key, v)
    assert not np.array_equal(got[2, 1], got[2, 3]) and not np.array_equal(got[2, 3], got[2, 5]) and not np.array_equal(got[2, 1], got[2, 5])
    if k * n >= 4 << 20:                                                  # (below, one part by cost is not this kernel)
        assert np.array_equal(got[1, 3], got[2, 3])
    for y in got.values():
        assert rel_err(y, got[2, 1]) <= 1e-5                                # (fp32 sums of the same products)


@pytest.mark.parametrize("n", [65, 97, 128])
def test_long_residual_projections_in_parts(gpu, n):
    """FFN-down of 2048 x 8192 behind 65 .. 128 rows, with a deferred norm: K in one part and in several, one to three 16-row tiles a wave, against the fp32 mode."""
    cfg = gpu.synth.tiny_config("llama", hidden=2048, num_heads=32, num_kv_heads=8, head_dim=64, ffn_dim=8192, num_layers=2, max_seq_len=64)
    w = gpu.synth.make_weights(cfg, seed=8, scale=0.02)
    r = np.random.default_rng(n)
    prompts = [r.integers(0, cfg["vocab_size"], 1 + i % 3).tolist() for i in range(n)]
    ids, got = list(range(n)), {}
    m = gpu.HipTransformerModel(cfg, w, precision="bf16", max_seqs=n, max_batch_tokens=512)

    def step(m):
        for i in ids:
            m.seq_reset(i)
        m.forward_batch(ids, prompts, [0] * n, want_logits=False)
        return m.forward_batch(ids, [[7]] * n, [len(p) for p in prompts])[0].copy()

    for parts in (1, 3, 4):
        old = [(key, gpu.lib().nvl_set_tuning(key, v)) for key, v in ((38, 2), (39, parts))]
        try:
            got[parts] = step(m)
            assert np.array_equal(step(m), got[parts]), parts            # (the counters of the parts are zero again)
        finally:
            for key, v in old:
                gpu.lib().nvl_set_tuning(key, v)
    m.close()
    m = gpu.HipTransformerModel(cfg, w, precision="f32", max_seqs=n, max_batch_tokens=512)
    want = step(m)
    m.close()
    assert not np.array_equal(got[1], got[3]) and not np.array_equal(got[3], got[4])
    for parts, y in got.items():
        assert rel_err(y, want) <= TOL, parts


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("parts", [0, 3])                             # K split over workgroups; 0: the launcher's choice
@pytest.mark.parametrize("n,mid", [(5, 2), (33, 2), (64, 1), (64, 2), (65, 1), (97, 1), (128, 1), (130, 1)])      # 130: past the deferred norm
def test_decode_and_prompt_batches(gpu, hd, parts, n, mid):
    """Every epilogue of the kernel in a model: decode batches (deferred norms, gate | up pairs) and short prompts (rotated heads, cache rows)
    against the fp32 mode; the same prompts again, and the greedy loop (graph replays) against single steps, bit for bit: the counters
    of a split are zero again after each launch, whichever shape comes next."""
    cfg = gpu.synth.tiny_config("llama", hidden=2048, num_heads=2048 // hd, num_kv_heads=512 // hd, head_dim=hd, ffn_dim=2048, max_seq_len=64)
    w = gpu.synth.make_weights(cfg, seed=4, scale=0.02)
    r = np.random.default_rng(n)
    prompts = [r.integers(0, cfg["vocab_size"], 1 + i % 3).tolist() for i in range(n)]
    ids, got = list(range(n)), {}
    old = [(key, gpu.lib().nvl_set_tuning(key, v)) for key, v in ((38, mid), (39, parts))]
    for precision in ("bf16", "f32"):
        m = gpu.HipTransformerModel(cfg, w, precision=precision, max_seqs=n, max_batch_tokens=512)
        for i in ids:
            m.seq_reset(i)
        first, _ = m.forward_batch(ids, prompts, [0] * n)
        step, am = m.forward_batch(ids, [[7]] * n, [len(p) for p in prompts])
        got[precision] = first, step
        if precision == "bf16":
            pos = [len(p) + 1 for p in prompts]
            one = []
            for j in range(3):
                _, am = m.forward_batch(ids, [[int(t)] for t in am], [p + j for p in pos], want_logits=False)
                one.append(am)
            for i in ids:
                m.seq_reset(i)
            again, _ = m.forward_batch(ids, prompts, [0] * n)
            assert np.array_equal(again, first)
            _, am = m.forward_batch(ids, [[7]] * n, [len(p) for p in prompts], want_logits=False)
            assert np.array_equal(m.decode_greedy(ids, am, 3), np.stack(one))
        m.close()
    for key, v in old:
        gpu.lib().nvl_set_tuning(key, v)
    assert rel_err(got["bf16"][0], got["f32"][0]) <= TOL and rel_err(got["bf16"][1], got["f32"][1]) <= TOL


@pytest.mark.parametrize("hidden,heads,hd,state,groups", [(512, 16, 64, 128, 2), (256, 16, 32, 32, 1), (256, 16, 32, 256, 4), (512, 32, 32, 64, 32)])
@pytest.mark.parametrize("n", [1, 16, 17, 64])
def test_mamba_decode_step(gpu, oracle, hidden, heads, hd, state, groups, n):
    """One launch from the input projection's rows to the output projection's operand, the gated norm deferred: logits and states of a
    few steps against the fp32 mode and, for one sequence, the oracle."""
    cfg = gpu.synth.tiny_config("granite_hybrid", hidden=hidden, num_heads=hidden // 64, num_kv_heads=hidden // 128, mamba_num_heads=heads, mamba_head_dim=hd,
                                mamba_state_size=state, mamba_n_groups=groups)
    w = gpu.synth.make_weights(cfg, seed=23, scale=0.05)
    r = np.random.default_rng(n)
    prompts = [r.integers(0, cfg["vocab_size"], 1 + i % 4).tolist() for i in range(n)]
    steps = r.integers(0, cfg["vocab_size"], (3, n)).tolist()
    ids, got = list(range(n)), {}
    for precision in ("bf16", "f32"):
        m = gpu.HipTransformerModel(cfg, w, precision=precision, max_seqs=n, max_batch_tokens=256)
        for i in ids:
            m.seq_reset(i)
        m.forward_batch(ids, prompts, [0] * n, want_logits=False)
        lg = [m.forward_batch(ids, [[t] for t in s], [len(p) + j for p in prompts])[0] for j, s in enumerate(steps)]
        got[precision] = lg, m.get_mamba_state(n - 1, 0), m.get_mamba_state(0, 3)
        m.close()
    for j in range(3):
        assert rel_err(got["bf16"][0][j], got["f32"][0][j]) <= TOL
    assert rel_err(got["bf16"][1], got["f32"][1]) <= TOL and rel_err(got["bf16"][2], got["f32"][2]) <= TOL
    om = oracle.OracleModel(cfg, w)
    kv = om.new_cache()
    om.forward_with_cache(prompts[0], kv, 0)
    if len(prompts[0]) == 1:              # (a one-token call does not reset the oracle's state: it starts at zero here)
        for j, s in enumerate(steps):
            want = om.forward_with_cache([s[0]], kv, 1 + j)[-1]
            assert rel_err(got["bf16"][0][j][0], want) <= TOL


@pytest.mark.parametrize("parts", [2, 3, 5])
@pytest.mark.parametrize("m,k,n", [(520, 2048, 1300), (1100, 2112, 2056), (2100, 2112, 2056), (256, 1984, 256 * 9), (1025, 2048, 256 * 53)])
def test_large_tiles_of_the_last_round_in_parts(gpu, parts, m, k, n):
    """The ping-pong kernel with its last round cut along K, uneven parts, XCDs with one tile less than others or none: exact on integers.
    18, 45, 81, 9 and 265 tiles, at most 3, 6, 11, 2 and 34 = 32 + 2 of them an XCD: 32 workgroups hold the parts, so that 81 are cut in two only
    and stay whole at 3 and 5."""
    a = (np.arange(m * k).reshape(m, k) % 7).astype(np.float32) - 1.0
    b = (np.arange(k * n).reshape(k, n) % 5).astype(np.float32) - 2.0
    old = [(key, gpu.lib().nvl_set_tuning(key, v)) for key, v in ((0, 5), (41, parts))]
    try:
        got = gpu.ops.mat_mul(a, b, precision="bf16")
    finally:
        for key, v in old:
            gpu.lib().nvl_set_tuning(key, v)
    want = (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("family,hd,tile", [("llama", 64, 5), ("llama", 128, 5), ("llama", 128, 0), ("gpt2", 64, 5)])
@pytest.mark.parametrize("hidden,parts", [(1024, 2), (2048, 3), (2048, 5)])
def test_epilogues_behind_large_tiles_in_parts(gpu, family, hd, tile, hidden, parts):
    """Every epilogue of the ping-pong kernel behind a split of K: residual, gate | up, GELU, rotated heads of 64, and (tile 0: the large tiles
    are not forced, heads of 128 take them all the same) of 128.  600 rows: 12 .. 48 tiles, 2 .. 6 an XCD, parts of 12 .. 21 K-steps.  The same
    call whole and in parts differs in the order of fp32 sums, each within the bf16 bound of the fp32 mode; again bit for bit (the counters)."""
    over = dict(num_kv_heads=256 // hd) if family == "llama" else {}
    cfg = gpu.synth.tiny_config(family, hidden=hidden, num_heads=hidden // hd, head_dim=hd, ffn_dim=hidden, max_seq_len=640, **over)
    m = gpu.HipTransformerModel(cfg, gpu.synth.make_weights(cfg, seed=12, scale=0.03), precision="bf16", max_seqs=1, max_batch_tokens=640)
    tokens = np.random.default_rng(hd).integers(0, cfg["vocab_size"], 600).tolist()
    got = []
    for cut in (1, parts):
        old = [(key, gpu.lib().nvl_set_tuning(key, v)) for key, v in ((0, tile), (41, cut))]
        try:
            for _ in range(2):
                m.seq_reset(0)
                got.append(m.forward_batch([0], [tokens], [0], all_logits=True)[0])
        finally:
            for key, v in old:
                gpu.lib().nvl_set_tuning(key, v)
    m.close()
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[2], got[3]) and not np.array_equal(got[0], got[2])
    assert rel_err(got[2], got[0]) <= TOL


@pytest.mark.parametrize("n", [1, 16, 17, 40, 64])
def test_moe_down_completes_its_slices(gpu, n):
    """The experts' down projection of a decode batch: the last of a tile's K slices adds them up and carries the next norm (gemm.h
    split_finish_wave), against slices left to a norm launch; graph replays against single steps (every counter back at zero)."""
    import torch
    from bench import gen_weights_on_device
    cfg = dict(gpu.synth.FULL_CONFIGS["granite-3.0-1b-a400m"], num_layers=2, vocab_size=1000)
    m = gpu.HipTransformerModel(cfg, None, precision="bf16", max_seqs=n, max_batch_tokens=256)
    gen_weights_on_device(gpu, cfg, m, torch, torch.device("cuda", 0), keep_host=False)
    m.finalize()
    ids, prompts, got = list(range(n)), [[3 + i % 900, 5] for i in range(n)], {}

    def prompt():
        for i in ids:
            m.seq_reset(i)
        m.forward_batch(ids, prompts, [0] * n, want_logits=False)

    for form in (0, 1):
        old = gpu.lib().nvl_set_tuning(33, form)
        prompt()
        got[form], am = m.forward_batch(ids, [[7]] * n, [2] * n)
        one = []
        for j in range(4):
            _, am = m.forward_batch(ids, [[int(t)] for t in am], [3 + j] * n, want_logits=False)
            one.append(am)
        prompt()
        _, am = m.forward_batch(ids, [[7]] * n, [2] * n, want_logits=False)
        assert np.array_equal(m.decode_greedy(ids, am, 4), np.stack(one)), form
        gpu.lib().nvl_set_tuning(33, old)
    m.close()
    # the norm's factor multiplies the bf16 operand in one form, the fp32 products in the other: one bf16 rounding (2^-9) a layer
    assert rel_err(got[1], got[0]) <= 2e-2


@pytest.mark.parametrize("heads,hd,groups", [(16, 64, 2), (8, 32, 1), (10, 64, 1)])      # 10 heads: rows that are no multiple of 16 bytes
@pytest.mark.parametrize("lens", [[1, 2, 3, 4, 117], [128], [5, 7, 9, 130, 1, 8, 23]])
def test_mamba_prompts(gpu, heads, hd, groups, lens):
    """The convolution over runs of tokens (sequences that begin anywhere in a run) and the gated norm row by row: a batch against each
    prompt alone in the fp32 mode (the same sums), and the bf16 mode against it."""
    cfg = gpu.synth.tiny_config("granite_hybrid", hidden=heads * hd // 2, num_heads=heads * hd // 128, num_kv_heads=1, mamba_num_heads=heads, mamba_head_dim=hd, mamba_state_size=32,
                                mamba_n_groups=groups, max_seq_len=256)
    w = gpu.synth.make_weights(cfg, seed=29, scale=0.05)
    r = np.random.default_rng(len(lens))
    prompts = [r.integers(0, cfg["vocab_size"], n).tolist() for n in lens]
    ids, got = list(range(len(lens))), {}
    for precision in ("bf16", "f32"):
        m = gpu.HipTransformerModel(cfg, w, precision=precision, max_seqs=len(lens), max_batch_tokens=256)
        for i in ids:
            m.seq_reset(i)
        got[precision] = m.forward_batch(ids, prompts, [0] * len(ids))[0]
        if precision == "f32":
            for i in ids:
                m.seq_reset(i)
                alone = m.forward_batch([i], [prompts[i]], [0])[0]
                assert rel_err(alone[0], got["f32"][i]) <= 1e-5, lens[i]
        m.close()
    assert rel_err(got["bf16"], got["f32"]) <= TOL


@pytest.mark.parametrize("heads,hd,groups", [(16, 64, 2), (8, 32, 1), (10, 64, 1)])
@pytest.mark.parametrize("lens", [[511], [512], [300, 217]])
def test_mamba_gate_rows_and_tiles(gpu, heads, hd, groups, lens):
    """The gated norm row by row up to 511 rows and in tiles of eight from 512 on: every row of the bf16 mode against the fp32 mode."""
    cfg = gpu.synth.tiny_config("granite_hybrid", hidden=heads * hd // 2, num_heads=heads * hd // 128, num_kv_heads=1, mamba_num_heads=heads, mamba_head_dim=hd, mamba_state_size=32,
                                mamba_n_groups=groups, max_seq_len=520)
    w = gpu.synth.make_weights(cfg, seed=37, scale=0.05)
    r = np.random.default_rng(sum(lens))
    prompts, ids, got = [r.integers(0, cfg["vocab_size"], n).tolist() for n in lens], list(range(len(lens))), {}
    for precision in ("bf16", "f32"):
        m = gpu.HipTransformerModel(cfg, w, precision=precision, max_seqs=len(lens), max_batch_tokens=520)
        for i in ids:
            m.seq_reset(i)
        got[precision] = m.forward_batch(ids, prompts, [0] * len(ids), all_logits=True)[0]
        m.close()
    assert rel_err(got["bf16"], got["f32"]) <= TOL


@pytest.mark.parametrize("lens,all_logits", [([600], True), ([641], False), ([700, 330], False), ([1100], True)])
def test_mamba_prompts_in_slices(gpu, lens, all_logits):
    """Residual projections of 600 .. 1100 rows whose K is cut and summed by the norm behind them, in Mamba and attention layers, up to the final norm: against the fp32
    mode, and a step from the state they leave."""
    cfg = gpu.synth.tiny_config("granite_hybrid", hidden=512, num_heads=4, num_kv_heads=2, ffn_dim=2048, mamba_num_heads=16, mamba_head_dim=64, mamba_state_size=32, max_seq_len=1200)
    w = gpu.synth.make_weights(cfg, seed=31, scale=0.03)
    r = np.random.default_rng(sum(lens))
    prompts, ids, got = [r.integers(0, cfg["vocab_size"], n).tolist() for n in lens], list(range(len(lens))), {}
    for precision in ("bf16", "f32"):
        m = gpu.HipTransformerModel(cfg, w, precision=precision, max_seqs=len(lens), max_batch_tokens=1200)
        for i in ids:
            m.seq_reset(i)
        z = m.forward_batch(ids, prompts, [0] * len(ids), all_logits=all_logits)[0]
        got[precision] = [z, m.forward_batch(ids, [[7]] * len(ids), lens)[0]]
        m.close()
    for a, b in zip(got["bf16"], got["f32"]):
        assert rel_err(a, b) <= TOL


@pytest.mark.parametrize("n", [65, 513, 530, 1040])
def test_moe_prompt_forms(gpu, n):
    """Routing in the router's launch, experts that read their rows from the norm's row-major result (beyond 512 tokens): against the separate
    launches and rows copied into expert order from the fragment-major operand."""
    import torch
    from bench import gen_weights_on_device
    cfg = dict(gpu.synth.FULL_CONFIGS["granite-3.0-1b-a400m"], num_layers=1, vocab_size=1000)
    m = gpu.HipTransformerModel(cfg, None, precision="bf16", max_seqs=1, max_batch_tokens=1088)
    gen_weights_on_device(gpu, cfg, m, torch, torch.device("cuda", 0), keep_host=False)
    m.finalize()
    tokens, got = np.random.default_rng(n).integers(0, 1000, n).tolist(), []
    for forms in ((1, 1), (0, 0)):
        old = [(key, gpu.lib().nvl_set_tuning(key, v)) for key, v in zip((9, 31), forms)]
        m.seq_reset(0)
        got.append(m.forward_batch([0], [tokens], [0], all_logits=True)[0])
        for key, v in old:
            gpu.lib().nvl_set_tuning(key, v)
    m.close()
    # the same bf16 operands; logits of the router that differ in the order of their fp32 sums may swap two experts of equal weight: few rows
    err = np.abs(got[0] - got[1]).max(-1) / np.abs(got[1]).max()
    assert np.mean(err > 5e-3) <= 0.01


@pytest.mark.parametrize("family,hd", [("gpt2", 64), ("llama", 64), ("llama", 128), ("falcon", 64)])
@pytest.mark.parametrize("lens", [[2], [16], [1, 15, 1], [33], [20, 44], [31, 1, 1]])
def test_short_prompts_place_their_heads(gpu, family, hd, lens):
    """Up to 64 tokens: the QKV projection rotates and places its heads itself (key 18 = 64: fp32 rows and a launch of their own).  The same
    fp32 sums and one rounding each way, so only the order of the K slices differs; the cache by a decode step that reads it."""
    cfg = gpu.synth.tiny_config(family, hidden=256, num_heads=256 // hd, head_dim=hd, num_kv_heads=1 if family == "falcon" else 256 // hd, max_seq_len=64)
    m = gpu.HipTransformerModel(cfg, gpu.synth.make_weights(cfg, seed=3, scale=0.05), precision="bf16", max_seqs=len(lens), max_batch_tokens=128)
    r = np.random.default_rng(sum(lens))
    prompts = [r.integers(0, cfg["vocab_size"], n).tolist() for n in lens]
    ids, got = list(range(len(lens))), []
    for rows in (0, 64):
        old = gpu.lib().nvl_set_tuning(18, rows)
        for i in ids:
            m.seq_reset(i)
        first = m.forward_batch(ids, prompts, [0] * len(ids))[0]
        got.append((first, m.forward_batch(ids, [[9]] * len(ids), lens)[0]))
        gpu.lib().nvl_set_tuning(18, old)
    m.close()
    assert rel_err(got[0][0], got[1][0]) <= TOL and rel_err(got[0][1], got[1][1]) <= TOL


@pytest.mark.parametrize("rows", [0, 2, 3])                          # 256, 128, 64 query rows per workgroup
@pytest.mark.parametrize("nH,nKV,S,T,hd", [(4, 2, 5, 5, 64), (2, 2, 33, 100, 64), (3, 1, 7, 64, 128), (71, 1, 2, 130, 64), (8, 2, 130, 130, 128),
                                           (4, 2, 300, 1400, 64), (4, 2, 65, 257, 128), (1, 1, 64, 64, 64), (1, 1, 129, 200, 128)])
def test_prefill_attention_rows(gpu, oracle, rows, nH, nKV, S, T, hd):
    """Ragged row counts, waves without a row, diagonal and whole key tiles, more of them than the LDS ring holds; the same products whatever
    the workgroup's rows: only the last tiles of the other rows differ, and those are masked."""
    r = np.random.default_rng(nH * 10 + T)
    q, k, v = (r.standard_normal(s, dtype=np.float32) for s in ((nH, S, hd), (nKV, T, hd), (nKV, T, hd)))
    old = gpu.lib().nvl_set_tuning(10, rows)
    got = gpu.ops.attention(q, k, v, precision="bf16")
    gpu.lib().nvl_set_tuning(10, old)
    assert rel_err(got, oracle.gqa_core(q, k, v)) <= TOL


@pytest.mark.parametrize("hd,kv", [(64, 1), (64, 4), (128, 2)])
@pytest.mark.parametrize("waves", [0, 2, 4, 8])                       # 0: the launcher's form
@pytest.mark.parametrize("rounds", [1, 2])
def test_decode_attention_in_parts(gpu, hd, kv, waves, rounds):
    """Each sequence dealt over as many workgroups as its own length asks for (one, some, the most; a last part of one key): a step against the
    whole form and the greedy loop (graph replays: the tickets are zero again) against single steps."""
    cfg = gpu.synth.tiny_config("llama", hidden=256, num_heads=256 // hd, head_dim=hd, num_kv_heads=min(kv, 256 // hd), max_seq_len=1536)
    m = gpu.HipTransformerModel(cfg, gpu.synth.make_weights(cfg, seed=5, scale=0.05), precision="bf16", max_seqs=5, max_batch_tokens=1536)
    r = np.random.default_rng(8)
    lens = [1400, 1, 256, 511, 700]
    prompts = [r.integers(0, cfg["vocab_size"], n).tolist() for n in lens]
    ids, got = list(range(5)), []

    def prompt():
        for i in ids:
            m.seq_reset(i)
            m.forward_batch([i], [prompts[i]], [0], want_logits=False)

    for form in (0, 1 + rounds if waves else 1):
        old = [(key, gpu.lib().nvl_set_tuning(key, v)) for key, v in ((25, form), (15, waves if form else 0))]
        prompt()
        first, am = m.forward_batch(ids, [[7]] * 5, lens)
        one = []
        for j in range(3):
            _, am = m.forward_batch(ids, [[int(t)] for t in am], [n + 1 + j for n in lens], want_logits=False)
            one.append(am)
        prompt()
        _, am = m.forward_batch(ids, [[7]] * 5, lens, want_logits=False)
        assert np.array_equal(m.decode_greedy(ids, am, 3), np.stack(one))
        got.append(first)
        for key, v in old:
            gpu.lib().nvl_set_tuning(key, v)
    m.close()
    assert rel_err(got[1], got[0]) <= TOL


@pytest.mark.parametrize("hd,n,longest", [(64, 10, 1900), (64, 12, 1500), (64, 16, 1300), (64, 16, 1000), (128, 8, 1500), (128, 12, 1500), (128, 16, 800),
                                             (128, 16, 1100)])
def test_decode_attention_parts_by_pairs(gpu, hd, n, longest):
    """The launcher's own parts where pairs bound them (parts of one, two and three rounds): ragged contexts down to one key, against the whole form."""
    cfg = gpu.synth.tiny_config("llama", hidden=8 * hd, num_heads=8, head_dim=hd, num_kv_heads=8, max_seq_len=2048)
    m = gpu.HipTransformerModel(cfg, gpu.synth.make_weights(cfg, seed=5, scale=0.05), precision="bf16", max_seqs=n, max_batch_tokens=2048)
    r = np.random.default_rng(n)
    lens = [longest, 1] + r.integers(2, longest + 1, n - 2).tolist()
    prompts = [r.integers(0, cfg["vocab_size"], x).tolist() for x in lens]
    ids, got = list(range(n)), []
    for form in (0, 1):
        old = gpu.lib().nvl_set_tuning(25, form)
        for i in ids:
            m.seq_reset(i)
            m.forward_batch([i], [prompts[i]], [0], want_logits=False)
        got.append([m.forward_batch(ids, [[7 + j]] * n, [x + j for x in lens])[0] for j in range(3)])      # (the tickets are zero again)
        gpu.lib().nvl_set_tuning(25, old)
    m.close()
    for whole, parts in zip(*got):
        assert rel_err(parts, whole) <= TOL and not np.array_equal(parts, whole)


@pytest.mark.parametrize("family,hidden,heads", [("llama", 192, 3), ("llama", 2048, 16), ("falcon", 2112, 33), ("llama", 4096, 32), ("falcon", 4544, 71),
                                                 ("llama", 4608, 36), ("llama", 4672, 73)])       # up to 2048 / 4096 / 4608 columns, and beyond
@pytest.mark.parametrize("lens", [[513], [1025], [600, 440], [1033]])      # a row per workgroup up to 1024 rows; tiles: remainders of 8 and of 16
def test_norm_tiles(gpu, family, hidden, heads, lens):
    """The prompt's norms in tiles of eight rows (also with a residual add left as slices) or a row per workgroup against one wave per row.
    The sums differ in order, so an operand may round the other way, one bf16 step of 2^-8; three norms lie on the way to the logits
    (before attention, before the FFN, before the head): 3 * 2^-8."""
    kv = 1 if family == "falcon" else heads
    cfg = gpu.synth.tiny_config(family, hidden=hidden, num_heads=heads, num_kv_heads=kv, head_dim=hidden // heads,
                                ffn_dim=512, num_layers=1, max_seq_len=1100)
    w = gpu.synth.make_weights(cfg, seed=6, scale=0.02)
    r = np.random.default_rng(hidden)
    prompts = [r.integers(0, cfg["vocab_size"], t).tolist() for t in lens]
    got = []
    for tiles in (1, 0):
        old = gpu.lib().nvl_set_tuning(9, tiles)
        m = gpu.HipTransformerModel(cfg, w, precision="bf16", max_seqs=len(lens), max_batch_tokens=2048)
        try:
            for i in range(len(lens)):
                m.seq_reset(i)
            got.append(m.forward_batch(list(range(len(lens))), prompts, [0] * len(lens), want_logits=True)[0])
        finally:
            gpu.lib().nvl_set_tuning(9, old)
            m.close()
    assert np.isfinite(got[0]).all() and rel_err(got[0], got[1]) < 3 * 2.0 ** -8


@pytest.mark.parametrize("m,k,n", [(33, 64, 128), (64, 2048, 128), (65, 768, 2304), (70, 2112, 256), (96, 3072, 768), (97, 1536, 1024), (128, 4544, 128), (129, 2048, 2048),
                                   (145, 960, 1280), (200, 2048, 1024), (250, 1088, 2048), (256, 2048, 2048), (80, 2048, 3072), (100, 1024, 4096)])
def test_rows_form_is_exact_on_integers(gpu, m, k, n):
    """Groups of 32, 48 and 64 rows by one and two column tiles with all of K in a workgroup (forced), five to eight waves, K steps that leave a rest of a block of
    four, waves without any; ragged last groups."""
    a = (np.arange(m * k).reshape(m, k) % 7).astype(np.float32) - 1.0
    b = (np.arange(k * n).reshape(k, n) % 5).astype(np.float32) - 2.0        # |sums| < 2^24
    old = gpu.lib().nvl_set_tuning(46, 2)
    try:
        got = gpu.ops.mat_mul(a, b, precision="bf16")
    finally:
        gpu.lib().nvl_set_tuning(46, old)
    assert np.array_equal(got, (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32))


@pytest.mark.parametrize("hidden,norm", [(768, "rmsnorm"), (2048, "rmsnorm"), (768, "layernorm")])
@pytest.mark.parametrize("n", [33, 49, 64, 65, 96, 97, 128, 129, 200, 256])      # 128: the most rows of a deferred norm
def test_rows_form_in_a_model(gpu, hidden, norm, n):
    """Its epilogues: rows of a deferred norm's consumer, residuals that carry the next norm and plain ones, in steps and short prompts, against the fp32 mode."""
    family = "llama" if norm == "rmsnorm" else "gpt2"
    cfg = gpu.synth.tiny_config(family, hidden=hidden, num_heads=hidden // 64, num_kv_heads=hidden // (256 if family == "llama" else 64), head_dim=64, ffn_dim=hidden, max_seq_len=64)
    w = gpu.synth.make_weights(cfg, seed=4, scale=0.02)
    tok, ids, got = np.random.default_rng(n).integers(0, cfg["vocab_size"], (3, n)).tolist(), list(range(n)), {}
    old = gpu.lib().nvl_set_tuning(46, 2)
    try:
        for precision in ("bf16", "f32"):
            m = gpu.HipTransformerModel(cfg, w, precision=precision, max_seqs=n, max_batch_tokens=512)
            for i in ids:
                m.seq_reset(i)
            got[precision] = [np.asarray(m.forward_batch(ids, [[t] for t in row], [p] * n)[0]) for p, row in enumerate(tok)]
            m.seq_reset(0)
            got[precision].append(np.asarray(m.forward_batch([0], [(tok[0] + tok[1])[:min(n, 64)]], [0])[0]))
            m.close()
    finally:
        gpu.lib().nvl_set_tuning(46, old)
    assert all(rel_err(a, b) <= TOL for a, b in zip(got["bf16"], got["f32"]))
