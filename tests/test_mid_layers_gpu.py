"""Projections of 65 .. 512 rows on their own kernel (gemm.h gemm_mid_bf16_kernel) in models described by a list of layers: each epilogue that these have,
K whole and in parts, ragged rows and column ranges.  Forced, for these models are narrower than the rule asks for."""
import numpy as np
import pytest

import bolinex_models as BM
import bolinex_oracle as BO
import lufazen_models as LM
import lufazen_oracle as LO
import medulorn_models as MM
import medulorn_oracle as MO
import potuzen_models as PM
import potuzen_oracle as PO
from layered_helpers import build, err

pytestmark = pytest.mark.gpu
ONE = 0.03              # a single bf16 layer against the plain restatement, as in the tests of these models

CASES = {       # K of 640 or 384 and more: two to five parts
    "gated-grouped": (BM, BO, BM.config([BM.attention(heads=10, kv_heads=2, dim=40, vdim=56, mlp=BM.dense(600))], width=600, vocab=130)),           # EPI_GROUPED, RELU2, GELU_TOK
    "normed-grouped": (MM, MO, MM.config([MM.attention(heads=8, kv_heads=2, dim=64, vdim=72, turn=MM.rot(64), mlp=MM.dense(500))], width=600, vocab=130)),     # EPI_GROUPED_RAW, REGLU
    "beside": (MM, MO, MM.config([MM.parallel(heads=6, kv_heads=2, dim=64, vdim=64, turn=MM.rot(64), heads2=5, dim2=20, vdim2=100, mlp=MM.dense(390))], width=600, vocab=130)),
    "latent": (LM, LO, LM.config([LM.latent(heads=5, dim=72, vdim=100, q_rank=500, kv_rank=400, ff=600)], width=600, vocab=130)),                     # clamped gate | up
    "delta": (LM, LO, LM.config([LM.delta(heads=6, kv_heads=3, dim=40, vdim=72, ff=600)], width=600, vocab=130)),
    "gla": (PM, PO, PM.config([PM.gla(heads=5, dim=36, vdim=100, ff=600)], width=600, vocab=130)),                                                 # GEGLU
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("rows", [70, 97, 200])
def test_prompts(gpu, tmp_path, name, rows):
    models, oracle, cfg = CASES[name]
    w = models.weights(cfg, 7)
    tok = np.random.default_rng(rows).integers(0, 130, rows).tolist()
    want = oracle.forward(cfg, w, tok)
    m = build(gpu, tmp_path, cfg, w, "bf16")
    lib, got = gpu.lib(), {}
    for form, parts in ((0, 0), (2, 0), (2, 1), (2, 2), (2, 3)):
        old = [(k, lib.nvl_set_tuning(k, v)) for k, v in ((38, form), (39, parts))]
        try:
            m.seq_open(0)
            got[form, parts] = m.forward_rows([0], [tok], [0], range(rows))[0]
            m.seq_close(0)
        finally:
            for k, v in old:
                lib.nvl_set_tuning(k, v)
    m.close()
    assert not any(np.array_equal(v, got[0, 0]) for k, v in got.items() if k != (0, 0))      # (another order of the sums)
    errs = {k: err(v, want, "bf16") for k, v in got.items()}
    assert max(errs.values()) < ONE, errs
