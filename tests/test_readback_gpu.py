"""Logits read back in pieces through the model's pinned memory against the plain copy, which memory that the runtime knows takes."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# one slot that is filled again and again (the ring is sized for max_seqs rows), a few pieces and threads, more pieces than slots, rows with and without padding
@pytest.mark.parametrize("vocab,max_seqs,rows", [(1003, 2, 1), (1003, 2, 200), (65536, 8, 8), (70001, 1, 40), (70001, 5, 5), (70001, 40, 40), (70001, 40, 150)])
def test_pieces_are_the_rows(gpu, vocab, max_seqs, rows):
    cfg = gpu.synth.tiny_config("llama", num_layers=1, vocab_size=vocab)
    m = gpu.HipTransformerModel(cfg, gpu.synth.make_weights(cfg, seed=3, scale=0.05), precision="bf16", max_seqs=max_seqs, max_batch_tokens=256)
    tokens = np.random.default_rng(rows).integers(0, vocab, rows).astype(np.int32)
    args = [np.zeros(1, np.int64), tokens, np.array([rows], np.int32), np.zeros(1, np.int32)]
    ptr = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
    plain = torch.empty(rows, vocab, pin_memory=True)
    m.seq_reset(0)
    assert m.lib.nvl_forward(m.h, 1, *map(ptr, args), gpu._lib.FWD_ALL_LOGITS, C.c_void_p(plain.data_ptr()), None) == 0
    want = plain.numpy().copy()
    for _ in range(2):
        m.seq_reset(0)
        got = np.full(rows * vocab + 2, np.nan, np.float32)[1:]          # (4-byte aligned, a value behind the end)
        am = np.empty(1, np.int32)
        assert m.lib.nvl_forward(m.h, 1, *map(ptr, args), gpu._lib.FWD_ALL_LOGITS, ptr(got), ptr(am)) == 0
        assert np.array_equal(got[:-1].reshape(rows, vocab), want) and np.isnan(got[-1])
        assert am[0] == want[-1].argmax()
    m.close()
