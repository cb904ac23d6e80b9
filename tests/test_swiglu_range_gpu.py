"""SwiGLU into bf16 over the gates' whole range, value by value, against 64 bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 24, 200, 1000])          # decode forms, 64-row groups or tiles, tiles
def test_every_gate(gpu, rows):
    """silu(g) 2^119 for g between -100 and 100: the smallest results of silu alone would be 1e-42 .. 1e-36."""
    g = np.concatenate([np.arange(-100, 100, 0.5), [-0.0, 1e-3, -1e-3, 3e-5, -127 / 128]])
    F = 448
    g = np.concatenate([g, np.full(F - len(g), 7.0)]).astype(np.float32)
    g = gpu.synth.round_bf16(g)
    x, w1 = np.zeros((rows, 64), np.float32), np.zeros((64, 2 * F), np.float32)
    x[:, 0] = x[:, 1] = 1.0
    w1[0, :F], w1[1, F:] = g, 2.0 ** 119
    g = g.astype(np.float64)
    want = g / (1.0 + np.exp(-g)) * 2.0 ** 119
    got = []
    for part in range(F // 64):          # (the result has as many columns as the operand: 64 of the F at a time)
        w2 = np.zeros((F, 64), np.float32)
        w2[part * 64:part * 64 + 64] = np.eye(64)
        got.append(gpu.ops.feed_forward(x, w1, None, w2, None, True, precision="bf16"))
    got = np.concatenate(got, axis=1).astype(np.float64)
    # bf16 (eight bits) rounds by up to 2^-8 of the value; exp of g, off by half a place of g log2(e) in fp32, by 2^-24 |g| more; e < 2^128 is the end of fp32: beyond it zero
    live = g > -88.7
    off = (np.abs(got - want) > np.abs(want) * (2.0 ** -8 + 1e-4)).any(axis=0) & live
    assert not off.any(), g[off]
    assert (np.abs(got[:, ~live]) <= np.abs(want[~live])).all()
