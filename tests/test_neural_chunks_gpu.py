"""The learned shader's gradient, evaluation and training at record counts on either side of their chunks (64 records,
1,024 blocks of them), against the numpy network."""
import ctypes

import numpy as np
import pytest

from oracle import nn_ref as nn
from softglrender_amd import _lib

from .test_neural_gpu import _random_params, _synthetic_records

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 64, 65, 4097, 70_001])
def test_gradient_and_evaluation_match_numpy(renderer, n):
    rec, p = _synthetic_records(n, 5 + n), _random_params(6)
    print(f"[gpu] gradient of {n} records", flush=True)
    renderer.neural_records(n)
    renderer.neural_write_records(0, rec)
    renderer.neural_set_weights(p)
    g, loss = renderer.neural_gradient(0, n)
    x, t = nn.features(rec), rec[:, nn.REC_TARGET:nn.REC_TARGET + 3]
    gw, lw = nn.gradient(p.astype(np.float64), x, t, bf=True)
    # FP32 sums of n products of bf16 values, and the odd bf16 operand one ulp apart (2^-8 of one of n records'
    # contributions; the sine features differ in the last bits of their float values)
    assert abs(loss - lw) <= 1e-3 * lw / np.sqrt(n) + 1e-4 * lw
    assert np.linalg.norm(g - gw) <= (1e-2 / np.sqrt(n) + 1e-4) * np.linalg.norm(gw)
    net, plain, out = renderer.neural_evaluate(0, n, outputs=True)
    y, _ = nn.forward(p.astype(np.float64), x, bf=True)
    assert np.abs(out - y).mean() < 1e-3 / np.sqrt(n) + 1e-5
    err = np.abs(np.clip(out, 0, 1).astype(np.float64) - t) * 255
    assert net["samples"] == n
    # the device's errors are floats of up to 255: 2^-24 of that each
    assert abs(net["mean"] - err.mean()) <= 1e-4 and abs(net["max"] - err.max()) <= 1e-3
    assert plain["mean"] == 0.0 and plain["max"] == 0.0


def test_training_step_is_adam_on_the_gradient(renderer):
    """One step over a batch that covers every record about once moves each weight by the learning rate against its
    gradient's sign (Adam's first step), and repeats bit for bit."""
    n = 300
    rec, p = _synthetic_records(n, 8), _random_params(9)
    renderer.neural_records(n)
    renderer.neural_write_records(0, rec)
    runs = []
    for _ in range(2):
        renderer.neural_set_weights(p)
        loss = renderer.neural_train(0, n, 1, batch=8192, lr_start=1e-3, lr_end=1e-3, seed=5)
        runs.append((renderer.neural_get_weights(), loss))
    assert np.array_equal(runs[0][0], runs[1][0]) and np.array_equal(runs[0][1], runs[1][1])
    step = runs[0][0].astype(np.float64) - p
    assert np.abs(step).max() <= 1.01e-3
    renderer.neural_set_weights(p)
    g, _ = renderer.neural_gradient(0, n)
    big = np.abs(g) > 0.3 * np.abs(g).max()  # far from zero: a resampled batch keeps their sign
    assert big.sum() > 5 and np.all(np.sign(step[big]) == -np.sign(g[big]))
    assert np.allclose(np.abs(step[big]), 1e-3, rtol=1e-2)


def _free_memory():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert _lib.load().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0  # librhip's own HIP runtime
    return free.value


def test_large_calls_give_their_buffers_back(renderer):
    """The outputs of 3M records (36 MB) are the call's own memory: after it, at most what a device may keep is gone."""
    n = 3_000_000
    print(f"[gpu] evaluation of {n} records", flush=True)
    renderer.neural_records(n)
    renderer.neural_write_records(0, np.tile(_synthetic_records(1000, 2), (n // 1000, 1)))
    renderer.neural_set_weights(_random_params(6))
    _, _, few = renderer.neural_evaluate(0, 1000, outputs=True)
    before = _free_memory()
    for _ in range(2):
        _, _, out = renderer.neural_evaluate(0, n, outputs=True)
        assert np.array_equal(out[:1000], few) and np.array_equal(out[-1000:], few)
        assert before - _free_memory() <= 16 << 20
