"""Rows of x near the smallest f32 values through the GEMMs on fp16 activations: their power-of-two scale stays finite."""
import numpy as np
import pytest

from coachwhip_amd import formats as F
from coachwhip_amd import ops, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SCALES = (2.0 ** -110, 2.0 ** -112, 2.0 ** -114, 2.0 ** -120, 2.0 ** -125)


def _rows(m, k, rng):
    x = rng.standard_normal((m, k)).astype(np.float32)
    for i, s in enumerate(SCALES):
        x[-1 - i] *= np.float32(s)
    x[-1, ::3] = 0
    return x


def _check(got, x, w):
    want = x.astype(np.float64) @ w.T
    for t in range(len(x)):
        # the GEMMs' gate on fp16 activations; the smallest outputs step by 2^-149
        assert np.linalg.norm(got[t] - want[t]) <= 1e-3 * np.linalg.norm(want[t]) + 2.0 ** -148 * np.sqrt(want.shape[1]), t


# k and m on both sides of the few-row GEMM's choice between f32 and packed rows (2 to 16 rows), and 40 rows
@pytest.mark.parametrize("k,m", [(4096, 8), (4096, 9), (4352, 6), (8192, 16), (768, 40)])
def test_q4k(k, m, monkeypatch):
    monkeypatch.setenv("CWMOE_MM_MIN_ROWS", "1")
    rng = np.random.default_rng(k + m)
    raw = synth.random_blocks(F.Q4_K, 48 * k, rng)
    x = _rows(m, k, rng)
    got = ops.QMatMul(ops.QTensor.from_blocks(raw, F.Q4_K, (48, k))).forward(ops.to_device(x)).cpu().numpy()
    _check(got, x, O.dequantize(F.Q4_K, raw, 48 * k).reshape(48, k).astype(np.float64))


@pytest.mark.parametrize("dtype", [F.Q8_0, F.Q2_K, F.IQ2_XXS, F.IQ2_S, F.IQ3_XXS, F.IQ3_S, F.IQ4_XS, F.MXFP4], ids=lambda d: F.NAMES[d])
def test_other_formats(dtype, monkeypatch):
    monkeypatch.setenv("CWMOE_MM_MIN_ROWS", "1")
    rng = np.random.default_rng(dtype)
    n, k = 130, 768
    raw = synth.random_blocks(dtype, n * k, rng)
    x = _rows(21, k, rng)
    got = ops.QMatMul(ops.QTensor.from_blocks(raw, dtype, (n, k))).forward(ops.to_device(x)).cpu().numpy()
    _check(got, x, O.dequantize(dtype, raw, n * k).reshape(n, k).astype(np.float64))
