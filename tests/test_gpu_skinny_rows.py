"""Dense Q4_K at 2..16 rows of x: the GEMM of few rows, which takes x as f32 where it is small
(up to 4,096 rows of W, 8 rows of x of 4,096 columns) and packed above."""
import numpy as np
import pytest

from coachwhip_amd import formats as F
from coachwhip_amd import ops, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


# one super-block, odd counts, both sides of each block size (512, 1,024, 2,048 and 4,096 columns), the longest row
@pytest.mark.parametrize("k", [256, 512, 768, 1280, 2048, 2304, 4096, 4352, 8192])
@pytest.mark.parametrize("m", [2, 8, 9, 16])
def test_rows_of_any_range(k, m, monkeypatch):
    monkeypatch.setenv("CWMOE_MM_MIN_ROWS", "1")
    rng = np.random.default_rng(k + m)
    n = 33
    raw = synth.random_blocks(F.Q4_K, n * k, rng)
    w = O.dequantize(F.Q4_K, raw, n * k).reshape(n, k).astype(np.float64)
    plain = rng.standard_normal((m, k)).astype(np.float32)
    # a range of its own for each super-block, zeros among them; the last row near the smallest f32 values
    wide = plain * np.repeat(np.ldexp(1.0, rng.integers(-60, 30, (m, k // 256))), 256, axis=1).astype(np.float32)
    wide[0, :256] = 0
    wide[-1] = plain[-1] * np.float32(2.0**-125)
    # (packed rows have one scale each, no finer than the row's largest value)
    block = 512 if k <= 512 else 1024 if k <= 1024 else 2048 if k <= 2048 else 4096
    for x in (plain, wide) if k <= 4096 and m * block <= 32768 else (plain,):
        got = ops.QMatMul(ops.QTensor.from_blocks(raw, F.Q4_K, (n, k))).forward(ops.to_device(x)).cpu().numpy()
        x = x.astype(np.float64)
        # fp16 holds an activation to 2^-11 of itself (values far below their super-block's largest to 2^-39 of
        # that); the f32 sums take less than as much again. The smallest outputs step by 2^-149.
        mag = np.repeat(np.abs(x).reshape(m, -1, 256).max(axis=2), 256, axis=1)
        tol = 2.0**-10 * (np.abs(x) @ np.abs(w).T) + 2.0**-38 * (mag @ np.abs(w).T) + 2.0**-140
        assert np.all(np.abs(got - x @ w.T) <= tol)
