"""Dense MXFP4 at the row counts where the GEMM's tiles change (pick blocks of 16, tiles of 80), with rows of whole and
ragged stages of K, split and not, against the f64 product."""
import numpy as np
import pytest

from coachwhip_amd import formats as F
from coachwhip_amd import ops, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


# k of 1 to 40 blocks of 32: part of one part of a stage, ends in its first and second half, one stage, many
@pytest.mark.parametrize("n,k", [(130, 32), (64, 128), (127, 160), (129, 256), (40, 288), (300, 1152), (96, 1280), (256, 8192)])
@pytest.mark.parametrize("m", [1, 16, 17, 33, 48, 64, 65, 80, 81, 115])
def test_dense(n, k, m, monkeypatch):
    monkeypatch.setenv("CWMOE_MM_MIN_ROWS", "1")
    rng = np.random.default_rng(n + k + m)
    raw = synth.random_blocks(F.MXFP4, n * k, rng)
    x = rng.standard_normal((m, k)).astype(np.float32)
    got = ops.QMatMul(ops.QTensor.from_blocks(raw, F.MXFP4, (n, k))).forward(ops.to_device(x)).cpu().numpy()
    want = x.astype(np.float64) @ O.dequantize(F.MXFP4, raw, n * k).reshape(n, k).astype(np.float64).T
    assert O.rel_l2(got, want) <= 1e-3  # fp16 activations: 2^-11 per value at most
