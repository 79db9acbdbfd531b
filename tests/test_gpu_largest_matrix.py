"""Dense products of the largest matrices that the GEMM takes: the last bytes below 4 GiB, off 16-byte alignment."""
import numpy as np
import pytest
import torch

from coachwhip_amd import formats as F
from coachwhip_amd import ops
from oracle import oracle as O

pytestmark = pytest.mark.gpu


# n * row bytes = 2^32 - 1 and 2^32 - 4
@pytest.mark.parametrize("dtype,n,k,first", [(F.MXFP4, 252645135, 32, [121]), (F.IQ2_XXS, 65075262, 256, [0, 32])], ids=["mxfp4", "iq2_xxs"])
def test_last_bytes_below_4_gib(dtype, n, k, first, monkeypatch):
    monkeypatch.setenv("CWMOE_MM_MIN_ROWS", "8")
    size = n * F.row_bytes(dtype, k)
    assert 2 ** 32 - 16 < size < 2 ** 32
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    raw = torch.empty(size + 6, dtype=torch.uint8, device="cuda")[6:]
    raw.random_(generator=gen)
    rows = raw.view(n, -1)
    for i, b in enumerate(first):  # the block's scale: 2^-6, 2^-7
        rows[:, i] = b
    x = np.random.default_rng(n).standard_normal((8, k)).astype(np.float32)
    y = ops.QMatMul(ops.QTensor(raw, dtype, (n, k))).forward(ops.to_device(x))
    for lo, hi in ((0, 300), (n // 2 - 7, n // 2 + 300), (n - 300, n)):
        w = O.dequantize(dtype, rows[lo:hi].cpu().numpy().reshape(-1), (hi - lo) * k).reshape(-1, k).astype(np.float64)
        assert O.rel_l2(y[:, lo:hi].cpu().numpy(), x.astype(np.float64) @ w.T) <= 1e-3  # fp16 activations
