"""The shared expert with Q5_K and Q6_K matrices: on the workspace it asks for, and on less (the matvecs)."""
import ctypes

import numpy as np
import pytest
import torch

import coachwhip_amd as cw
from coachwhip_amd import _lib
from coachwhip_amd import formats as F
from coachwhip_amd import ops, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _layer(dtypes, hidden, inter, rng):
    shapes = [(inter, hidden)] * 2 + [(hidden, inter)]
    raw = [synth.random_blocks(t, n * k, rng) for t, (n, k) in zip(dtypes, shapes)]
    gate_inp = (rng.standard_normal(hidden) * 0.02).astype(np.float32)
    se = ops.SharedExpert(*[ops.QTensor.from_blocks(r, t, s) for r, t, s in zip(raw, dtypes, shapes)], ops.to_device(gate_inp))
    w = [O.dequantize(t, r, n * k).reshape(n, k).astype(np.float64) for t, r, (n, k) in zip(dtypes, raw, shapes)]

    def exact(x):
        x = x.astype(np.float64)
        g, u = x @ w[0].T, x @ w[1].T
        with np.errstate(over="ignore"):
            h = g / (1 + np.exp(-g)) * u
        return h @ w[2].T / (1 + np.exp(-(x @ gate_inp.astype(np.float64))))[:, None]

    return se, exact


def _size(se, tokens):
    return cw.lib().cw_shared_expert_workspace_size(ctypes.byref(se.desc), tokens)


def _call(se, x, ws_bytes):
    ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device="cuda")
    out = torch.empty_like(x)
    rc = cw.lib().cw_shared_expert(ctypes.byref(se.desc), _p(x), x.shape[0], _p(out), 0, _p(ws), ws_bytes, None)
    torch.cuda.synchronize()
    return rc, out.cpu().numpy()


def _rows_bytes(hidden, inter, tokens):
    """Everything but the matmuls' region."""
    return sum(-(-b // 256) * 256 for b in (4 * tokens * inter, 4 * tokens * inter, 4 * tokens * hidden, 4 * tokens))


# a product is f32-accurate: an f32 sum of k products errs by a few times 2^-24, three follow one another
REL_L2_F32, REL_L2_F16 = 2e-6, 1e-3


@pytest.mark.parametrize("dtypes,least", [((F.Q6_K, F.Q6_K, F.Q6_K), "rows"), ((F.Q5_K, F.Q5_K, F.Q6_K), "rows"), ((F.Q8_0, F.Q5_K, F.Q6_K), "mfma")],
                         ids=["q6", "q5q6", "q8q5q6"])
def test_less_workspace_takes_the_matvecs(dtypes, least, monkeypatch):
    monkeypatch.delenv("CWMOE_MM_MIN_ROWS", raising=False)
    rng = np.random.default_rng(dtypes[0])
    hidden, inter, tokens = 2048, 768, 60
    se, exact = _layer(dtypes, hidden, inter, rng)
    x = rng.standard_normal((tokens, hidden)).astype(np.float32)
    want, xd = exact(x), ops.to_device(x)
    full, rows = _size(se, tokens), _rows_bytes(hidden, inter, tokens)
    if least == "mfma":  # the fp16 GEMM of gate has no other path
        rows += -(-cw.lib().cw_qmatmul_workspace_size(F.Q8_0, inter, hidden, tokens) // 256) * 256
    assert full > rows
    got = {}
    for name, size in (("full", full), ("short", full - 256), ("least", rows)):
        rc, got[name] = _call(se, xd, size)
        assert rc == _lib.CW_OK, (name, cw.lib().cw_last_error())
        assert O.rel_l2(got[name], want) <= (REL_L2_F16 if least == "mfma" else REL_L2_F32), name
    assert not np.array_equal(got["full"], got["least"])
    rc, _ = _call(se, xd, rows - 256)
    assert rc == _lib.CW_EINVAL and b"workspace" in cw.lib().cw_last_error()


def test_workspace_of_a_larger_batch_serves_a_smaller_one(monkeypatch):
    """161 rows need less than 160: the products are split over fewer parts."""
    monkeypatch.delenv("CWMOE_MM_MIN_ROWS", raising=False)
    rng = np.random.default_rng(160)
    se, exact = _layer((F.Q6_K,) * 3, 4096, 4096, rng)
    x = rng.standard_normal((160, 4096)).astype(np.float32)
    assert _size(se, 161) < _size(se, 160)
    rc, got = _call(se, ops.to_device(x), _size(se, 161))
    assert rc == _lib.CW_OK and O.rel_l2(got, exact(x)) <= REL_L2_F32
