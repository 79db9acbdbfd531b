"""Q5_K and Q6_K GEMMs at f32 accuracy (activations as two fp16 terms, exact weight codes): dense
products and MoE layers, against the f64 oracle and the f32 matvec they stand in for."""
import numpy as np
import pytest
import torch

from coachwhip_amd import formats as F
from coachwhip_amd import ops, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# An f32 sum of k products errs by a few times 2^-24 (the matvec measures 1.2e-7 to 2.5e-7); two fp16 terms
# add 2^-23 / sqrt(3) per activation at most. Both stay below 4e-7.
REL_L2 = 4e-7


def _matmul(raw, dtype, n, k, x, monkeypatch, rows):
    monkeypatch.setenv("CWMOE_MM_MIN_ROWS", str(rows))
    return ops.QMatMul(ops.QTensor.from_blocks(raw, dtype, (n, k))).forward(ops.to_device(x)).cpu().numpy()


# rows at the edges of the 16-row blocks and 80-row tiles; W rows around the 128-row items; one
# super-block, an odd count, and rows long enough to be split
@pytest.mark.parametrize("dtype", [F.Q5_K, F.Q6_K])
@pytest.mark.parametrize("n,k,m", [(128, 256, 8), (127, 768, 16), (129, 1024, 17), (16, 256, 80), (300, 2048, 81), (513, 8192, 97),
                                   (1, 512, 33), (2000, 2816, 165)])
def test_dense(dtype, n, k, m, monkeypatch):
    rng = np.random.default_rng(n + k + m)
    raw = synth.random_blocks(dtype, n * k, rng)
    x = rng.standard_normal((m, k)).astype(np.float32)
    want = O.qmatmul_f64(dtype, raw, n, k, x)
    got = _matmul(raw, dtype, n, k, x, monkeypatch, 1)
    plain = _matmul(raw, dtype, n, k, x, monkeypatch, 1000000)
    assert not np.array_equal(got, plain)  # the GEMM ran
    assert O.rel_l2(got, want) <= min(REL_L2, 2 * O.rel_l2(plain, want))


@pytest.mark.parametrize("dtype", [F.Q5_K, F.Q6_K])
def test_dense_scales_and_activations_at_their_limits(dtype, monkeypatch):
    rng = np.random.default_rng(dtype)
    n, k, m = 96, 1024, 40
    raw = synth.random_blocks(dtype, n * k, rng).reshape(-1, F.type_size(dtype)).copy()
    o = F.D_OFFSET[dtype]
    raw[::3, o:o + 2] = 0                        # d = 0
    raw[1::5, o:o + 2] = [0x01, 0x80]            # smallest negative subnormal d
    if dtype == F.Q6_K:
        raw[2::4, 192:208] = np.tile([0x80, 0x7F], 8)  # sub-block scales -128 and 127
        raw[3::4, 0:192] = np.tile([0x00, 0xFF], 96)   # codes -32 and 31
    raw = raw.reshape(-1)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[0] *= np.float32(1e30)
    x[1] *= np.float32(1e-36)                    # rows of subnormal products
    x[2] = 0
    x[3, 1:] *= np.float32(1e-7)                 # one value far above the others
    want = O.qmatmul_f64(dtype, raw, n, k, x)
    got, plain = (_matmul(raw, dtype, n, k, x, monkeypatch, r) for r in (1, 1000000))
    for t in range(m):
        err, ref = O.rel_l2(got[t], want[t]), O.rel_l2(plain[t], want[t])
        assert err <= max(2 * ref, 4 * REL_L2), (t, err, ref)  # (a single row's sum of 1,024: twice the average)
    x[5, 7], x[6, 9], x[7, 3] = np.inf, np.nan, -np.inf
    got, plain = (_matmul(raw, dtype, n, k, x, monkeypatch, r) for r in (1, 1000000))
    live = np.ones(m, bool)
    live[5:8] = False
    assert np.isfinite(got[live]).all()
    assert np.array_equal(np.isfinite(got[5:8]), np.isfinite(plain[5:8]))


# 16 tokens and up; piles of one pick, of a whole 80-pick tile and of more; mixed formats
@pytest.mark.parametrize("pair", [(F.Q4_K, F.Q6_K), (F.Q5_K, F.Q6_K), (F.Q6_K, F.Q5_K), (F.Q8_0, F.Q6_K), (F.Q5_K, F.Q8_0), (F.Q5_K, F.Q4_K)],
                         ids=lambda p: F.NAMES[p[0]] + "-" + F.NAMES[p[1]])
@pytest.mark.parametrize("tokens,experts,top_k,hidden,inter", [(16, 24, 3, 512, 256), (101, 3, 2, 256, 512), (37, 12, 5, 1280, 768)])
def test_layer(pair, tokens, experts, top_k, hidden, inter, monkeypatch):
    rng = np.random.default_rng(tokens)
    w = synth.moe_weights(experts, top_k, hidden, inter, (pair[0],) + pair, rng)
    banks = [ops.ExpertBank.from_blocks(w.host[m], w.dtypes[m], *s, experts) for m, s in enumerate([(inter, hidden)] * 2 + [(hidden, inter)])]
    x, logits = rng.standard_normal((tokens, hidden)).astype(np.float32), rng.standard_normal((tokens, experts)).astype(np.float32)
    out, err = {}, {}
    want, wids, _, _ = O.moe_layer(w, x, logits)
    for path, rows in (("gemm", "16"), ("matvec", "1000000")):
        monkeypatch.setenv("CWMOE_PREFILL_MIN_TOKENS", rows)
        got, ids, _ = ops.MoeLayer(*banks, n_experts=experts, top_k=top_k).forward(ops.to_device(x), ops.to_device(logits))
        assert np.array_equal(ids.cpu().numpy().view(np.uint32), wids)
        out[path] = got.cpu().numpy()
        err[path] = O.rel_l2(out[path], want)
    assert not np.array_equal(out["gemm"], out["matvec"])
    assert err["gemm"] <= min(2 * REL_L2, 2 * err["matvec"])  # (two products after one another)
