"""Q5_K and Q6_K GEMMs at f32 accuracy (activations as two fp16 terms, exact weight codes): dense
products and MoE layers, against the f64 oracle and the f32 matvec they stand in for."""
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


def _banks(w, experts):
    shapes = [(w.inter, w.hidden)] * 2 + [(w.hidden, w.inter)]
    return [ops.ExpertBank.from_blocks(w.host[m], w.dtypes[m], *s, experts) for m, s in enumerate(shapes)]


def _call(layer, x, logits, entry="workspace", ws_bytes=None):
    """cw_moe_layer with a workspace of ws_bytes (what it asks for by default), or the entry point without one."""
    L, (tokens, hidden) = cw.lib(), x.shape
    out = torch.empty((tokens, hidden), device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    if entry == "noalloc":
        _lib.check(L.cw_moe_layer_noalloc(ctypes.byref(layer.desc), p(x), p(logits), tokens, p(out), None, None, None, None))
    else:
        need = L.cw_moe_workspace_size(ctypes.byref(layer.desc), tokens) if ws_bytes is None else ws_bytes
        ws = torch.zeros(need, dtype=torch.uint8, device="cuda")
        _lib.check(L.cw_moe_layer(ctypes.byref(layer.desc), p(x), p(logits), tokens, p(out), None, None, None, p(ws), need, None))
    torch.cuda.synchronize()
    return out.cpu().numpy()


# no override: every token picks all four experts, 264 million weights beyond the distinct ones at 15 tokens
# and 246 million at 14 of the second shape
@pytest.mark.parametrize("pair", [(F.Q4_K, F.Q4_K), (F.Q8_0, F.Q8_0), (F.Q4_K, F.Q8_0), (F.Q8_0, F.Q4_K), (F.Q4_K, F.Q6_K)],
                         ids=lambda p: F.NAMES[p[0]] + "-" + F.NAMES[p[1]])
@pytest.mark.parametrize("tokens,hidden,inter", [(15, 1024, 1536), (14, 2048, 768)])
def test_layer_by_the_rule_and_with_less_workspace(pair, tokens, hidden, inter, monkeypatch):
    monkeypatch.delenv("CWMOE_PREFILL_MIN_TOKENS", raising=False)
    rng = np.random.default_rng(tokens + inter)
    w = synth.moe_weights(4, 4, hidden, inter, (pair[0],) + pair, rng)
    layer = ops.MoeLayer(*_banks(w, 4), n_experts=4, top_k=4)
    x, logits = rng.standard_normal((tokens, hidden)).astype(np.float32), rng.standard_normal((tokens, 4)).astype(np.float32)
    want = O.moe_layer(w, x, logits)[0]
    x, logits = ops.to_device(x), ops.to_device(logits)
    gemm, noalloc = _call(layer, x, logits), _call(layer, x, logits, "noalloc")
    matvec = cw.lib().cw_moe_workspace_size(ctypes.byref(layer.desc), 4)  # below the line: the matvecs' layout
    matvec += 3 * 1024 + (tokens - 4) * 4 * 4 * inter                    # for all tokens
    less = _call(layer, x, logits, ws_bytes=matvec)
    monkeypatch.setenv("CWMOE_PREFILL_MIN_TOKENS", "1000000")
    plain = _call(layer, x, logits)
    assert np.array_equal(gemm.view(np.uint32), noalloc.view(np.uint32))  # the GEMMs' layout fits its array
    assert np.array_equal(less.view(np.uint32), plain.view(np.uint32)) and not np.array_equal(gemm, plain)
    assert O.rel_l2(gemm, want) <= min(2 * REL_L2, 2 * O.rel_l2(plain, want))


def test_noalloc_layer_whose_gemms_do_not_fit(monkeypatch):
    """110 tokens of 8 picks: 2.2 MB for the matvecs, 15 MB for the GEMMs."""
    monkeypatch.delenv("CWMOE_PREFILL_MIN_TOKENS", raising=False)
    rng = np.random.default_rng(9)
    w = synth.moe_weights(8, 8, 2816, 512, (F.Q4_K, F.Q4_K, F.Q6_K), rng)
    layer = ops.MoeLayer(*_banks(w, 8), n_experts=8, top_k=8)
    x, logits = rng.standard_normal((110, 2816)).astype(np.float32), rng.standard_normal((110, 8)).astype(np.float32)
    want = O.moe_layer(w, x, logits)[0]
    x, logits = ops.to_device(x), ops.to_device(logits)
    assert cw.lib().cw_moe_workspace_size(ctypes.byref(layer.desc), 110) > 8 << 20
    gemm, noalloc = _call(layer, x, logits), _call(layer, x, logits, "noalloc")
    assert not np.array_equal(gemm, noalloc)
    for got in (gemm, noalloc):
        assert O.rel_l2(got, want) <= 2 * REL_L2


@pytest.mark.parametrize("dtype", [F.Q5_K, F.Q6_K])
def test_dense_by_the_rule_and_without_workspace(dtype, monkeypatch):
    monkeypatch.delenv("CWMOE_MM_MIN_ROWS", raising=False)
    rng = np.random.default_rng(dtype)
    n, k, m = 640, 2048, 40  # 248 million of 215 needed
    raw = synth.random_blocks(dtype, n * k, rng)
    x = rng.standard_normal((m, k)).astype(np.float32)
    want = O.qmatmul_f64(dtype, raw, n, k, x)
    L, w, xd = cw.lib(), ops.to_device(raw), ops.to_device(x)
    p = lambda t: None if t is None else ctypes.c_void_p(t.data_ptr())  # noqa: E731
    need, got = L.cw_qmatmul_workspace_size(dtype, n, k, m), {}
    assert need > 0
    for name, size in (("gemm", need), ("short", need - 1), ("none", 0)):
        ws = torch.empty(size, dtype=torch.uint8, device="cuda") if size else None
        y = torch.empty((m, n), device="cuda")
        _lib.check(L.cw_qmatmul(dtype, p(w), n, k, p(xd), m, p(y), p(ws), size, None))
        torch.cuda.synchronize()
        got[name] = y.cpu().numpy()
    monkeypatch.setenv("CWMOE_MM_MIN_ROWS", "1000000")
    plain = ops.QMatMul(ops.QTensor.from_blocks(raw, dtype, (n, k))).forward(xd).cpu().numpy()
    assert np.array_equal(got["short"], plain) and np.array_equal(got["none"], plain) and not np.array_equal(got["gemm"], plain)
    assert O.rel_l2(got["gemm"], want) <= min(REL_L2, 2 * O.rel_l2(plain, want))


def _outlier_blocks(dtype, n, k, rng):
    """Weights that are 0 where the test puts large activations: super-block 0 (its scale), and column 300 (Q6_K:
    the code 32) or the sub-block around it (Q5_K: its scale and minimum)."""
    raw = synth.random_blocks(dtype, n * k, rng).reshape(n, k // 256, -1).copy()
    o = F.D_OFFSET[dtype]
    raw[:, 0, o:o + (4 if dtype == F.Q5_K else 2)] = 0
    if dtype == F.Q5_K:  # sub-block 1: the low 6 bits of scale bytes 1 and 5
        raw[:, 1, 5] &= 0xC0
        raw[:, 1, 9] &= 0xC0
    else:  # quadrant 1, weight 12: the low nibble of ql[44], bits 2 and 3 of qh[12]
        raw[:, 1, 44] &= 0xF0
        raw[:, 1, 128 + 12] = raw[:, 1, 128 + 12] & 0xF3 | 2 << 2
    return raw.reshape(-1)


@pytest.mark.parametrize("dtype", [F.Q5_K, F.Q6_K])
def test_dense_outliers_against_zero_weights(dtype, monkeypatch):
    """Large activations whose weights are 0 do not cost the others their bits: each output row is held to the f32
    bar by itself, as the matvec's is."""
    rng = np.random.default_rng(dtype)
    n, k, m = 80, 1024, 24
    raw = _outlier_blocks(dtype, n, k, rng)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[0, 7] = 2.0 ** 25
    x[1, 200] = -(2.0 ** 60)
    x[2, :256] *= np.float32(1e30)
    x[3, 300] = 2.0 ** 25
    x[4, 300] = -1e7
    x[5, 512:] *= np.float32(1e-20)     # super-blocks of their own size
    x[5, 300] = 3e4
    want = O.qmatmul_f64(dtype, raw, n, k, x)
    got, plain = (_matmul(raw, dtype, n, k, x, monkeypatch, r) for r in (1, 1000000))
    for t in range(m):
        err, ref = O.rel_l2(got[t], want[t]), O.rel_l2(plain[t], want[t])
        assert err <= max(2 * ref, REL_L2), (t, err, ref)


@pytest.mark.parametrize("dtype", [F.Q5_K, F.Q6_K])
def test_dense_infinities_and_nans(dtype, monkeypatch):
    """An infinite activation gives the infinity of its weight's sign, or a NaN where the weight is 0; a NaN stays one;
    other rows do not see them."""
    rng = np.random.default_rng(dtype + 1)
    n, k, m = 160, 1024, 20
    raw = _outlier_blocks(dtype, n, k, rng)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[3, 700], x[4, 300], x[5, 9], x[6, 1023], x[7, 400] = np.inf, np.inf, -np.inf, -np.inf, np.nan
    x[8, 600], x[8, 601], x[9, 600], x[9, 900] = np.inf, np.nan, np.inf, -np.inf
    with np.errstate(invalid="ignore"):
        want = O.qmatmul_f64(dtype, raw, n, k, x)
    got = _matmul(raw, dtype, n, k, x, monkeypatch, 1)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.isnan(want[7]).all() and np.isnan(want[4]).all()
    inf = np.isinf(want)
    assert inf[3].any() and inf[6].any() and np.array_equal(got[inf], want[inf].astype(np.float32))
    live = np.isfinite(want).all(1)
    assert live.sum() == m - 7 and O.rel_l2(got[live], want[live]) <= REL_L2


# rows of Q8_0 that end inside a stage, beside whole super-blocks of the other format
@pytest.mark.parametrize("pair,tokens,hidden,inter", [((F.Q8_0, F.Q6_K), 33, 544, 256), ((F.Q6_K, F.Q8_0), 90, 512, 288), ((F.Q8_0, F.Q5_K), 20, 32, 512)],
                         ids=str)
def test_layer_of_ragged_rows(pair, tokens, hidden, inter, monkeypatch):
    monkeypatch.setenv("CWMOE_PREFILL_MIN_TOKENS", "16")
    rng = np.random.default_rng(hidden)
    w = synth.moe_weights(6, 3, hidden, inter, (pair[0],) + pair, rng)
    layer = ops.MoeLayer(*_banks(w, 6), n_experts=6, top_k=3)
    x, logits = rng.standard_normal((tokens, hidden)).astype(np.float32), rng.standard_normal((tokens, 6)).astype(np.float32)
    want = O.moe_layer(w, x, logits)[0]
    assert O.rel_l2(_call(layer, ops.to_device(x), ops.to_device(logits)), want) <= 2 * REL_L2


@pytest.mark.parametrize("pair", [(F.Q4_K, F.Q6_K), (F.Q5_K, F.Q8_0), (F.Q6_K, F.Q5_K)], ids=lambda p: F.NAMES[p[0]] + "-" + F.NAMES[p[1]])
def test_layer_with_biases_padding_and_slots(pair, monkeypatch):
    """The clamped SwiGLU with biases per expert, hidden rows padded with zeros, a permuted slot table, and a
    slot past the bank (NaN rows)."""
    monkeypatch.setenv("CWMOE_PREFILL_MIN_TOKENS", "16")
    rng = np.random.default_rng(pair[0])
    experts, slots, top_k, hidden, inter, pad, tokens = 24, 12, 4, 512, 512, 768, 61
    w = synth.moe_weights(experts, top_k, hidden, inter, (pair[0],) + pair, rng, n_slots=slots, act=1, pad=pad)
    w.bias = [20 * b for b in w.bias]
    shapes = [(inter, hidden)] * 2 + [(hidden, pad)]
    banks = [ops.ExpertBank.from_blocks(w.host[m], w.dtypes[m], *s, slots) for m, s in enumerate(shapes)]
    table = np.full(experts, 0xFFFFFFFF, np.uint32)
    resident = rng.choice(experts, slots, replace=False)
    table[resident] = rng.permutation(slots)
    # (x small: the clamp leaves most of the gates and ups to their weights)
    x = (rng.standard_normal((tokens, hidden)) * 2.0 ** -8).astype(np.float32)
    logits = rng.standard_normal((tokens, experts)).astype(np.float32)
    logits[:, table == 0xFFFFFFFF] -= np.float32(1e30)
    want, wids, _, _ = O.moe_layer(w, x, logits, slot_table=table, n_slots=slots)
    act = ops.ExpertAct.clamped_swiglu(w.alpha, w.limit, *[ops.to_device(b) for b in w.bias], pad=pad)
    xd, ld = ops.to_device(x), ops.to_device(logits)

    def run(tab):
        layer = ops.MoeLayer(*banks, n_experts=experts, top_k=top_k, act=act, slot_table=ops.to_device(tab))
        out, ids, _ = layer.forward(xd, ld)
        assert np.array_equal(ids.cpu().numpy().view(np.uint32), wids)
        return out.cpu().numpy()

    assert O.rel_l2(run(table), want) <= 2 * REL_L2
    bad = wids[0, 0]
    table[bad] = slots
    out = run(table)
    hit = (wids == bad).any(1)
    assert np.isnan(out[hit]).all() and O.rel_l2(out[~hit], want[~hit]) <= 2 * REL_L2
