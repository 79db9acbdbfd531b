"""The layer for a few tokens (per-token gate/up and down kernels, f32 activations) at the shapes where
their row splits change, against the f64 oracle at the f32 bar."""
import numpy as np
import pytest
import torch

from coachwhip_amd import formats as F
from coachwhip_amd import ops, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu

REL_L2_F32 = 2e-5


def _layer(w):
    shapes = [(w.inter, w.hidden), (w.inter, w.hidden), (w.hidden, max(w.pad, w.inter))]
    banks = [ops.ExpertBank.from_blocks(w.host[m], w.dtypes[m], *shapes[m], w.n_slots) for m in range(3)]
    act = ops.ExpertAct.silu()
    if w.act:
        act = ops.ExpertAct.clamped_swiglu(w.alpha, w.limit, *[ops.to_device(b) for b in w.bias], pad=w.pad)
    return ops.MoeLayer(*banks, n_experts=w.n_experts, top_k=w.top_k, norm_topk_prob=w.norm, act=act)


# formats x (hidden, inter, top_k, tokens): one sub-block row, 48 and 96 sub-blocks (three per lane), 64, 128 and 256;
# picks below, at and above 8 and 16 (one, two and four per wave of down); rows that leave a ragged last item
@pytest.mark.parametrize("hidden,inter,top_k,tokens", [(256, 256, 3, 2), (1536, 512, 8, 3), (2048, 768, 9, 5), (2816, 256, 2, 15),
                                                        (4096, 256, 17, 2), (8192, 256, 4, 2)])
@pytest.mark.parametrize("pair", [(F.IQ2_XXS, F.IQ2_S), (F.IQ3_S, F.Q4_K), (F.Q4_K, F.Q6_K), (F.Q5_K, F.Q2_K), (F.Q8_0, F.IQ4_XS),
                                  (F.IQ3_XXS, F.Q8_0)], ids=lambda p: F.NAMES[p[0]] + "-" + F.NAMES[p[1]])
def test_few_tokens_match_the_oracle(pair, hidden, inter, top_k, tokens):
    rng = np.random.default_rng(hidden + inter + top_k)
    w = synth.moe_weights(20, top_k, hidden, inter, (pair[0],) + pair, rng)
    x, logits = rng.standard_normal((tokens, hidden)).astype(np.float32), rng.standard_normal((tokens, 20)).astype(np.float32)
    out, ids, _ = _layer(w).forward(ops.to_device(x), ops.to_device(logits))
    want, wids, _, _ = O.moe_layer(w, x, logits)
    assert np.array_equal(ids.cpu().numpy().view(np.uint32), wids)
    assert O.rel_l2(out.cpu().numpy(), want) <= REL_L2_F32


# 256 experts and their neighbours, 512 and theirs (a lane of the routing wave holds 4, 8 or 16 logits), the most
@pytest.mark.parametrize("experts", [255, 256, 257, 512, 513, 1024])
def test_few_tokens_over_many_experts(experts):
    rng = np.random.default_rng(experts)
    w = synth.moe_weights(experts, 8, 256, 256, (F.IQ2_XXS, F.IQ2_XXS, F.IQ2_S), rng)
    x, logits = rng.standard_normal((5, 256)).astype(np.float32), rng.standard_normal((5, experts)).astype(np.float32)
    logits[0] = np.round(2 * logits[0])  # ties
    logits[1, -1] = logits[2, 0] = 9  # the last expert and the first
    out, ids, weights = _layer(w).forward(ops.to_device(x), ops.to_device(logits))
    want, wids, wweights, _ = O.moe_layer(w, x, logits)
    assert np.array_equal(ids.cpu().numpy().view(np.uint32), wids)
    assert np.allclose(weights.cpu().numpy(), wweights, rtol=1e-5, atol=0)
    assert O.rel_l2(out.cpu().numpy(), want) <= REL_L2_F32


@pytest.mark.parametrize("inter,pad", [(37, 64), (320, 0), (2880, 0)])
def test_few_tokens_with_biases_padding_and_absent_slots(inter, pad):
    """MXFP4 with the clamped SwiGLU: odd rows, hidden rows padded with zeros, a slot past the bank giving a NaN row."""
    rng = np.random.default_rng(inter)
    hidden, top_k, tokens = 640, 4, 3
    w = synth.moe_weights(12, top_k, hidden, inter, (F.MXFP4,) * 3, rng, act=1, pad=pad)
    x, logits = rng.standard_normal((tokens, hidden)).astype(np.float32), rng.standard_normal((tokens, 12)).astype(np.float32)
    layer = _layer(w)
    out, ids, _ = layer.forward(ops.to_device(x), ops.to_device(logits))
    want, wids, _, _ = O.moe_layer(w, x, logits)
    assert np.array_equal(ids.cpu().numpy().view(np.uint32), wids)
    assert O.rel_l2(out.cpu().numpy(), want) <= REL_L2_F32
    table = np.arange(12, dtype=np.uint32)
    table[wids[1, 2]] = 12
    missing = torch.zeros(1, dtype=torch.int32, device="cuda")
    table[wids[0, 0]] = 0xFFFFFFFF  # reads slot 0, counted
    behind = ops.MoeLayer(*layer.banks, n_experts=12, top_k=top_k, act=layer.act, slot_table=ops.to_device(table))
    got = behind.forward(ops.to_device(x), ops.to_device(logits), missing=missing)[0].cpu().numpy()
    nan = (wids == wids[1, 2]).any(1)
    assert np.array_equal(np.isnan(got).all(1), nan) and np.array_equal(np.isnan(got).any(1), nan)
    assert int(missing.item()) == int((wids == wids[0, 0]).sum()) or wids[0, 0] == wids[1, 2]
