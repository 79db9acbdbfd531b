"""Layers of many tokens with a bias per expert behind a slot table: experts that the bank does not hold all read
slot 0, each with its own bias, on every grouped path, as the per-pick kernels and the oracle do."""
import numpy as np
import pytest
import torch

from coachwhip_amd import formats as F
from coachwhip_amd import ops, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu

REL_L2 = 1e-3  # the fp16 GEMMs' gate; a bias row of another expert moves the output by more than 0.1


# fp16 GEMMs, the f32-accurate ones, the scaled MXFP4 ones in both layouts; one pile per expert at the edges of a tile
@pytest.mark.parametrize("formats", [(F.Q4_K, F.IQ4_XS), (F.Q4_K, F.Q6_K), (F.MXFP4, F.MXFP4), (F.MXFP4_R16, F.MXFP4_R16)],
                         ids=lambda f: F.NAMES[f[0]] + "-" + F.NAMES[f[1]])
@pytest.mark.parametrize("tokens,experts,slots,top_k", [(40, 24, 9, 4), (200, 10, 3, 5), (17, 700, 40, 8)])
def test_absent_experts_keep_their_biases(formats, tokens, experts, slots, top_k, monkeypatch):
    monkeypatch.setenv("CWMOE_PREFILL_MIN_TOKENS", "16")
    rng = np.random.default_rng(tokens)
    hidden, inter = 512, 256
    r16 = formats[0] == F.MXFP4_R16
    dts = (F.MXFP4,) * 3 if r16 else (formats[0],) + formats
    w = synth.moe_weights(experts, top_k, hidden, inter, dts, rng, n_slots=slots, act=1)
    w.bias = [50 * b for b in w.bias]
    shapes = [(inter, hidden)] * 2 + [(hidden, inter)]
    banks = [ops.ExpertBank.from_blocks(w.host[m], w.dtypes[m], *s, slots) for m, s in enumerate(shapes)]
    if r16:
        banks = [b.rows16() for b in banks]
    table = np.full(experts, 0xFFFFFFFF, np.uint32)
    table[rng.choice(experts, slots - 1, replace=False)] = rng.permutation(slots)[:slots - 1]
    # (exact in fp16, and small: the gates and ups stay inside the clamp)
    x = (rng.standard_normal((tokens, hidden)) * 2.0 ** -8).astype(np.float16).astype(np.float32)
    logits = rng.standard_normal((tokens, experts)).astype(np.float32)
    act = ops.ExpertAct.clamped_swiglu(w.alpha, w.limit, *[ops.to_device(b) for b in w.bias])
    missing = torch.zeros(1, dtype=torch.int32, device="cuda")

    def run():
        layer = ops.MoeLayer(*banks, n_experts=experts, top_k=top_k, act=act, slot_table=ops.to_device(table))
        return layer.forward(ops.to_device(x), ops.to_device(logits), missing=missing)[0].cpu().numpy()

    want, wids, _, wmiss = O.moe_layer(w, x, logits, slot_table=table, n_slots=slots)
    assert O.rel_l2(run(), want) <= REL_L2 and int(missing.item()) == wmiss > 0
    # a slot past the bank still is in no pile
    table[wids[1, 1]] = slots
    got, hit = run(), (wids == wids[1, 1]).any(1)
    assert np.isnan(got[hit]).all() and O.rel_l2(got[~hit], want[~hit]) <= REL_L2
