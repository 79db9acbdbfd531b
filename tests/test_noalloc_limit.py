"""Which calls cw_moe_layer_noalloc takes near the size of its array: layers behind a slot table with gate and up
biases, whose tile list (per expert) is longer than one per slot, are held to the latter. On the CPU: a call that
fits gets as far as the missing device, or its null inputs."""
import ctypes

import pytest
import torch

import coachwhip_amd as cw
from coachwhip_amd import _lib
from coachwhip_amd import formats as F

LIMIT = 8 << 20


def _desc(experts, slots, top_k, hidden, inter, biases):
    d = _lib.MoeDesc()
    d.n_experts, d.top_k, d.hidden, d.inter, d.act = experts, top_k, hidden, inter, 1
    d.slot_table, d.n_slots, d.alpha, d.limit = 0x1000, slots, 1.702, 7.0
    for m, (n, k) in enumerate([(inter, hidden), (inter, hidden), (hidden, inter)]):
        d.dtype[m], d.w[m], d.slot_stride[m] = F.Q4_K, 0x1000, F.matrix_bytes(F.Q4_K, n, k)
        if biases:
            d.bias[m] = 0x1000
    return d


def _refused(d, tokens):
    rc = cw.lib().cw_moe_layer_noalloc(ctypes.byref(d), None, None, tokens, None, None, None, None, None)
    assert rc != 0
    return b"bytes of scratch" in cw.lib().cw_last_error()


@pytest.mark.skipif(torch.cuda.is_available(), reason="the accepted calls must stop before a launch")
@pytest.mark.parametrize("experts,slots,top_k,hidden,inter", [(1024, 8, 8, 256, 256), (768, 8, 4, 256, 256), (700, 3, 2, 256, 512)])
def test_biases_do_not_change_what_fits(experts, slots, top_k, hidden, inter):
    plain, biased = _desc(experts, slots, top_k, hidden, inter, False), _desc(experts, slots, top_k, hidden, inter, True)
    size = cw.lib().cw_moe_workspace_size
    fits = [t for t in range(16, 2400) if size(ctypes.byref(plain), t) <= LIMIT]
    edge = [t for t in fits if size(ctypes.byref(biased), t) > LIMIT]
    assert edge  # calls whose longer list takes them past the limit
    for t in edge + [fits[0], fits[-1]]:
        assert not _refused(plain, t) and not _refused(biased, t)
    assert _refused(plain, fits[-1] + 1) and _refused(biased, fits[-1] + 1)
