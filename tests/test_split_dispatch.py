"""Which products and layers take the GEMMs on two fp16 activation terms, by the size rules that programs
get (no override): seen in the workspace sizes, on the CPU."""
import ctypes
import itertools

import pytest

import coachwhip_amd as cw
from coachwhip_amd import _lib
from coachwhip_amd import formats as F

EXPERT_TYPES = [F.Q8_0, F.Q2_K, F.Q4_K, F.Q5_K, F.Q6_K, F.IQ2_XXS, F.IQ3_XXS, F.IQ3_S, F.IQ2_S, F.IQ4_XS, F.MXFP4]


@pytest.fixture(autouse=True)
def _no_overrides(monkeypatch):
    monkeypatch.delenv("CWMOE_MM_MIN_ROWS", raising=False)
    monkeypatch.delenv("CWMOE_PREFILL_MIN_TOKENS", raising=False)


def _desc(gu, dn, experts, top_k, hidden, inter):
    d = _lib.MoeDesc()
    d.n_experts, d.top_k, d.hidden, d.inter = experts, top_k, hidden, inter
    for m, (t, n, k) in enumerate([(gu, inter, hidden), (gu, inter, hidden), (dn, hidden, inter)]):
        d.dtype[m], d.w[m], d.slot_stride[m] = t, 0x1000, F.matrix_bytes(t, n, k)
    return d


def _size(d, tokens):
    return cw.lib().cw_moe_workspace_size(ctypes.byref(d), tokens)


# (experts, top_k, hidden, inter): layers whose picks pass the GEMMs' line below and above 16 tokens
LAYERS = [(32, 8, 4096, 1536), (64, 8, 2048, 1536), (128, 8, 2048, 768), (256, 8, 2048, 512), (8, 2, 512, 256)]


@pytest.mark.parametrize("shape", LAYERS, ids=str)
def test_layer_workspace_does_not_shrink_with_tokens(shape):
    """A workspace (or a captured graph's buffer) sized for a layer's largest batch serves the smaller ones."""
    for gu, dn in itertools.product(EXPERT_TYPES, repeat=2):
        d = _desc(gu, dn, *shape)
        sizes = [_size(d, t) for t in range(1, 65)]
        assert sizes[0] > 0 and sizes == sorted(sizes), (F.NAMES[gu], F.NAMES[dn])


def _matvec_size(d, tokens):
    tk = tokens * d.top_k
    return 8448 + 3 * (-(-4 * tk // 256) * 256) + -(-4 * tk * d.inter // 256) * 256


@pytest.mark.parametrize("shape", LAYERS, ids=str)
@pytest.mark.parametrize("pair", list(itertools.product((F.Q4_K, F.Q8_0), repeat=2)) + [(F.Q4_K, F.Q6_K), (F.Q5_K, F.Q5_K)],
                         ids=lambda p: F.NAMES[p[0]] + "-" + F.NAMES[p[1]])
def test_layer_line(pair, shape):
    """The GEMMs from the token whose picks beyond the distinct experts reach 230 million weights (the fp16 ones
    from 16 tokens where they take both formats), the matvecs' layout and nothing else before."""
    d = _desc(*pair, *shape)
    experts, top_k, hidden, inter = shape
    for t in range(1, 65):
        beyond = (top_k * t - experts * (1 - (1 - top_k / experts) ** t)) * hidden * 3 * inter
        gemms = beyond >= 230e6 or (t >= 16 and not {F.Q5_K, F.Q6_K} & set(pair))
        assert (_size(d, t) > _matvec_size(d, t)) == gemms, t


@pytest.mark.parametrize("dtype", [F.Q5_K, F.Q6_K])
@pytest.mark.parametrize("n,k", [(4096, 4096), (1024, 2048), (16384, 2048), (4001, 4096)])
def test_dense_line(dtype, n, k):
    L = cw.lib()
    for m in range(1, 80):
        assert (L.cw_qmatmul_workspace_size(dtype, n, k, m) > 0) == (m > 2 and (5 * m - 12) * n * k >= 215000000)
