"""Router logits of many tokens (32 x 32 tiles on the f32 matrix instruction)."""
import numpy as np
import pytest

from coachwhip_amd import ops

pytestmark = pytest.mark.gpu


# one past a tile, one short of it, rows shorter than, equal to and just over the 256-wide chunks
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
@pytest.mark.parametrize("experts,hidden,tokens", [(1, 4, 9), (33, 252, 33), (31, 256, 65), (64, 260, 31), (130, 2048, 301)])
def test_router_tiles(experts, hidden, tokens, dtype):
    rng = np.random.default_rng(experts + hidden)
    w = rng.standard_normal((experts, hidden)).astype(dtype)
    x = rng.standard_normal((tokens, hidden)).astype(np.float32)
    bias = rng.standard_normal(experts).astype(np.float32)
    got = ops.router_logits(ops.to_device(w), ops.to_device(x), ops.to_device(bias)).cpu().numpy()
    want = x.astype(np.float64) @ w.astype(np.float64).T + bias
    # a chain of `hidden` f32 fused multiply-adds: each rounding is at most 2^-24 of the partial sum,
    # which stays below 4 sqrt(hidden) sigma here; the largest error over all is below a quarter of the bound
    assert np.abs(got - want).max() <= hidden * 2.0 ** -24 * 4 * np.sqrt(hidden) + 2.0 ** -22
    # a logit does not depend on where its token and expert lie in the tiles
    p, q = rng.permutation(tokens), rng.permutation(experts)
    moved = ops.router_logits(ops.to_device(w[q]), ops.to_device(x[p]), ops.to_device(bias[q])).cpu().numpy()
    assert np.array_equal(moved.view(np.uint32), got[p][:, q].view(np.uint32))
