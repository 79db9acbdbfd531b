"""The shrink's level steps: clamp((int)(n / scale + 0.5f), 0, 3) in f32 against the comparisons that the
kernel makes instead (cw_requant.hip, Steps), restated here, around every step and over random values."""
import numpy as np

M = (0.5 - 1.5 * 2.0 ** -25, 1.5 - 2.0 ** -24, 2.5 - 2.0 ** -23)  # the midpoints below 0.5 - 2^-25, 1.5, 2.5


def steps(scale):
    out = []
    for m in M:
        v = scale.astype(np.float64) * m
        with np.errstate(over="ignore"):
            f = v.astype(np.float32)
        up = (f.view(np.uint32) + np.uint32(1)).view(np.float32)
        out.append(np.where(f.astype(np.float64) <= v, up, f))
    return out


def level_by_division(n, scale):
    with np.errstate(over="ignore", under="ignore", invalid="ignore"):
        v = (n / scale).astype(np.float32) + np.float32(0.5)
    return np.where(v >= 3, 3, np.where(v >= 2, 2, np.where(v >= 1, 1, 0)))


def level_by_steps(n, scale):
    t1, t2, t3 = steps(scale)
    with np.errstate(invalid="ignore"):
        return np.where(n >= t3, 3, np.where(n >= t2, 2, np.where(n >= t1, 1, 0)))


def test_midpoints():
    assert M[0] == float.fromhex("0x1p-1") - float.fromhex("0x1.8p-25")
    for m, q in zip(M, (np.float32(0.5) - np.float32(2.0 ** -25), np.float32(1.5), np.float32(2.5))):
        below = np.nextafter(q, np.float32(0))
        assert m == (float(q) + float(below)) / 2


def test_levels_equal_the_division():
    rng = np.random.default_rng(5)
    bits = np.concatenate([rng.integers(1, 0x7F800001, 400000), np.arange(1, 3000), np.arange(0x7F7FF000, 0x7F800001),
                           (127 << 23) + np.arange(-3000, 3000), rng.integers(0, 1 << 23, 100000) + (127 << 23)]).astype(np.uint32)
    scale = bits.view(np.float32)
    for t in steps(scale):
        b = t.view(np.uint32).astype(np.int64)
        for d in (-2, -1, 0, 1, 2):
            n = np.clip(b + d, 0, 0x7F800000).astype(np.uint32).view(np.float32)  # (a NaN step becomes the infinity below it)
            assert np.array_equal(level_by_steps(n, scale), level_by_division(n, scale))
    ratio = rng.uniform(-0.5, 4, scale.size)
    with np.errstate(over="ignore", invalid="ignore"):
        n = (scale.astype(np.float64) * ratio).astype(np.float32)
    assert np.array_equal(level_by_steps(n, scale), level_by_division(n, scale))
    for n in (np.inf, -np.inf, np.nan, 0.0, -0.0):
        v = np.full(scale.size, n, np.float32)
        assert np.array_equal(level_by_steps(v, scale), level_by_division(v, scale))
