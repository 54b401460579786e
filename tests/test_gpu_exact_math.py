"""The division by a shared denominator and the light tree's logarithm, whose
results the traversal and the light choice take for correctly rounded: bit
for bit against numpy's binary32 division, and against an 80-bit logarithm
rounded once."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bits(x):
    return np.ascontiguousarray(x, np.float32).view(np.uint32)


def _random(rng, n, lo, hi):
    """Random mantissas, exponents in [lo, hi)."""
    return np.ldexp(rng.uniform(1, 2, n), rng.integers(lo, hi, n)).astype(np.float32) * rng.choice([-1, 1], n).astype(np.float32)


def test_shared_division_rounds_like_division(engine):
    rng = np.random.default_rng(1)
    n = 1 << 22
    one_ulp = (rng.integers(0, 1 << 23, n) | 0x3F800000).astype(np.uint32)
    pairs = [(_random(rng, n, -60, 80), _random(rng, n, -40, 40)),           # the whole range of its conditions
             (_random(rng, n, -1, 1), _random(rng, n, -1, 1)),               # quotients near one
             (one_ulp.view(np.float32), (one_ulp ^ 1).view(np.float32)),     # ... and a bit apart
             (_random(rng, n, -149, 127), _random(rng, n, -149, 127))]       # past the conditions too
    edge = np.float32([0.0, -0.0, np.inf, -np.inf, np.nan, 1e-45, 2.0 ** -60, 2.0 ** -61, 2.0 ** 80, 2.0 ** 40, 2.0 ** 41,
                       2.0 ** -40, 2.0 ** -41, 3.4e38, 1.0, 3.0])
    a, b = (x.ravel() for x in np.meshgrid(edge, edge))
    pairs.append((a, b))
    for a, b in pairs:
        q, _ = engine.selftest_math(a, b)
        with np.errstate(all="ignore"):
            want = a / b
        nan = np.isnan(want)
        assert np.array_equal(np.isnan(q), nan)
        assert np.array_equal(_bits(q)[~nan], _bits(want)[~nan])


def test_light_tree_log2_rounds_once(engine):
    rng = np.random.default_rng(2)
    mantissas = np.arange(1 << 23, dtype=np.uint32)
    parts = [mantissas | np.uint32(e << 23) for e in (126, 127, 128)]  # every argument around one
    parts.append(rng.integers(0x00800000, 0x7F800000, 1 << 23).astype(np.uint32))
    parts.append(rng.integers(1, 0x00800000, 1 << 12).astype(np.uint32))  # denormals
    for x in parts:
        x = x.view(np.float32)
        _, got = engine.selftest_math(np.ones_like(x), x)
        want = np.log2(x.astype(np.longdouble)).astype(np.float32)
        assert np.array_equal(_bits(got), _bits(want))
    _, got = engine.selftest_math(np.ones(5, np.float32), np.float32([0.0, -0.0, -1.0, np.inf, np.nan]))
    assert got[0] == got[1] == -np.inf and np.isnan(got[2]) and got[3] == np.inf and np.isnan(got[4])
