"""Sequential sums of the GoldenC steps (k_chains): the device folds 4096
terms a step, 256 a wave, and equals the oracle's term-by-term loop bit for
bit.  The edge step's three sums (|grad d|^2, d^2, n d^2) set its step size, so
its result shows any difference.  Sizes around a wave and a step; values of
one scale, of scales 2^-40 .. 2^40 (the running sum changes its binade often
and late), mostly zero, and few-bit values (terms halfway between two units)."""
import numpy as np
import pytest

import oracle_py as O

pytestmark = pytest.mark.gpu


def _values(kind, shape, rng):
    f, v = rng.random(shape), rng.random(shape)
    if kind == "scales":
        f = f * 2.0 ** rng.integers(-40, 40, shape)
    elif kind == "zeros":
        f[rng.random(shape) < 0.97] = 0.0
        v[:] = 1.0
    elif kind == "few_bits":
        f, v = np.floor(f * 8) / 8, np.floor(v * 8) / 8
    return f, v


@pytest.mark.parametrize("kind", ["one_scale", "scales", "zeros", "few_bits"])
@pytest.mark.parametrize("shape", [(1, 1), (1, 257), (16, 16), (64, 64), (64, 65), (63, 131), (200, 311)])
def test_edge_step_sums_bitwise(ctx, shape, kind):
    f, v = _values(kind, shape, np.random.default_rng(shape[0] * 1000 + shape[1]))
    for alpha, beta, eps in ((1000.0, 0.002, 1e-4), (1.0, 0.5, 0.25)):
        got = ctx.edge_step(f, v, alpha, beta, eps, 3)
        want, _ = O.edge_step(f, v, alpha, beta, eps, 3)
        assert np.array_equal(got.view(np.uint64), want.view(np.uint64))
