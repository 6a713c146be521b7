"""Sequential sums of the GoldenC steps at the edges of their groups: 64 terms
a chunk, 1024 a group, 65536 a scan step.  Bit for bit the oracle's
term-by-term loop, through the edge step's three sums (|grad d|^2 has two
terms a pixel)."""
import numpy as np
import pytest

import oracle_py as O
from test_gpu_chains import _values

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["one_scale", "scales", "zeros", "few_bits"])
@pytest.mark.parametrize("shape", [(1, 31), (1, 32), (1, 33), (8, 8), (1, 65), (16, 32), (32, 32), (25, 41),
                                   (128, 256), (256, 256), (256, 257)])
def test_edge_step_sums_at_group_edges(ctx, shape, kind):
    f, v = _values(kind, shape, np.random.default_rng(shape[0] * 999 + shape[1]))
    print(f"[chain groups] {shape} {kind}", flush=True)
    got = ctx.edge_step(f, v, 1000.0, 0.002, 1e-4, 2)
    want, _ = O.edge_step(f, v, 1000.0, 0.002, 1e-4, 2)
    assert np.array_equal(got.view(np.uint64), want.view(np.uint64))
