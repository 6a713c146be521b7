"""mi_forward of fan beams in FP32, which goes along the rays' lines, against
the FP64 oracle's sum of the tracer's entries.  A line's weight, its product
with a pixel and the result are rounded to FP32 once each (6e-8), the sum is in
double: 1e-6 relative L2 bounds it.  A pixel that is not finite reaches the
rays whose traced entries hold it and no others."""
import numpy as np
import pytest

import oracle_py as O
from test_gpu_lines import GEOMS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", sorted(GEOMS))
def test_line_forward_matches_oracle(ctx, name):
    g = GEOMS[name]
    img = np.random.default_rng(len(name)).random((g.nx, g.ny)).astype(np.float32)
    ref = O.fan_fp(O.fan_from(g), img.astype(np.float64))
    dev = ctx.forward(g, img)
    err = float(np.linalg.norm(dev - ref) / np.linalg.norm(ref))
    print(f"[line forward {name}] {err:.1e}", flush=True)
    assert err < 1e-6
    assert np.array_equal(dev, ctx.forward(g, img))


@pytest.mark.parametrize("name", ["square", "tall", "arc"])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_line_forward_not_finite(ctx, name, value):
    g = GEOMS[name]
    rng = np.random.default_rng(5)
    img = rng.random((g.nx, g.ny)).astype(np.float32)
    pix = [0, g.nx * g.ny - 1, (g.nx // 2) * g.ny + g.ny // 3]   # two corners, one inside
    rowptr, ind, ln = ctx.matrix(g)
    hit = np.zeros(len(rowptr) - 1, bool)
    for p in pix:
        img.ravel()[p] = value
        hit[np.searchsorted(rowptr, np.flatnonzero(ind == p), side="right") - 1] = True
    assert hit.any() and not hit.all()
    ok = np.where(np.isfinite(img), img, 0.0)
    ref = O.fan_fp(O.fan_from(g), ok.astype(np.float64)).ravel()
    print(f"[line forward {name}] {value}", flush=True)
    dev = ctx.forward(g, img).ravel()
    assert np.all(np.isfinite(dev[~hit]))
    assert np.abs(dev[~hit] - ref[~hit]).max() < 1e-6 * np.abs(ref).max()
    assert np.array_equal(np.isnan(dev[hit]), np.full(hit.sum(), np.isnan(value)))
