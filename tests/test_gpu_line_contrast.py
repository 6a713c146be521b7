"""Rays along lines (FP32 fan beams) beside pixels that are finite and very
large: what a ray does not cross adds nothing to it.  The bars are those of
the comparisons without such pixels: 1e-6 of the largest value for a
projection; for an update, whose step follows from sums of FP32 residuals
(2^-24 each, some ten of them in a row), 1e-5 of the largest change and u's
own rounding."""
import numpy as np
import pytest

import medimage_amd as mi
import oracle_py as O
from test_gpu_lines import GEOMS, _fan

pytestmark = pytest.mark.gpu


def _rays_of(ctx, g, pix):
    """Per ray: crosses one of the pixels; per pixel: lies on such a ray."""
    rowptr, ind, ln = ctx.matrix(g)
    row = np.repeat(np.arange(len(rowptr) - 1), np.diff(rowptr))
    hit = np.zeros(len(rowptr) - 1, bool)
    hit[row[np.isin(ind, pix)]] = True
    on = np.zeros(g.nx * g.ny, bool)
    on[ind[hit[row]]] = True
    return hit, on


@pytest.mark.parametrize("name", ["square", "tall", "arc", "one_group"])
@pytest.mark.parametrize("value", [1e6, 1e9, 1e12])
def test_line_forward_large_pixels(ctx, name, value):
    g = GEOMS[name]
    img = np.random.default_rng(5).random((g.nx, g.ny)).astype(np.float32)
    pix = [0, g.nx * g.ny - 1, (g.nx // 2) * g.ny + g.ny // 3]   # two corners, one inside
    hit, _ = _rays_of(ctx, g, pix)
    assert hit.any() and not hit.all()
    img.ravel()[pix] = value
    print(f"[large pixels {name}] {value}", flush=True)
    dev = ctx.forward(g, img).ravel()
    img.ravel()[pix] = 0.0
    ref = O.fan_fp(O.fan_from(g), img.astype(np.float64)).ravel()
    assert np.abs(dev[~hit] - ref[~hit]).max() < 1e-6 * np.abs(ref).max()


@pytest.mark.parametrize("value", [1e6, 1e9])
def test_line_update_large_pixel(ctx, value):
    g = _fan(64, 64, 4.0, 3, 96, 4.0)
    rng = np.random.default_rng(6)
    u0 = (0.02 * rng.random((64, 64))).astype(np.float32)
    sino = O.fan_fp(O.fan_from(g), 0.02 * rng.random((64, 64))).astype(np.float32)
    pix = 20 * 64 + 41
    _, on = _rays_of(ctx, g, [pix])
    for o in (-65, -64, -63, -1, 0, 1, 63, 64, 65):   # the regulariser's reach
        on[pix + o] = True
    assert (~on).sum() > 1000
    u0.ravel()[pix] = value
    p = mi.at_params(1e-3, 1e-4, 1e-2, n_subsets=1, max_iters=1, iter_edge=0)
    u, _, _ = ctx.at_reconstruct(g, sino, p, u0=u0)
    ou, _, _, _ = O.os_at(O.op_fan(O.fan_from(g)), sino.astype(np.float64), 1e-3, 1e-4, 1e-2, 1, 1, iter_edge=0,
                          u0=u0.astype(np.float64))
    u, ou, u0 = u.ravel()[~on], ou.ravel()[~on], u0.ravel()[~on]
    change = np.abs(ou - u0).max()
    print(f"[large pixel, update] {value}: change {change:.1e}, off by {np.abs(u - ou).max():.1e}", flush=True)
    assert change > 1e-4
    assert np.all(np.abs(u - ou) <= 1e-5 * change + 2.0**-24 * np.abs(ou))
