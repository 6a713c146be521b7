"""The back projection along lines (FP32 fan beams), through one AT pass from
u = 0 without regulariser and edges (u = c A^T g): how many bits the weights
hold, and residuals that are not finite.

Bits: with a sinogram of random signs the pixel's sum cancels down to the
square root of its terms, so that each rounding of a term shows.  One rounding
to FP32 is off by 2^-24 / sqrt(3) times sqrt(3 / (8 ln 2)), the mean over a
binade, 2.53e-8 relative.  Residual, weight, d and u rounded once each are
2 x 2.53e-8 = 5.1e-8."""
import numpy as np
import pytest

import medimage_amd as mi
import oracle_py as O
from test_gpu_lines import GEOMS

pytestmark = pytest.mark.gpu

NAMES = ["square", "tall", "arc", "coarse_bins", "two_groups", "one_group"]


def _pass(ctx, g, sino):
    p = mi.at_params(0.0, 1e-4, 1e-2, n_subsets=1, max_iters=1, iter_edge=0)
    u, _, _ = ctx.at_reconstruct(g, sino, p)
    ou, _, _, _ = O.os_at(O.op_fan(O.fan_from(g)), sino.astype(np.float64), 0.0, 1e-4, 1e-2, 1, 1, iter_edge=0)
    return u, ou


@pytest.mark.parametrize("name", NAMES)
def test_line_weights_bits(ctx, name):
    g = GEOMS[name]
    sino = np.random.default_rng(3).standard_normal((g.n_views, g.n_bins)).astype(np.float32)
    u, ou = _pass(ctx, g, sino)
    err = float(np.linalg.norm(u - ou) / np.linalg.norm(ou))
    print(f"[line weights {name}] {err:.2e}", flush=True)
    assert err < 5.1e-8


@pytest.mark.parametrize("name", NAMES)
def test_line_residual_not_finite(ctx, name):
    """The step is 0 then (the sums are not numbers): u is NaN where a ray
    without a number crosses, 0 elsewhere."""
    g = GEOMS[name]
    sino = np.random.default_rng(4).random((g.n_views, g.n_bins)).astype(np.float32)
    for v, b in ((1, g.n_bins // 2), (g.n_views // 2, g.n_bins // 3), (g.n_views - 1, g.n_bins - 1)):
        sino[v, b] = np.nan
    print(f"[line residual {name}]", flush=True)
    u, ou = _pass(ctx, g, sino)
    assert np.isnan(ou).any() and not np.isnan(ou).all()
    assert np.array_equal(np.isnan(u), np.isnan(ou)) and not np.nan_to_num(u).any()
