"""The cone beam's back projection with a few detector values that are finite
and far larger than the rest: voxels off their rays keep what they have without
them, within the back projection's own bar (1e-5 of the largest value), and
voxels on their rays what the oracle has."""
import numpy as np
import pytest

import oracle_py as O
from test_gpu_cone_patch import GEOMS

pytestmark = pytest.mark.gpu


def _sino(g):
    return np.random.default_rng(1).random((g.n_views, g.n_rows, g.n_cols)).astype(np.float32)


def _check(ctx, g, big):
    """big: the large values, 0 elsewhere."""
    sino = _sino(g)
    sino[big != 0] = 0.0
    hit = ctx.cone_backproject(g, (big != 0).astype(np.float32)) != 0
    assert hit.any() and not hit.all()
    ref = O.cone_bp(O.cone_from(g), sino.astype(np.float64))
    dev = ctx.cone_backproject(g, sino + big).astype(np.float64)
    assert np.abs(dev - ref)[~hit].max() < 1e-5 * np.abs(ref).max()
    all_ = O.cone_bp(O.cone_from(g), (sino + big).astype(np.float64))
    assert np.abs(dev - all_)[hit].max() < 1e-5 * np.abs(all_).max()


@pytest.mark.parametrize("gi", [0, 4])
@pytest.mark.parametrize("value", [1e4, 1e8, 1e12, 1e20, 1e30])
def test_cone_patch_large_value(ctx, gi, value):
    g = GEOMS[gi]
    print(f"cone back projection {g} with {value}", flush=True)
    big = np.zeros((g.n_views, g.n_rows, g.n_cols), np.float32)
    big[g.n_views // 2, g.n_rows // 2 + 3, g.n_cols // 2 - 2] = value
    _check(ctx, g, big)


@pytest.mark.parametrize("value", [1e8, 1e16])
def test_cone_patch_large_column(ctx, value):
    """A column of the panel in one view, and a part of another view."""
    g = GEOMS[0]
    print(f"cone back projection, large column {value}", flush=True)
    big = np.zeros((g.n_views, g.n_rows, g.n_cols), np.float32)
    big[7, :, 20] = value
    big[11, : g.n_rows // 3, :] = -value
    _check(ctx, g, big)


def test_cone_patch_single_view_scale(ctx):
    """Views of very different scale, each even in itself; panel inside the volume's shadow."""
    g = GEOMS[1]
    sino = _sino(g)
    sino[3] *= 1e12
    ref = O.cone_bp(O.cone_from(g), sino.astype(np.float64))
    one = np.zeros_like(sino)
    one[3] = 1.0
    hit = ctx.cone_backproject(g, one) != 0
    sino[3] = 0.0
    off = O.cone_bp(O.cone_from(g), sino.astype(np.float64))
    sino[3] = _sino(g)[3] * np.float32(1e12)
    print("cone back projection, one view 1e12 times as large", flush=True)
    dev = ctx.cone_backproject(g, sino).astype(np.float64)
    assert (~hit).any()
    assert np.abs(dev - off)[~hit].max() < 1e-5 * np.abs(off).max()
    assert np.abs(dev - ref)[hit].max() < 1e-5 * np.abs(ref).max()


@pytest.mark.parametrize("value", [1e10, 1e25])
def test_cone_patch_sparse(ctx, value):
    """Two rays alone, one far larger: voxels on the smaller one's only."""
    g = GEOMS[0]
    print(f"cone back projection, two rays, {value}", flush=True)
    at, to = (5, g.n_rows // 2 - 4, 30), (29, g.n_rows // 2 + 6, 33)
    sino = np.zeros((g.n_views, g.n_rows, g.n_cols), np.float32)
    sino[at] = 1.0
    small = O.cone_bp(O.cone_from(g), sino.astype(np.float64))
    sino[to] = value
    dev = ctx.cone_backproject(g, sino).astype(np.float64)
    sino[at] = 0.0
    big = O.cone_bp(O.cone_from(g), sino.astype(np.float64))
    only = (big == 0) & (small != 0)
    assert only.any()
    assert np.abs(dev - small)[only].max() < 1e-5 * small.max()
    assert not dev[(big == 0) & (small == 0)].any()


@pytest.mark.parametrize("gi", [0, 1, 4])
def test_cone_patch_noise(ctx, gi):
    """Noise about 0, with rows of values 2e4 times as large: voxels that cancel by chance."""
    g = GEOMS[gi]
    print(f"cone back projection of noise {g}", flush=True)
    sino = np.random.default_rng(4).standard_normal((g.n_views, g.n_rows, g.n_cols)).astype(np.float32)
    sino[:, g.n_rows // 2 :] *= np.float32(2e4)
    ref = O.cone_bp(O.cone_from(g), sino.astype(np.float64))
    dev = ctx.cone_backproject(g, sino).astype(np.float64)
    assert np.abs(dev - ref).max() < 1e-5 * np.abs(ref).max()
    # an FP32 value of the sums' own: the voxels of the smaller values to as much
    one = np.zeros_like(sino)
    one[:, g.n_rows // 2 :] = 1.0
    small = O.cone_bp(O.cone_from(g), one.astype(np.float64)) == 0
    if small.any():
        assert np.abs(dev - ref)[small].max() < 1e-5 * np.abs(ref[small]).max()


@pytest.mark.parametrize("value", [1e6, 1e13, 1e16, 1e22, 1e33])
def test_cone_patch_large_row(ctx, value):
    """A row of the panel in every view: no voxel's sums are free of it where they reach it."""
    g = GEOMS[0]
    print(f"cone back projection, large row {value}", flush=True)
    big = np.zeros((g.n_views, g.n_rows, g.n_cols), np.float32)
    big[:, g.n_rows // 3, :] = value
    _check(ctx, g, big)


@pytest.mark.parametrize("value", [1e13, 1e16, 1e20, 1e33])
def test_cone_patch_large_anywhere(ctx, value):
    """One large value at each of many places: at the edge of blocks too."""
    g = GEOMS[0]
    print(f"cone back projection, large value {value} at many rows", flush=True)
    for row in range(1, g.n_rows - 1, 5):
        big = np.zeros((g.n_views, g.n_rows, g.n_cols), np.float32)
        big[row % g.n_views, row, g.n_cols // 2 + row % 5 - 2] = value
        if (ctx.cone_backproject(g, (big != 0).astype(np.float32)) != 0).any():
            _check(ctx, g, big)
