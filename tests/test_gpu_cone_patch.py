"""The cone beam's back projection from panel patches against the oracle's
double transpose of the exact lengths: partial tiles and slice runs, the
source's height inside a run, between two and on a plane, panels smaller than
the volume's shadow, coarse and fine pixels, more views than one group, the
16-slice form, and geometries that keep the ray by ray form.  The bar is the
back projection's own (1e-5 of the largest value).  A value that is not
finite reaches the voxels of its ray and no others."""
import numpy as np
import pytest

import medimage_amd as mi
import oracle_py as O

pytestmark = pytest.mark.gpu

GEOMS = [
    mi.cone_geometry(17, 15, 33, 40, 64, 64, 1.0, 1.0, 90.0, 150.0),      # source between planes, two view groups
    mi.cone_geometry(33, 18, 24, 36, 21, 24, 1.0, 1.3, 90.0, 150.0),      # panel inside the shadow, odd rows
    mi.cone_geometry(16, 16, 8, 37, 16, 12, 1.0, 4.0, 60.0, 100.0),       # coarse pixels
    mi.cone_geometry(20, 20, 9, 12, 120, 160, 1.0, 0.3, 200.0, 260.0),    # fine pixels: 3 to 6 rays per voxel
    mi.cone_geometry(128, 128, 127, 5, 192, 192, 1.0, 1.0, 300.0, 480.0),  # 16 slices per workgroup
    mi.cone_geometry(128, 128, 128, 4, 192, 130, 0.5, 0.5, 150.0, 240.0),
    mi.cone_geometry(20, 20, 12, 9, 40, 40, 1.0, 0.5, 17.0, 30.0),        # near source: several rows per chord
    mi.cone_geometry(30, 30, 16, 6, 300, 500, 1.0, 0.1, 90.0, 120.0),     # patch beyond LDS
]


@pytest.mark.parametrize("gi", range(len(GEOMS)))
def test_cone_patch_backprojection(ctx, gi):
    g = GEOMS[gi]
    print(f"cone back projection {g}", flush=True)
    sino = np.random.default_rng(30 + gi).random((g.n_views, g.n_rows, g.n_cols)).astype(np.float32)
    dev = ctx.cone_backproject(g, sino).astype(np.float64)
    ref = O.cone_bp(O.cone_from(g), sino.astype(np.float64))
    assert np.abs(ref).max() > 0
    assert np.abs(dev - ref).max() < 1e-5 * np.abs(ref).max()
    assert np.all(dev[ref == 0] == 0) or gi in (6, 7)


@pytest.mark.parametrize("gi", [0, 4])
@pytest.mark.parametrize("value", [np.nan, np.inf, 3e38])
def test_cone_patch_not_finite(ctx, gi, value):
    g = GEOMS[gi]
    print(f"cone back projection {g} with {value}", flush=True)
    at = (g.n_views // 2, g.n_rows // 2 + 3, g.n_cols // 2 - 2)
    one = np.zeros((g.n_views, g.n_rows, g.n_cols), np.float32)
    one[at] = 1.0
    hit = ctx.cone_backproject(g, one) != 0
    assert hit.any()
    sino = np.random.default_rng(1).random(one.shape).astype(np.float32)
    sino[at] = 0.0
    ref = ctx.cone_backproject(g, sino).astype(np.float64)
    sino[at] = value
    dev = ctx.cone_backproject(g, sino).astype(np.float64)
    assert np.all(np.isfinite(dev[~hit]))
    assert np.abs(dev - ref)[~hit].max() < 1e-5 * np.abs(ref).max()
    assert not np.isfinite(dev[hit]).all() or np.abs(dev[hit]).max() > 1e30
