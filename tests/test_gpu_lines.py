"""Fan-beam projection along the rays' lines (FP32 engine) against the FP64
oracle, which sums the tracer's entries.

u is stored in FP32 and updated 12 times (3 passes of 4 subsets); a step's
rounding (2^-24 of u) and its projections' (2^-24 of the entries) are below
12 x 2 x 6e-8 = 1.5e-6 together, so 2e-6 relative L2 bounds u, and v, which
follows from it, as well."""
import numpy as np
import pytest

import medimage_amd as mi
from medimage_amd import configs
import oracle_py as O

pytestmark = pytest.mark.gpu


def _fan(nx, ny, pixel, views, bins, bin_mm, sod=541.0, sdd=949.0, span=360.0, off=0.0):
    return mi.Geometry(mi.MI_BEAM_FAN_FLAT, nx, ny, pixel, views, span, bins, bin_mm, sod, sdd, off, 0, 0)


GEOMS = {
    "square": _fan(64, 64, 4.0, 60, 96, 4.0),
    "tiny": _fan(7, 7, 20.0, 8, 9, 30.0),
    "wide": _fan(37, 150, 2.0, 24, 129, 4.0),          # a group of one ray
    "tall": _fan(201, 33, 1.5, 21, 64, 8.0),           # one full group a view
    "one_bin": _fan(40, 40, 5.0, 90, 1, 4.0, off=0.5),  # the central ray, on the grid line at 0, 90, 180, 270
    "half_offset": _fan(64, 64, 4.0, 48, 96, 4.0, off=-0.5),
    "quarter_offset": _fan(65, 65, 4.0, 45, 97, 4.0, off=0.25),
    "fine_bins": _fan(24, 24, 8.0, 30, 520, 0.5),      # many rays a pixel
    "coarse_bins": _fan(120, 120, 1.0, 40, 20, 12.0),  # many pixels between rays
    "half_turn": _fan(90, 90, 2.5, 31, 111, 3.3, span=180.0),
    "source_in_corner": _fan(64, 64, 4.0, 40, 96, 6.0, sod=150.0, sdd=500.0),
    "fine_pixels": _fan(48, 48, 0.04, 24, 80, 0.05, sod=20.0, sdd=40.0),   # pixels below the tracer's exit margin
    "two_groups": _fan(336, 336, 1.0, 70, 96, 4.0),    # 441 blocks: two groups share a block's views
    "one_group": _fan(432, 420, 0.8, 270, 64, 6.0),    # 729 blocks; 67 or 68 views a subset: two windows
    "arc": mi.arc_geometry(96, 3.0, 48, 98, 0.45, 595.0, 1085.6, 1.75),
    "arc_wide": mi.arc_geometry(61, 4.0, 40, 64, 1.6, 250.0, 600.0, -0.25),
}


@pytest.mark.parametrize("name", sorted(GEOMS))
def test_lines_match_oracle(ctx, name):
    g = GEOMS[name]
    rng = np.random.default_rng(len(name))
    img = rng.random((g.nx, g.ny)) * 0.02 / g.pixel_mm
    sino = O.fan_fp(O.fan_from(g), img)
    sino32 = (sino + 0.01 * rng.random(sino.shape)).astype(np.float32)
    p = mi.at_params(1e-3, 1e-4, 1e-2, n_subsets=4, max_iters=3)
    u, v, rep = ctx.at_reconstruct(g, sino32, p)
    ou, ov, _, hist = O.os_at(O.op_fan(O.fan_from(g)), sino32.astype(np.float64), 1e-3, 1e-4, 1e-2, 4, 3)
    eu, ev = (float(np.linalg.norm(a - b) / np.linalg.norm(b)) for a, b in ((u, ou), (v, ov)))
    print(f"[lines {name}] u {eu:.1e} v {ev:.1e}", flush=True)
    assert eu < 2e-6 and ev < 2e-6
    assert abs(rep.data_fidelity - hist[-1]) <= 1e-5 * hist[-1]
