"""Which fan-beam geometries go along lines, at the limits of that form; what
its tables hold; and its results there against the FP64 oracle.

The form shows in the context's memory: a stored matrix holds at least 8 bytes
an entry (index and length), the lines some 100 bytes a ray and 32 bytes a
block and view.  The bar of a reconstruction is that of the line form's other
comparison (2e-6 after 12 updates)."""
import numpy as np
import pytest

import medimage_amd as mi
import oracle_py as O
from test_gpu_lines import GEOMS, _fan

pytestmark = pytest.mark.gpu

EDGE = {
    # seven or eight rays a pixel, the most that the back projection takes
    "eight_rays": _fan(96, 96, 3.0, 20, 330, 1.8),
    # a source just behind the least distance (2% of it beyond the image and a block)
    "near_source": _fan(64, 64, 4.0, 40, 137, 6.0, sod=279.0, sdd=480.0),
    # an arc just inside its 45 degrees
    "wide_arc": mi.arc_geometry(96, 3.0, 48, 76, 1.2, 295.0, 600.0, 1.75),
    # a detector so long that a float does not hold its bins' places
    "long_detector": _fan(48, 48, 4.0, 2, 16000001, 4.0, off=0.3),
    "view_pairs": _fan(80, 80, 3.0, 9, 111, 3.3),
}
LINES = ["square", "wide", "half_turn", "two_groups", "one_group", "arc", "coarse_bins", "eight_rays", "near_source", "wide_arc",
         "view_pairs"]
MATRIX = ["source_in_corner", "fine_pixels", "arc_wide", "fine_bins"]


@pytest.mark.parametrize("name", LINES + MATRIX)
def test_line_form(ctx, name):
    g = {**GEOMS, **EDGE}[name]
    ctx.trim()
    nnz, mem = ctx.prepare(g, 4), ctx.mem_bytes()
    print(f"[line form {name}] {nnz} entries, {mem} bytes", flush=True)
    assert (mem < 8 * nnz) == (name in LINES)


@pytest.mark.parametrize("name,subsets", [("eight_rays", 4), ("near_source", 4), ("wide_arc", 4), ("long_detector", 1),
                                          ("view_pairs", 9), ("view_pairs", 8), ("view_pairs", 4)])
def test_line_limits_match_oracle(ctx, name, subsets):
    g = EDGE[name]
    rng = np.random.default_rng(len(name))
    img = rng.random((g.nx, g.ny)) * 0.02 / g.pixel_mm
    of = O.fan_from(g)
    sino = O.fan_fp(of, img)
    sino32 = np.where(sino > 0, sino + 0.01 * rng.random(sino.shape), 0.0).astype(np.float32)
    p = mi.at_params(1e-3, 1e-4, 1e-2, n_subsets=subsets, max_iters=3)
    u, v, rep = ctx.at_reconstruct(g, sino32, p)
    ou, ov, _, hist = O.os_at(O.op_fan(of), sino32.astype(np.float64), 1e-3, 1e-4, 1e-2, subsets, 3)
    eu, ev = (float(np.linalg.norm(a - b) / np.linalg.norm(b)) for a, b in ((u, ou), (v, ov)))
    print(f"[line limits {name} {subsets}] u {eu:.1e} v {ev:.1e}", flush=True)
    assert eu < 2e-6 and ev < 2e-6
    assert abs(rep.data_fidelity - hist[-1]) <= 1e-5 * hist[-1]


def test_line_tables(ctx):
    """Subsets of one view need no more room than larger ones; a forward
    projection none of the back projection's tables; an FP64 run no lines."""
    g = mi.fan_geometry(512, 0.7, 720, 736, 1.0)
    rows = g.n_views * g.n_bins
    ctx.trim()
    ctx.prepare(g, 12)
    few = ctx.mem_bytes()
    ctx.trim()
    ctx.prepare(g, 720)
    many = ctx.mem_bytes()
    print(f"[line tables] 12 subsets {few}, 720 subsets {many} bytes", flush=True)
    assert many < 1.1 * few
    ctx.trim()
    ctx.forward(g, np.zeros((512, 512), np.float32))
    one = ctx.mem_bytes()
    print(f"[line tables] forward {one} bytes", flush=True)
    assert one < 60 * rows
    ctx.trim()
    small = GEOMS["square"]
    nnz = ctx.prepare(small, 4)
    lines = ctx.mem_bytes()
    sino = np.random.default_rng(1).random((small.n_views, small.n_bins))
    p32 = mi.at_params(n_subsets=4, max_iters=2)
    p64 = mi.at_params(n_subsets=4, max_iters=2, precision=mi.MI_FP64)
    before = ctx.at_reconstruct(small, sino.astype(np.float32), p32)
    ctx.at_reconstruct(small, sino, p64)
    both = ctx.mem_bytes()
    after = ctx.at_reconstruct(small, sino.astype(np.float32), p32)
    assert ctx.mem_bytes() == both > lines
    assert np.array_equal(before[0], after[0]) and np.array_equal(before[1], after[1])
    ctx.trim()
    ctx.at_reconstruct(small, sino, p64)
    assert ctx.mem_bytes() == both - lines


def test_line_bytes(ctx):
    """A timed launch reports what it reads and writes, not a matrix's entries."""
    g = mi.fan_geometry(256, 1.4, 360, 512, 1.44)
    ctx.trim()
    nnz = ctx.prepare(g, 1)
    job = ctx.job(g, np.ones((g.n_views, g.n_bins), np.float32), mi.at_params(n_subsets=1, max_iters=2))
    ctx.stats_reset()
    ctx.stats_enable(True)
    job.enqueue(1)
    job.synchronize()
    ctx.forward(g, np.ones((256, 256), np.float32))
    ctx.stats_enable(False)
    fp, bp, sq = (ctx.stats(k) for k in (mi.MI_K_FP, mi.MI_K_BP, mi.MI_K_FPSQ))
    job.close()
    rows, pix = g.n_views * g.n_bins, g.nx * g.ny
    print(f"[line bytes] {nnz} entries; {fp.bytes} {bp.bytes} {sq.bytes}", flush=True)
    assert (fp.launches, bp.launches, sq.launches) == (2, 1, 1)
    assert sq.bytes == 36.0 * rows + 4 * pix
    assert fp.bytes == 36.0 * rows + 8 * pix + 8 * rows + 36.0 * rows + 4 * (pix + rows)
    assert bp.bytes == 24.0 * rows + 32.0 * 256 * g.n_views + 24 * pix
    assert max(fp.bytes, bp.bytes, sq.bytes) < 4 * nnz
