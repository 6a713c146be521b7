"""Jobs whose edge steps stop early (largest change below 1e-5) before the
pass's last edge step, alone and in one batch with jobs that do not stop.  The
oracle's own stop is the reference; the bar is that of the FP64 engine's other
comparisons."""
import numpy as np
import pytest

import medimage_amd as mi
import oracle_py as O

pytestmark = pytest.mark.gpu

G = mi.fan_geometry(64, 4.0, 60, 96, 4.0)
# (scale of the sinogram, edge steps a pass): small slopes stop after the first step
JOBS = [(1.0, 7), (30.0, 7), (1.0, 2), (1.0, 1), (30.0, 1)]


def test_edge_stop(ctx):
    img = np.zeros((64, 64))
    img[20:40, 25:45] = 0.02
    sino = O.fan_fp(O.fan_from(G), img)
    op = O.op_fan(O.fan_from(G))
    ref = [O.os_at(op, sino * s, 1e-3, 1e-4, 1e-2, 4, 5, iter_edge=e) for s, e in JOBS]
    assert np.array_equal(ref[0][1], ref[3][1]) and not np.array_equal(ref[1][1], ref[4][1])
    b = ctx.batch(4, mi.MI_FP64)
    ids = [b.submit(G, sino * s, mi.at_params(n_subsets=4, max_iters=5, iter_edge=e, precision=mi.MI_FP64))
           for s, e in JOBS]
    b.run()
    out = [b.read(i) for i in ids]
    b.close()
    for k, (s, e) in enumerate(JOBS):
        p = mi.at_params(n_subsets=4, max_iters=5, iter_edge=e, precision=mi.MI_FP64)
        u, v, rep = ctx.at_reconstruct(G, sino * s, p)
        ou, ov, n, hist = ref[k]
        assert rep.iterations == n == 5
        assert abs(rep.data_fidelity - hist[-1]) <= 1e-10 * hist[-1]
        for a, r in ((u, ou), (v, ov)):
            assert np.linalg.norm(a - r) < 1e-10 * np.linalg.norm(r)
        assert np.array_equal(out[k][0], u) and np.array_equal(out[k][1], v)
