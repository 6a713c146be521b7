"""Performance cases: the work a user of medimage_amd has it do, through the
public Python entry points, from the smallest calls to the largest.

A case is a dict of plain values; its "kind" says which call it is:

  at       Context.at_reconstruct of one slice whose geometry the program
           keeps (fan, arc or parallel beam; FP32 or FP64)
  slice    one slice of a helical scan: each slice has source angles of its
           own, so its geometry is built for it and dropped after it
  batch    many slices of mixed geometries as one batch (submit, run, read)
  forward  Context.forward / "back": Context.backproject, host arrays
  cone_fp  3D projection of a volume on the device / "cone_bp": its transpose
  cone_at  one ordered-subset pass on a volume, in place on the device
  goldenc  GoldenC's MumfordShah (FP64, the reference's summation order)

Sinograms are exact line integrals of seeded ellipses (ellipsoids in 3D) with
Poisson noise, the inputs this path meets in earnest.
"""
import math

import numpy as np
import torch

import medimage_amd as mi

SOD, SDD, FOV = 541.0, 949.0, 358.4           # mm: the 2D scanner and its field of view
ARC_SOD, ARC_SDD, ARC_PITCH, ARC_OFF = 595.0, 1085.6, 0.06786112, 1.75   # the helical scanner
ALPHA, BETA, EPS = 1e-3, 1e-4, 1e-2


def listed():
    return [
        # a thumbnail reconstruction, three passes: what a call costs before any work
        dict(name="at_small", kind="at", beam="fan", n=64, views=60, bins=96, subsets=4, iters=3, f64=False),
        # one 256 x 256 slice without subsets, fifty iterations
        dict(name="at_c1", kind="at", beam="fan", n=256, views=360, bins=512, subsets=1, iters=50, f64=False),
        # one 512 x 512 slice, 720 views, 12 ordered subsets: the benchmark's slice
        dict(name="at_c2", kind="at", beam="fan", n=512, views=720, bins=736, subsets=12, iters=20, f64=False),
        # the same solver in double precision, odd sizes
        dict(name="at_f64", kind="at", beam="fan", n=243, views=331, bins=365, subsets=8, iters=6, f64=True),
        # msbeam's own parallel beam
        dict(name="at_parallel", kind="at", beam="parallel", n=512, views=180, bins=768, subsets=1, iters=20,
             f64=False),
        # one slice of a helical scan at the clinical size, its own angle table
        dict(name="slice_helical", kind="slice", n=874, views=576, bins=736, subsets=8, iters=6),
        # a mixed worklist, eight slices over several geometries
        dict(name="batch_mixed", kind="batch", jobs=8, pick=3, subsets=8, iters=12),
        # single projections on host arrays, each direction
        dict(name="forward_f32", kind="forward", n=512, views=720, bins=736, f64=False),
        dict(name="back_f64", kind="back", n=300, views=359, bins=451, f64=True),
        # industry3d's 128^3 cone-beam configuration, its back projection
        dict(name="cone_bp_128", kind="cone_bp", nx=128, ny=128, nz=128, views=180, rows=256, cols=256),
        # GoldenC's own program: one alternation of its ten
        dict(name="goldenc", kind="goldenc", iter_alt=1, iter_image=10, iter_edge=10),
        # a 512^3 volume from 720 views of a 1024 x 768 panel, one pass of 20 subsets: both projections at size
        dict(name="cone_at_c4", kind="cone_at", nx=512, ny=512, nz=512, views=720, rows=1024, cols=768, subsets=20),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["at", "at", "at", "slice", "batch", "forward", "back", "cone_fp", "cone_bp", "cone_at",
                       "goldenc"])
    if kind == "at":
        beam = rng.choice(["fan", "fan", "arc", "parallel"])
        f64 = rng.random() < 0.25
        n = _log(rng, 48, 320 if f64 else 640)
        views = _log(rng, 40, 360 if f64 else 720)
        bins = 2 * (int(n * rng.uniform(1.0, 1.5)) // 2)
        return dict(kind=kind, beam=beam, n=n, views=views, bins=bins, subsets=rng.randint(1, 16),
                    iters=rng.randint(3, 20), f64=f64)
    if kind == "slice":
        n = _log(rng, 160, 874)
        return dict(kind=kind, n=n, views=_log(rng, 96, 576), bins=2 * rng.randint(128, 368), subsets=rng.randint(2, 12),
                    iters=rng.randint(3, 8))
    if kind == "batch":
        return dict(kind=kind, jobs=rng.randint(3, 8), pick=rng.randint(10, 10000), subsets=rng.randint(4, 12),
                    iters=rng.randint(4, 12))
    if kind in ("forward", "back"):
        f64 = rng.random() < 0.5
        n = _log(rng, 48, 400 if f64 else 640)
        return dict(kind=kind, n=n, views=_log(rng, 40, 720), bins=int(n * rng.uniform(1.0, 1.5)), f64=f64)
    if kind == "goldenc":
        return dict(kind=kind, iter_alt=1, iter_image=rng.randint(2, 10), iter_edge=rng.randint(2, 10))
    n = _log(rng, 24, 176)
    c = dict(kind=kind, nx=n, ny=max(16, int(n * rng.uniform(0.7, 1.0))), nz=max(8, int(n * rng.uniform(0.4, 1.2))),
             views=_log(rng, 24, 240), rows=2 * max(8, int(n * rng.uniform(0.6, 1.1))),
             cols=2 * max(8, int(n * rng.uniform(0.7, 1.2))))
    if kind == "cone_at":
        c["subsets"] = rng.randint(2, 12)
    return c


# ---- geometries ---------------------------------------------------------------


def _geometry(c, seed=0):
    k = c["kind"]
    if k == "slice":
        g = mi.arc_geometry(c["n"], 0.5859 * 874 / c["n"], c["views"], c["bins"], ARC_PITCH * 736 / c["bins"], ARC_SOD,
                            ARC_SDD, ARC_OFF)
        r = np.random.default_rng(seed)
        # one turn of the table, each view a little off its even place
        step = 360.0 / c["views"]
        return g.with_views(r.uniform(0.0, 360.0) + step * (np.arange(c["views"]) + r.uniform(-0.2, 0.2, c["views"])))
    if c.get("beam") == "arc":
        return mi.arc_geometry(c["n"], 0.5859 * 874 / c["n"], c["views"], c["bins"], ARC_PITCH * 736 / c["bins"],
                               ARC_SOD, ARC_SDD, ARC_OFF)
    if c.get("beam") == "parallel":
        return mi.parallel_geometry(c["n"], c["views"], c["bins"], 0)
    return mi.fan_geometry(c["n"], FOV / c["n"], c["views"], c["bins"], 736.0 / c["bins"], SOD, SDD)


def _jobs(c):
    """The worklist: slices over a few protocols, as a department runs them."""
    r = np.random.default_rng(c["pick"])
    protocols = [(int(r.choice([256, 384, 512])), int(r.choice([360, 720, 1152])), int(r.choice([512, 736])))
                 for _ in range(max(2, c["jobs"] // 3))]
    return [dict(kind="at", n=n, views=v, bins=b) for n, v, b in (protocols[int(r.integers(len(protocols)))]
                                                                 for _ in range(c["jobs"]))]


def _cone(c):
    n = max(c["nx"], c["ny"])
    if n == 512:
        return mi.cone_geometry(c["nx"], c["ny"], c["nz"], c["views"], c["rows"], c["cols"], 0.5, 0.4, 600.0, 1000.0)
    return mi.cone_geometry(c["nx"], c["ny"], c["nz"], c["views"], c["rows"], c["cols"], 128.0 / n, 256.0 / (2 * n),
                            450.0, 836.7)


def _params(c, f64=False, iters=None):
    return mi.at_params(ALPHA, BETA, EPS, n_subsets=min(c.get("subsets", 1), c.get("views", 1 << 30)),
                        max_iters=iters or c.get("iters", 1), precision=mi.MI_FP64 if f64 else mi.MI_FP32)


# ---- rays and inputs, on the GPU in float64 -----------------------------------


def _rays(g):
    """End points (sx, sy, dx, dy) [views, bins] of a 2D beam's rays in mm, image corner at the origin."""
    V, B = g.n_views, g.n_bins
    half = g.nx * g.pixel_mm / 2.0
    v = torch.arange(V, dtype=torch.float64, device="cuda")
    if g.beam == mi.MI_BEAM_PARALLEL:
        th = (math.pi / V * v)[:, None]
        off = (torch.arange(B, dtype=torch.float64, device="cuda") - B // 2)[None, :]
        px, py = -torch.sin(th) * off + g.nx / 2.0, torch.cos(th) * off + g.nx / 2.0
        reach = 2.0 * g.nx
        return (py - reach * torch.sin(th), px - reach * torch.cos(th), py + reach * torch.sin(th),
                px + reach * torch.cos(th))
    if g.beam == mi.MI_BEAM_FAN_ARC:
        a = torch.from_numpy(g._views.copy()).cuda() if getattr(g, "_views", None) is not None else g.span_deg * v / V
        a = (a / 180.0 * math.pi)[:, None]
        b = ((torch.arange(B, dtype=torch.float64, device="cuda") - B // 2 + g.det_offset) * (g.bin_mm * math.pi / 180.0)
             + math.pi)[None, :]
        sx, sy = g.sod_mm * torch.cos(a) + half, g.sod_mm * torch.sin(a) + half
        return (sx.expand(V, B), sy.expand(V, B), g.sdd_mm * torch.cos(a + b) + sx, g.sdd_mm * torch.sin(a + b) + sy)
    th = (g.span_deg * (math.pi / 180.0) * v / V)[:, None]
    c, s = torch.cos(th), torch.sin(th)
    x1 = ((torch.arange(B, dtype=torch.float64, device="cuda") - B // 2) + 0.5 + g.det_offset)[None, :] * g.bin_mm
    y1 = g.sdd_mm - g.sod_mm
    return ((s * g.sod_mm + half).expand(V, B), (-c * g.sod_mm + half).expand(V, B), c * x1 - s * y1 + half,
            s * x1 + c * y1 + half)


def _ellipses(n, fov, seed, mu_max):
    r = np.random.default_rng(seed)
    return [(r.uniform(-0.35 * fov, 0.35 * fov), r.uniform(-0.35 * fov, 0.35 * fov), r.uniform(0.015, 0.28) * fov,
             r.uniform(0.015, 0.28) * fov, r.uniform(0.0, math.pi), r.uniform(0.0, mu_max)) for _ in range(n)]


def _noisy(p, i0, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    n = torch.poisson(i0 * torch.exp(-p), generator=gen)
    return -torch.log(n.clamp_(min=1.0) / i0)


def _sinogram(g, seed):
    sx, sy, dx, dy = _rays(g)
    half = g.nx * g.pixel_mm / 2.0
    L = torch.hypot(dx - sx, dy - sy)
    ux, uy = (dx - sx) / L, (dy - sy) / L
    p = torch.zeros_like(L)
    fov = g.nx * g.pixel_mm
    for cx, cy, a, b, t, mu in _ellipses(10, fov, seed, 0.02 * FOV / fov):
        ct, st = math.cos(t), math.sin(t)
        qx, qy = sx - half - cx, sy - half - cy
        qx, qy = (ct * qx + st * qy) / a, (-st * qx + ct * qy) / b
        vx, vy = (ct * ux + st * uy) / a, (-st * ux + ct * uy) / b
        A = vx * vx + vy * vy
        B = 2 * (qx * vx + qy * vy)
        p += mu * torch.sqrt((B * B - 4 * A * (qx * qx + qy * qy - 1)).clamp_(min=0.0)) / A
    return _noisy(p, 2e4, seed)


def _image(n, pixel, seed):
    half = n * pixel / 2.0
    c = (torch.arange(n, dtype=torch.float64, device="cuda") + 0.5) * pixel - half
    X, Y = c[:, None], c[None, :]
    img = torch.zeros(n, n, dtype=torch.float64, device="cuda")
    for cx, cy, a, b, t, mu in _ellipses(10, n * pixel, seed, 0.02 * FOV / (n * pixel)):
        xr = math.cos(t) * (X - cx) + math.sin(t) * (Y - cy)
        yr = -math.sin(t) * (X - cx) + math.cos(t) * (Y - cy)
        img += mu * ((xr / a) ** 2 + (yr / b) ** 2 <= 1.0)
    return img


def _ellipsoids(g, seed):
    r = np.random.default_rng(seed)
    fov = [g.nx * g.sample_mm, g.ny * g.sample_mm, g.nz * g.sample_mm]
    m = min(fov)
    return [([r.uniform(-0.35, 0.35) * f for f in fov], [r.uniform(0.03, 0.25) * m for _ in range(3)],
             r.uniform(0.0, math.pi), r.uniform(0.0, 2.0) / m) for _ in range(10)]


def _volume(g, seed):
    ax = [((torch.arange(n, device="cuda", dtype=torch.float32) + 0.5) - n / 2) * g.sample_mm for n in (g.nx, g.ny, g.nz)]
    X, Y, Z = ax[0][None, :, None], ax[1][None, None, :], ax[2][:, None, None]
    vol = torch.zeros(g.nz, g.nx, g.ny, device="cuda")
    for (cx, cy, cz), (a, b, c), t, mu in _ellipsoids(g, seed):
        xr = math.cos(t) * (X - cx) + math.sin(t) * (Y - cy)
        yr = -math.sin(t) * (X - cx) + math.cos(t) * (Y - cy)
        vol += mu * (((xr / a) ** 2 + (yr / b) ** 2 + ((Z - cz) / c) ** 2) <= 1.0)
    return vol


def _cone_sinogram(g, seed):
    """[view][row][col] noisy line integrals of the ellipsoids along the cone beam's rays."""
    out = torch.empty(g.n_views, g.n_rows, g.n_cols, device="cuda")
    h = g.n_rows // 2
    x1 = ((torch.arange(g.n_cols, device="cuda", dtype=torch.float32) - h) + 0.5) * g.pixel_mm
    z1 = (((h - torch.arange(g.n_rows, device="cuda", dtype=torch.float32)) - 0.5) * g.pixel_mm)[:, None]
    y1 = g.sdd_mm - g.sod_mm
    things = _ellipsoids(g, seed)
    for v in range(g.n_views):
        c, s = math.cos(2 * math.pi * v / g.n_views), math.sin(2 * math.pi * v / g.n_views)
        sx, sy = s * g.sod_mm, -c * g.sod_mm
        rx, ry = c * x1 - s * y1 - sx, s * x1 + c * y1 - sy
        L = torch.sqrt(rx * rx + ry * ry + z1 * z1)
        p = torch.zeros_like(L)
        for (cx, cy, cz), (a, b, d), t, mu in things:
            ct, st = math.cos(t), math.sin(t)
            qx, qy, qz = (ct * (sx - cx) + st * (sy - cy)) / a, (-st * (sx - cx) + ct * (sy - cy)) / b, -cz / d
            vx, vy, vz = (ct * rx + st * ry) / a, (-st * rx + ct * ry) / b, z1 / d
            A = vx * vx + vy * vy + vz * vz
            B = vx * qx + vy * qy + vz * qz
            p += mu * torch.sqrt((B * B - A * (qx * qx + qy * qy + qz * qz - 1)).clamp_(min=0.0)) / A
        out[v] = p * L
    return _noisy(out, 5e4, seed)


# ---- prepare / run ---------------------------------------------------------------

_CTX = None
_FOR = None


def _context(c):
    """The program's context.  It keeps the geometries of one case at a time."""
    global _CTX, _FOR
    if _CTX is None:
        _CTX = mi.Context(0)
    key = sorted((k, v) for k, v in c.items() if k != "name")
    if key != _FOR:
        _CTX.trim()
        _FOR = key
    return _CTX


def _host(t, f64):
    return t.to(torch.float64 if f64 else torch.float32).cpu().numpy()


def prepare(case, seed):
    k = case["kind"]
    ctx = _context(case)
    st = dict(kind=k, ctx=ctx)
    if k in ("at", "slice"):
        f64 = case.get("f64", False)
        g = _geometry(case, seed)
        st.update(g=g, p=_params(case, f64), sino=_host(_sinogram(g, seed), f64))
        if k == "at":
            ctx.prepare(g, st["p"].n_subsets)
    elif k == "batch":
        st["S"] = case["subsets"]
        st["jobs"] = []
        for i, j in enumerate(_jobs(case)):
            g = _geometry(j)
            st["jobs"].append((g, _host(_sinogram(g, seed * 64 + i), False), _params(case)))
            ctx.prepare(g, case["subsets"])
    elif k in ("forward", "back"):
        f64 = case["f64"]
        g = _geometry(case)
        st.update(g=g, dtype=np.float64 if f64 else np.float32)
        st["x"] = _host(_image(g.nx, g.pixel_mm, seed) if k == "forward" else _sinogram(g, seed), f64)
    elif k == "goldenc":
        g = mi.goldenc_geometry()
        st.update(g=g, p=mi.at_params(1000.0, 0.002, 1e-4, iter_alt=case["iter_alt"], iter_image=case["iter_image"],
                                      iter_edge=case["iter_edge"], precision=mi.MI_FP64))
        st["sino"] = ctx.forward(g, _host(_image(512, 1.0, seed), True) * 50.0, np.float64)
    else:
        g = _cone(case)
        st["g"] = g
        if k == "cone_fp":
            st.update(vol=_volume(g, seed), sino=torch.empty(g.n_views, g.n_rows, g.n_cols, device="cuda"))
        else:
            st["sino"] = _cone_sinogram(g, seed)
            shape = (g.nz, g.nx, g.ny)
            if k == "cone_bp":
                st["vol"] = torch.empty(shape, device="cuda")
            else:
                st.update(p=_params(case, iters=1), u=torch.zeros(shape, device="cuda"), v=torch.ones(shape, device="cuda"))
    return st


def run(st):
    k, ctx = st["kind"], st["ctx"]
    if k == "at":
        u, v, rep = ctx.at_reconstruct(st["g"], st["sino"], st["p"])
        return [u, v, rep.data_fidelity, rep.iterations]
    if k == "slice":
        ctx.trim()   # the slice before it: its geometry never comes back
        u, v, rep = ctx.at_reconstruct(st["g"], st["sino"], st["p"])
        return [u, v, rep.data_fidelity, rep.iterations]
    if k == "batch":
        b = ctx.batch(st["S"])
        ids = [b.submit(g, sino, p) for g, sino, p in st["jobs"]]
        b.run()
        out = [b.read(i) for i in ids]
        b.close()
        return out
    if k == "forward":
        return ctx.forward(st["g"], st["x"], st["dtype"])
    if k == "back":
        return ctx.backproject(st["g"], st["x"], st["dtype"])
    if k == "goldenc":
        f, v, _ = ctx.mumford_shah(st["g"], st["sino"], st["p"])
        return [f, v]
    if k == "cone_fp":
        ctx.cone_forward_dev(st["g"], st["vol"].data_ptr(), st["sino"].data_ptr())
        return st["sino"]
    if k == "cone_bp":
        ctx.cone_backproject_dev(st["g"], st["sino"].data_ptr(), st["vol"].data_ptr())
        return st["vol"]
    rep = ctx.cone_at_reconstruct_dev(st["g"], st["sino"].data_ptr(), st["u"].data_ptr(), st["v"].data_ptr(), st["p"])
    return [st["u"], st["v"], rep.data_fidelity]


# ---- what a pass cannot do without ---------------------------------------------------


def work(case):
    """Bytes: each input read and each output written once.  Flops: a multiply and an add for each (ray, pixel)
    crossing of each projection (a ray meets about 1.1 pixels per image row, 1.34 voxels per volume row)."""
    k = case["kind"]
    if k == "batch":
        w = [work(dict(j, iters=case["iters"])) for j in _jobs(case)]
        return {"bytes": sum(x["bytes"] for x in w), "flops": sum(x["flops"] for x in w)}
    if k == "goldenc":
        # two projections per CG iteration, A twice for the energies
        return {"bytes": 8.0 * (180 * 767 + 2 * 512 * 512),
                "flops": 2.0 * 1.1 * 512 * 180 * 767 * 3 * case["iter_alt"] * case["iter_image"]}
    if k.startswith("cone"):
        rays, vox = case["views"] * case["rows"] * case["cols"], case["nx"] * case["ny"] * case["nz"]
        proj = 3 if k == "cone_at" else 1
        return {"bytes": 4.0 * (rays + (4 if k == "cone_at" else 1) * vox),
                "flops": 2.0 * 1.34 * rays * max(case["nx"], case["ny"]) * proj}
    sz = 8.0 if case.get("f64") else 4.0
    rays, pix = case["views"] * case["bins"], case["n"] ** 2
    if k in ("forward", "back"):
        return {"bytes": sz * (rays + pix), "flops": 2.0 * 1.1 * rays * case["n"]}
    return {"bytes": sz * (rays + 2 * pix), "flops": 2.0 * 1.1 * rays * case["n"] * 3 * case["iters"]}


# ---- the same in 64 bits, plain torch ------------------------------------------------


def _system(g, views):
    """(index, length) [rays, k] of the rays of `views`: all crossings of the grid lines, sorted; a piece that begins
    within 0.05 mm of the exit is left out, as the tracer this beam stands for leaves it out."""
    sx, sy, dx, dy = (t[views].reshape(-1, 1) for t in _rays(g))
    rx, ry = dx - sx, dy - sy
    L = torch.sqrt(rx * rx + ry * ry)
    w = g.pixel_mm
    gx = torch.arange(g.nx + 1, dtype=torch.float64, device="cuda")[None, :] * w
    gy = torch.arange(g.ny + 1, dtype=torch.float64, device="cuda")[None, :] * w
    ax, ay = L * (gx - sx) / rx, L * (gy - sy) / ry
    lo = torch.maximum(torch.minimum(ax[:, :1], ax[:, -1:]), torch.minimum(ay[:, :1], ay[:, -1:])).clamp(min=0.0)
    hi = torch.minimum(torch.minimum(torch.maximum(ax[:, :1], ax[:, -1:]), torch.maximum(ay[:, :1], ay[:, -1:])), L)
    hi = torch.maximum(hi, lo)
    t = torch.cat([ax, ay], 1)
    t = torch.minimum(torch.maximum(t, lo), hi).sort(1).values
    ln = t[:, 1:] - t[:, :-1]
    ln *= t[:, :-1] < hi - 5e-2
    mid = 0.5 * (t[:, 1:] + t[:, :-1])
    ix = ((sx + mid * (rx / L)) / w).floor_().clamp_(0, g.nx - 1).to(torch.int32)
    ix *= g.ny
    ix += ((sy + mid * (ry / L)) / w).floor_().clamp_(0, g.ny - 1).to(torch.int32)
    return ix, ln


def _fp(A, x):
    ix, ln = A
    out = torch.empty(ix.shape[0], dtype=torch.float64, device="cuda")
    for r in range(0, ix.shape[0], 1 << 16):
        out[r:r + (1 << 16)] = (x[ix[r:r + (1 << 16)]] * ln[r:r + (1 << 16)]).sum(1)
    return out


def _bp(A, y, npix):
    ix, ln = A
    out = torch.zeros(npix, dtype=torch.float64, device="cuda")
    for r in range(0, ix.shape[0], 1 << 16):
        out.index_add_(0, ix[r:r + (1 << 16)].reshape(-1), (ln[r:r + (1 << 16)] * y[r:r + (1 << 16), None]).reshape(-1))
    return out


def _shift(a, di, dj, pad):
    """a at (i + di, j + dj), `pad` outside."""
    p = torch.nn.functional.pad(a, (1, 1, 1, 1), value=pad)
    return p[1 + di:1 + di + a.shape[0], 1 + dj:1 + dj + a.shape[1]]


def _reversed_bits(S):
    bits = max(0, (S - 1).bit_length())
    return [r for r in (int(format(i, "0%db" % bits)[::-1], 2) if bits else 0 for i in range(1 << bits)) if r < S]


def _os_at(g, sino, S, iters):
    """The ordered-subset Ambrosio-Tortorelli iteration from u = 0, v = 1 (one edge step a pass, no median)."""
    n, npix = g.nx, g.nx * g.ny
    subs = []
    for s in _reversed_bits(S):
        views = torch.arange(s, g.n_views, S, device="cuda")
        subs.append((_system(g, views), sino[views].reshape(-1)))
    u = torch.zeros(n, g.ny, dtype=torch.float64, device="cuda")
    v = torch.ones_like(u)
    e2 = 0.01 * EPS * EPS
    df = 0.0
    for _ in range(iters):
        df = 0.0
        for A, y in subs:
            r = y - _fp(A, u.reshape(-1))
            df += float((r * r).sum())
            ud, ur, uu, ul = (_shift(u, *o, 0.0) for o in ((1, 0), (0, 1), (-1, 0), (0, -1)))
            vu, vl = _shift(v, -1, 0, 1.0), _shift(v, 0, -1, 1.0)
            reg = v * v * (ud - u) + v * v * (ur - u) - vu * vu * (u - uu) - vl * vl * (u - ul) + e2 * (
                ud + ur - 4 * u + uu + ul)
            d = S * _bp(A, r, npix).reshape(n, g.ny) + ALPHA * reg
            ad = _fp(A, d.reshape(-1))
            nv = ((v * v + e2) * ((d - _shift(d, -1, 0, 0.0)) ** 2 + (d - _shift(d, 0, -1, 0.0)) ** 2)).sum()
            den = S * (ad * ad).sum() + ALPHA * nv
            u = u + ((d * d).sum() / den if den > 0 else 0.0) * d
        fx = 0.5 * (_shift(u, 1, 0, 0.0) - _shift(u, -1, 0, 0.0))
        fy = 0.5 * (_shift(u, 0, 1, 0.0) - _shift(u, 0, -1, 0.0))
        m = fx * fx + fy * fy
        lap = 0.25 * (_shift(v, 1, 0, 1.0) + _shift(v, 0, 1, 1.0) - 4 * v + _shift(v, -1, 0, 1.0) + _shift(v, 0, -1, 1.0))
        w = -(ALPHA * v * m - BETA * EPS * lap + BETA * (v - 1) / (4 * EPS))
        wx = 0.5 * (_shift(w, 1, 0, 0.0) - _shift(w, -1, 0, 0.0))
        wy = 0.5 * (_shift(w, 0, 1, 0.0) - _shift(w, 0, -1, 0.0))
        nd = (w * w).sum()
        c = nd / (ALPHA * (m * w * w).sum() + BETA * EPS * (wx * wx + wy * wy).sum() + BETA / (4 * EPS) * nd)
        v = (v + c * w).clamp(0.0, 1.0)
    return u, v, df


def _cone_lengths_bp(g, sino):
    """Transpose of the exact lengths of the cone beam's rays in the voxels, gathered voxel by voxel.  The rays' end
    points are the geometry's own float32 ones."""
    f = torch.float32
    h = g.n_rows // 2
    dev = "cuda"
    vol = torch.zeros(g.nz, g.nx, g.ny, dtype=torch.float64, device=dev)
    col, row = torch.arange(g.n_cols, device=dev), torch.arange(g.n_rows, device=dev)
    X1 = ((col - h).double() + 0.5).to(f) * f_(g.pixel_mm)
    dz = (((h - row).double() - 0.5).to(f) * f_(g.pixel_mm) / f_(g.sample_mm)).double().add(g.nz / 2.0).to(f).double()
    sz = g.nz / 2.0
    w = dz - sz
    x = torch.arange(g.nx, dtype=torch.float64, device=dev)[None, :, None]
    y = torch.arange(g.ny, dtype=torch.float64, device=dev)[None, None, :]
    z = torch.arange(g.nz, dtype=torch.float64, device=dev)[:, None, None]
    k, r0 = g.sdd_mm / g.pixel_mm, g.sod_mm / g.sample_mm
    for v in range(g.n_views):
        th = np.float32(np.float64(np.float32(np.float32(v) / np.float32(g.n_views)) * np.float32(2)) * math.pi)
        c, s = torch.tensor(np.cos(th), device=dev, dtype=f), torch.tensor(np.sin(th), device=dev, dtype=f)
        Ys, Y1 = torch.tensor(-np.float32(g.sod_mm), device=dev), torch.tensor(np.float32(g.sdd_mm) - np.float32(g.sod_mm),
                                                                              device=dev)
        sx = (-s * Ys / f_(g.sample_mm)).double().add(g.nx / 2.0).to(f).double()
        sy = (c * Ys / f_(g.sample_mm)).double().add(g.ny / 2.0).to(f).double()
        dx = ((c * X1 + -s * Y1) / f_(g.sample_mm)).double().add(g.nx / 2.0).to(f).double()
        dy = ((s * X1 + c * Y1) / f_(g.sample_mm)).double().add(g.ny / 2.0).to(f).double()
        rx, ry = dx - sx, dy - sy
        # panel columns and rows a voxel can meet
        cf, zf = [], []
        for a in (0, 1):
            for b in (0, 1):
                px, py = x + a - g.nx / 2.0, y + b - g.ny / 2.0
                dep = -float(s) * px + float(c) * py + r0
                cf.append((float(c) * px + float(s) * py) * k / dep + h - 0.5)
                zf += [h - 0.5 - (z - sz) * k / dep, h - 0.5 - (z + 1 - sz) * k / dep]
        c0 = torch.stack(cf).amin(0).sub(0.01).ceil().long()
        z0 = torch.stack(zf).amin(0).sub(0.01).ceil().long()
        nc = int((torch.stack(cf).amax(0) + 0.01).floor().long().sub(c0).max()) + 1
        nr = int((torch.stack(zf).amax(0) + 0.01).floor().long().sub(z0).max()) + 1
        for i in range(nc):
            ci = c0 + i
            cin = (ci >= 0) & (ci < g.n_cols)
            cc = ci.clamp(0, g.n_cols - 1)
            tx0, tx1 = (x - sx) / rx[cc], (x + 1 - sx) / rx[cc]
            ty0, ty1 = (y - sy) / ry[cc], (y + 1 - sy) / ry[cc]
            lo = torch.maximum(torch.minimum(tx0, tx1), torch.minimum(ty0, ty1)).clamp(min=0.0)
            hi = torch.minimum(torch.maximum(tx0, tx1), torch.maximum(ty0, ty1)).clamp(max=1.0)
            l2 = rx[cc] ** 2 + ry[cc] ** 2
            for j in range(nr):
                rj = z0 + j
                ok = cin & (rj >= 0) & (rj < g.n_rows)
                rr = rj.clamp(0, g.n_rows - 1)
                wr = w[rr]
                ta, tb = (z - sz) / wr, (z + 1 - sz) / wr
                e = torch.minimum(hi, torch.maximum(ta, tb)) - torch.maximum(lo, torch.minimum(ta, tb))
                vol += torch.where(ok, e.clamp(min=0.0) * torch.sqrt(l2 + wr * wr) * sino[v][rr, cc], 0.0)
    return vol


def f_(x):
    return torch.tensor(np.float32(x), device="cuda")


def exact(case, seed):
    k = case["kind"]
    if k in ("at", "slice"):
        if case.get("beam") == "parallel":
            return None   # its lengths are the float tracer's own
        g = _geometry(case, seed)
        f64 = case.get("f64", False)
        y = torch.from_numpy(_host(_sinogram(g, seed), f64)).cuda().double()
        u, v, df = _os_at(g, y, min(case["subsets"], g.n_views), case["iters"])
        return [u, v, df, None]
    if k == "batch":
        out = []
        for i, j in enumerate(_jobs(case)):
            g = _geometry(j)
            y = torch.from_numpy(_host(_sinogram(g, seed * 64 + i), False)).cuda().double()
            out.append(list(_os_at(g, y, case["subsets"], case["iters"])[:2]))
        return out
    if k in ("forward", "back"):
        g = _geometry(case)
        every = torch.arange(g.n_views, device="cuda")
        x = _image(g.nx, g.pixel_mm, seed) if k == "forward" else _sinogram(g, seed)
        x = torch.from_numpy(_host(x, case["f64"])).cuda().double()
        if k == "forward":
            return torch.cat([_fp(_system(g, v), x.reshape(-1)).reshape(-1, g.n_bins) for v in every.split(64)])
        return sum(_bp(_system(g, v), x[v].reshape(-1), g.nx * g.ny) for v in every.split(64)).reshape(g.nx, g.ny)
    if k == "cone_bp" and case["nx"] <= 192:
        g = _cone(case)
        return _cone_lengths_bp(g, _cone_sinogram(g, seed).double())
    return None
