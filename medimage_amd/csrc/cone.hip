// 3D cone-beam projectors, industry3d geometry (flat panel, circular orbit).
//
// Rays.  cone() of industry3d/src/tracing.cpp:51-81 with rotate_2d of
// industry3d/src/utility.cpp:82-98, in float: the source (0, -SOD, 0) and
// the panel pixel ((col - HALFDET + 0.5) PIXELSIZE, SDD - SOD,
// (HALFDET - row - 0.5) PIXELSIZE) are rotated by the view angle, divided
// by SAMPLESIZE and shifted by N / 2 (in double, as the reference's
// `+= NX / 2.0` does).  The view's cos / sin come from host tables made
// with the C library's cosf / sinf, which the reference calls.  BEAM
// "Parallel" takes parallel() (tracing.cpp:9-49) instead: start and end share
// the column's x and the row's z, every axis shifted by HALFSIZE.
//
// Forward projection.  One lane per ray walks forward_proj
// (industry3d/src/tracing.cpp:123-307) in float, operation for operation,
// so the (voxel, length) sequence is the reference's bit for bit; the walk
// ends where the reference's does (lambda0 >= lambda_max - 0.05, tested in
// double) or when its voxel leaves the volume (where the reference would
// index outside its arrays; only rays through an edge or corner of the
// volume).  Products vol * len are summed in double in walk order and
// rounded once.  Each wave takes an 8 x 8 tile of one view's panel, so the
// 64 rays of a wave cross neighbouring voxels at each step; workgroups (16
// x 16 pixels) go by band of panel rows.
// Steps are taken in groups of 8: the group's voxel offsets and lengths are
// computed first, its 8 loads issued together, then accumulated in order.
//
// Back projection (gather form, no atomics).  The usual cone beam goes by
// panel patches (k_cone_bp_patch, where it is described); the parallel beam
// and a source so near that a voxel's chord spans several rows go ray by ray
// (k_cone_bp): one lane per voxel column
// (x, y) and a chunk of kZc slices along z.  For each view the four corners
// of the column are projected onto the panel: the columns whose rays can
// cross it, and per slice the rows.  For each candidate ray the exact length
// inside the voxel is the slab clip of the ray's parameter interval: the x / y
// slab in double once per (view, column) from a per-geometry table of
// 1 / (d - s), shared by the lane's kZc slices; the z slab per row from a
// per-row 1 / w table (copied to LDS), relative to the column's entry
// parameter so that the float differences keep full precision; times the ray
// length in float.  For the parallel beam the footprint is orthographic and
// a row's ray crosses a slice over its whole x / y chord or not at all.
// sino * length is summed in double, per (view, column, slice) over the rows
// in a register and then into the voxel's sum in LDS, in a fixed order.  A
// back projection over many views runs in chunks of kBpViewChunk views (their
// sinogram rows stay in the caches while every workgroup sweeps them), the
// double sums carried between chunks in a scratch volume.
#include "cone.hpp"

#include <mutex>

#include <cfloat>
#include <climits>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

namespace mi {

namespace {

constexpr int kConeTile = 16;   // forward: 16 x 16 panel pixels per workgroup
constexpr int kConeGroup = 8;   // forward: walk steps per load group
// Back projection: slices per lane.  A lane's per-view work on its column
// (footprint, panel columns, x / y clip) is shared by its kZc slices, whose
// double sums live in LDS (kZc x 2 KiB per workgroup, beside the rows' 1 / w):
// 512^3, 720 views of 1024 x 768 (without k_cone_bp_patch): 644 ms with 6 (18 KiB, 8 workgroups
// per CU), 663 with 7, 674 with 5, 680 with 8 (22 KiB, 7 per CU), 689 with 4.
#ifndef MI_CONE_ZC
#define MI_CONE_ZC 6
#endif
constexpr int kZc = MI_CONE_ZC;
constexpr int kBpViewChunk = 36; // back projection: views per launch (their rows stay in the caches)
constexpr int kBpRowLds = 4096;  // back projection: panels up to this many rows keep 1 / w in LDS

__device__ __forceinline__ void cone_rot(float &x, float &y, float c, float s) {
    float d0 = 0.0f, d1 = 0.0f;
    d0 += c * x;
    d1 += s * x;
    d0 += -s * y;
    d1 += c * y;
    x = d0;
    y = d1;
}

// Source point of a view (voxel units, volume corner at the origin).
__device__ __forceinline__ void cone_source(const ConeDev &g, float c, float s, float &sx, float &sy, float &sz) {
    float X = 0.0f, Y = -g.sod, Z = 0.0f;
    cone_rot(X, Y, c, s);
    X /= g.sample;
    Z /= g.sample;
    Y /= g.sample;
    sx = (float)((double)X + g.nx / 2.0);
    sy = (float)((double)Y + g.ny / 2.0);
    sz = (float)((double)Z + g.nz / 2.0);
}

// In-plane detector point of column col (x, y).
__device__ __forceinline__ void cone_det_xy(const ConeDev &g, float c, float s, int col, float &dx, float &dy) {
    float X = (float)((double)(col - g.halfdet) + 0.5);
    X *= g.pixel;
    float Y = g.sdd - g.sod;
    cone_rot(X, Y, c, s);
    X /= g.sample;
    Y /= g.sample;
    dx = (float)((double)X + g.nx / 2.0);
    dy = (float)((double)Y + g.ny / 2.0);
}

// Height of row `row` of the panel.
__device__ __host__ __forceinline__ float cone_det_z(const ConeDev &g, int row) {
    float Z = (float)((double)(g.halfdet - row) - 0.5);
    Z *= g.pixel;
    Z /= g.sample;
    return (float)((double)Z + g.nz / 2.0);
}

// parallel() of industry3d/src/tracing.cpp:9-49: start and end share the
// panel column's x and the row's z; every axis is shifted by HALFSIZE (a
// float), in float.
__device__ __forceinline__ void par_endpoints(const ConeDev &g, float c, float s, int row, int col, float &sx,
                                              float &sy, float &sz, float &dx, float &dy, float &dz) {
    float X0 = (float)((double)col + 0.5 - g.halfdet);
    X0 *= g.pixel;
    float Y0 = -g.sod;
    float Z0 = (float)((double)(g.halfdet - row) - 0.5);
    Z0 *= g.pixel;
    float X1 = X0, Y1 = g.sdd - g.sod, Z1 = Z0;
    cone_rot(X0, Y0, c, s);
    cone_rot(X1, Y1, c, s);
    sx = X0 / g.sample + g.halfsize;
    sy = Y0 / g.sample + g.halfsize;
    sz = Z0 / g.sample + g.halfsize;
    dx = X1 / g.sample + g.halfsize;
    dy = Y1 / g.sample + g.halfsize;
    dz = Z1 / g.sample + g.halfsize;
}

// End points of ray (view with cos c / sin s, row, col) of either beam.
__device__ __forceinline__ void ray_points(const ConeDev &g, float c, float s, int row, int col, float &sx, float &sy,
                                           float &sz, float &dx, float &dy, float &dz) {
    if (g.parallel) {
        par_endpoints(g, c, s, row, col, sx, sy, sz, dx, dy, dz);
    } else {
        cone_source(g, c, s, sx, sy, sz);
        cone_det_xy(g, c, s, col, dx, dy);
        dz = cone_det_z(g, row);
    }
}

// LAMBDA_X of industry3d/src/tracing.cpp:83-85.
__device__ __forceinline__ float cone_lam(float i, float s, float d, float L) { return L * (i - s) / (d - s); }

// Walk state of forward_proj: lam0 the current parameter, l* the next
// crossings, st* their increments, (vx, vy, vz) the voxel.
struct ConeWalk {
    float lam0, lx, ly, lz, stx, sty, stz, stop;
    int vx, vy, vz, sgx, sgy, sgz;
};

// Entry part of forward_proj (tracing.cpp:142-249).  stop is the smallest
// float T with (double)T >= (double)lambda_max - 5.e-2, so that the float
// test lam0 < T equals the reference's double test.
__device__ __forceinline__ bool cone_walk_init(const ConeDev &g, float sx, float sy, float sz, float dx, float dy,
                                               float dz, ConeWalk &w) {
    const float rx = dx - sx, ry = dy - sy, rz = dz - sz;
    const float L = sqrtf(rx * rx + ry * ry + rz * rz);
    float lmin = 0.0f, lmax = L, l0, lN, t;
    const int sgx = (rx > 0) ? 1 : -1, sgy = (ry > 0) ? 1 : -1, sgz = (rz > 0) ? 1 : -1;
    const float ax = fabsf(rx), ay = fabsf(ry), az = fabsf(rz);
    const float stx = ((double)ax > 1.e-4) ? (L / ax) : 1.e6f;
    const float sty = ((double)ay > 1.e-4) ? (L / ay) : 1.e6f;
    const float stz = ((double)az > 1.e-4) ? (L / az) : 1.e6f;
    int index = 0;
    l0 = cone_lam(0.0f, sx, dx, L);
    lN = cone_lam((float)g.nx, sx, dx, L);
    t = (l0 < lN) ? l0 : lN;
    lmin = (lmin > t) ? lmin : t;
    if (lmin == t) index = 1;
    t = (l0 > lN) ? l0 : lN;
    lmax = (lmax < t) ? lmax : t;
    l0 = cone_lam(0.0f, sy, dy, L);
    lN = cone_lam((float)g.ny, sy, dy, L);
    t = (l0 < lN) ? l0 : lN;
    lmin = (lmin > t) ? lmin : t;
    if (lmin == t) index = 2;
    t = (l0 > lN) ? l0 : lN;
    lmax = (lmax < t) ? lmax : t;
    l0 = cone_lam(0.0f, sz, dz, L);
    lN = cone_lam((float)g.nz, sz, dz, L);
    t = (l0 < lN) ? l0 : lN;
    lmin = (lmin > t) ? lmin : t;
    if (lmin == t) index = 3;
    t = (l0 > lN) ? l0 : lN;
    lmax = (lmax < t) ? lmax : t;
    if (lmin >= lmax) return false;

    const float lam0 = lmin;
    float lx, ly, lz;
    int vx, vy, vz;
    if (index == 1) {
        vx = (sgx == 1) ? 0 : g.nx - 1;
        lx = lam0 + stx;
        vy = (int)(sy + lam0 * ry / L);
        ly = ((double)ay < 1.e-4) ? 1.e6f : cone_lam((float)vy + (float)(sgy > 0), sy, dy, L);
        vz = (int)(sz + lam0 * rz / L);
        lz = ((double)az < 1.e-4) ? 1.e6f : cone_lam((float)vz + (float)(sgz > 0), sz, dz, L);
    } else if (index == 2) {
        vy = (sgy == 1) ? 0 : g.ny - 1;
        ly = lam0 + sty;
        vx = (int)(sx + lam0 * rx / L);
        lx = ((double)ax < 1.e-4) ? 1.e6f : cone_lam((float)vx + (float)(sgx > 0), sx, dx, L);
        vz = (int)(sz + lam0 * rz / L);
        lz = ((double)az < 1.e-4) ? 1.e6f : cone_lam((float)vz + (float)(sgz > 0), sz, dz, L);
    } else {
        vz = (sgz == 1) ? 0 : g.nz - 1;
        lz = lam0 + stz;
        vx = (int)(sx + lam0 * rx / L);
        lx = ((double)ax < 1.e-4) ? 1.e6f : cone_lam((float)vx + (float)(sgx > 0), sx, dx, L);
        vy = (int)(sy + lam0 * ry / L);
        ly = ((double)ay < 1.e-4) ? 1.e6f : cone_lam((float)vy + (float)(sgy > 0), sy, dy, L);
    }
    const double hi = (double)lmax - 5.e-2;
    float stop = (float)hi;
    if ((double)stop < hi) stop = nextafterf(stop, INFINITY);
    w = ConeWalk{lam0, lx, ly, lz, stx, sty, stz, stop, vx, vy, vz, sgx, sgy, sgz};
    return true;
}

// One step when `live` (the walk has not ended): the current voxel's offset
// and length; state unchanged and length 0 otherwise.  The branches of the
// reference loop (tracing.cpp:268-305) become selects.
__device__ __forceinline__ void cone_step(const ConeDev &g, ConeWalk &w, bool &live, unsigned &idx, float &len) {
    // Bitwise, not short-circuit: no branch per step.  `live` never turns
    // back on, so after the end the state may keep moving: its offsets and
    // lengths are masked.
    live = live & (w.lam0 < w.stop) & ((unsigned)w.vx < (unsigned)g.nx) & ((unsigned)w.vy < (unsigned)g.ny) &
           ((unsigned)w.vz < (unsigned)g.nz);
    // The reference's branch choice (x if lx <= ly and lx <= lz, else y if
    // ly <= lz, else z) is "the first axis whose crossing equals the
    // minimum": the crossings are finite (parallel axes carry the 1e6
    // sentinel) and positive, so one three-way minimum and two equality
    // tests give the same choice and the same value.
    const float nxt = fminf(fminf(w.lx, w.ly), w.lz);
    const bool bx = w.lx == nxt;
    const bool by = !bx && w.ly == nxt;
    const bool bz = !bx && !by;
    // get_img_addr (tracing.cpp:119-121); 24-bit products (each factor is
    // below 2^24 and the volume below 2^31 voxels).
    const unsigned at = __umul24(__umul24((unsigned)w.vz, (unsigned)g.nx) + (unsigned)w.vx, (unsigned)g.ny) +
                        (unsigned)w.vy;
    idx = live ? at : 0u;
    len = live ? nxt - w.lam0 : 0.0f;
    w.lam0 = nxt;
    w.lx = bx ? w.lx + w.stx : w.lx;
    w.ly = by ? w.ly + w.sty : w.ly;
    w.lz = bz ? w.lz + w.stz : w.lz;
    w.vx += bx ? w.sgx : 0;
    w.vy += by ? w.sgy : 0;
    w.vz += bz ? w.sgz : 0;
}

__device__ __forceinline__ bool cone_ray_init(const ConeDev &g, const float *cs, int view, int row, int col,
                                              ConeWalk &w) {
    const float c = cs[2 * view], s = cs[2 * view + 1];
    float sx, sy, sz, dx, dy, dz;
    ray_points(g, c, s, row, col, sx, sy, sz, dx, dy, dz);
    return cone_walk_init(g, sx, sy, sz, dx, dy, dz, w);
}

__global__ void k_cone_trace(ConeDev g, const float *cs, int view, int row, int col, int64_t *ind, float *len,
                             int cap, int *numb) {
    if (threadIdx.x != 0) return;
    ConeWalk w;
    int n = 0;
    if (cone_ray_init(g, cs, view, row, col, w)) {
        bool live = true;
        for (;;) {
            unsigned idx;
            float l;
            cone_step(g, w, live, idx, l);
            if (!live) break;
            if (n < cap) {
                ind[n] = idx;
                len[n] = l;
            }
            ++n;
        }
    }
    *numb = n;
}

// Panel pixel of this lane: workgroup = 16 x 16 pixels of one view of the
// list (q-th entry), wave = 8 x 8 of them.  Workgroups are ordered by band of
// 16 panel rows first, then view, then column tile, so that the workgroups in
// flight trace rays through the same few slices of the volume.  Consecutive
// workgroups go to different XCDs (no XCD regrouping here): all eight XCDs
// then work on one band at a time and share its slices through the Infinity
// Cache (368 ms at C4 against 385 ms with each XCD on its own range of
// bands).  Returns false for the padding workgroups of the grid (all lanes
// alike); `ok` is false for lanes outside the panel.
__device__ __forceinline__ bool cone_fp_pixel(const ConeDev &g, int nv, unsigned &tile_id, int &q, int &row,
                                              int &col, bool &ok) {
    const int tc = (g.ncols + kConeTile - 1) / kConeTile, tr = (g.nrows + kConeTile - 1) / kConeTile;
    const unsigned b = blockIdx.x;
    const unsigned per_band = (unsigned)(nv * tc);
    tile_id = b;
    const int band = (int)(b / per_band);
    const unsigned rem = b % per_band;
    q = (int)(rem / tc);
    const int ct = (int)(rem % tc);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    row = band * kConeTile + (wv >> 1) * 8 + (lane >> 3);
    col = ct * kConeTile + (wv & 1) * 8 + (lane & 7);
    ok = row < g.nrows && col < g.ncols;
    return band < tr;
}

// Double sum over a workgroup of 256 lanes in a fixed pairing; lane 0 of
// wave 0 gets the total.
__device__ __forceinline__ double block_sum256(double x) {
    __shared__ double red[kBlock / kWave];
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}

// kConeGroup steps of a walk, none of which may be the walk's last: the
// crossings and lengths of cone_step without its tests and without the voxel's
// coordinates (its byte offset, and how many crossings of each axis are left
// before the walk leaves the volume: coordinates and lam0 only move one way,
// so a group whose last step is inside and before the end has only such
// steps).  21 instructions a step where cone_step has 33.  Returns whether
// the group was such a one; if not, nothing has changed.
//
// Bounded by the L1: its 64 lanes' loads touch 44 lines, one a clock and CU,
// and that is all of the kernel's time (512^3, 36 views of 1024 x 768: 18.6
// ms; 19.0 with cone_step alone, then with the vector issue at 90%, now at
// 50%; 176^3, 240 views of 192 x 208: 1.75 and 1.83 ms).  Groups of 6, 12 and
// 16 steps take the same time.
struct ConeFast {
    float lam0, lx, ly, lz;
    int ib;              // byte offset of the voxel
    int rx, ry, rz;      // crossings left
};
__device__ __forceinline__ bool cone_fast(ConeFast &f, const ConeWalk &w, int bx, int by, int bz,
                                          __amdgpu_buffer_rsrc_t rs, double &acc) {
    ConeFast n = f;
    float ln[kConeGroup], v[kConeGroup], before = f.lam0;
    int at[kConeGroup], cx = 0, cy = 0, ex = 0, ey = 0;
#pragma unroll
    for (int k = 0; k < kConeGroup; ++k) {
        const float nxt = fminf(fminf(n.lx, n.ly), n.lz);
        const bool isx = n.lx == nxt, isy = !isx && n.ly == nxt;
        if (k == kConeGroup - 1) {
            before = n.lam0;
            ex = cx;
            ey = cy;
        }
        at[k] = n.ib;
        ln[k] = nxt - n.lam0;
        n.lam0 = nxt;
        n.lx = isx ? n.lx + w.stx : n.lx;
        n.ly = isy ? n.ly + w.sty : n.ly;
        n.lz = (isx || isy) ? n.lz : n.lz + w.stz;
        n.ib += isx ? bx : (isy ? by : bz);
        cx += isx;
        cy += isy;
    }
    if (!(before < w.stop && f.rx > ex && f.ry > ey && f.rz > kConeGroup - 1 - ex - ey)) return false;
#pragma unroll
    for (int k = 0; k < kConeGroup; ++k)
        v[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, at[k], 0, 0));
    n.rx -= cx;
    n.ry -= cy;
    n.rz -= kConeGroup - cx - cy;
    f = n;
#pragma unroll
    for (int k = 0; k < kConeGroup; ++k) acc = __builtin_fma((double)v[k], (double)ln[k], acc);
    return true;
}

// Forward projection of the views views[0 .. nv) (sinogram [view][row][col]).
//   CFP_WRITE: out = A vol;
//   CFP_RESID: out = meas - A vol (float), part[tile] = sum of out^2;
//   CFP_SQ:    part[tile] = sum of (A vol)^2, nothing written.

template <int MODE>
__global__ __launch_bounds__(kBlock) void k_cone_fp(ConeDev g, const float *cs, const int *views, int nv,
                                                    const float *__restrict__ vol, const float *__restrict__ meas,
                                                    float *__restrict__ out, double *__restrict__ part) {
    unsigned tile_id;
    int q, row, col;
    bool ok;
    if (!cone_fp_pixel(g, nv, tile_id, q, row, col, ok)) return;   // padding workgroup
    double acc = 0.0;
    int view = 0;
    ConeWalk w;
    if (ok && (view = views[q], cone_ray_init(g, cs, view, row, col, w))) {
        bool live = true;
        // Whole groups first (the voxel's byte offset fits 32 bits); where the
        // walk ends, and for larger volumes, step by step below.
        const size_t bytes = (size_t)g.nx * g.ny * g.nz * sizeof(float);
        if (bytes < (size_t)1 << 32 && w.lam0 < w.stop && (unsigned)w.vx < (unsigned)g.nx &&
            (unsigned)w.vy < (unsigned)g.ny && (unsigned)w.vz < (unsigned)g.nz) {
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)vol, 0, (int)(uint32_t)bytes, 0x00020000);
            const int sy = 4, sx = g.ny * 4, sz = g.nx * g.ny * 4;
            ConeFast f{w.lam0, w.lx, w.ly, w.lz, (int)((unsigned)w.vz * (unsigned)sz + (unsigned)w.vx * (unsigned)sx + (unsigned)w.vy * 4u),
                       w.sgx > 0 ? g.nx - w.vx : w.vx + 1, w.sgy > 0 ? g.ny - w.vy : w.vy + 1,
                       w.sgz > 0 ? g.nz - w.vz : w.vz + 1};
            while (cone_fast(f, w, w.sgx * sx, w.sgy * sy, w.sgz * sz, rs, acc)) {
            }
            w.lam0 = f.lam0;
            w.lx = f.lx;
            w.ly = f.ly;
            w.lz = f.lz;
            w.vx = w.sgx > 0 ? g.nx - f.rx : f.rx - 1;
            w.vy = w.sgy > 0 ? g.ny - f.ry : f.ry - 1;
            w.vz = w.sgz > 0 ? g.nz - f.rz : f.rz - 1;
        }
        while (live) {
            unsigned id[kConeGroup];
            float ln[kConeGroup];
            bool lv[kConeGroup];
#pragma unroll
            for (int k = 0; k < kConeGroup; ++k) cone_step(g, w, live, id[k], ln[k]), lv[k] = live;
            float v[kConeGroup];
#pragma unroll
            for (int k = 0; k < kConeGroup; ++k) v[k] = vol[id[k]];
            // The product of two floats is exact in double, so the fused
            // multiply-add rounds once, as acc + (double)v * (double)len does.
#pragma unroll
            for (int k = 0; k < kConeGroup; ++k)
                acc = __builtin_fma((double)(lv[k] ? v[k] : 0.0f), (double)ln[k], acc);
        }
    }
    const size_t at = ((size_t)view * g.nrows + row) * g.ncols + col;
    if (MODE == CFP_WRITE) {
        if (ok) out[at] = (float)acc;
        return;
    }
    double sq = 0.0;
    if (MODE == CFP_RESID && ok) {
        const float r = (float)((double)meas[at] - acc);
        out[at] = r;
        sq = (double)r * (double)r;
    }
    if (MODE == CFP_SQ && ok) sq = acc * acc;
    const double tot = block_sum256(sq);
    if (threadIdx.x == 0) part[tile_id] = tot;
}

// Entry count of every ray (for the algorithmic-byte figure).
__global__ __launch_bounds__(kBlock) void k_cone_count(ConeDev g, const float *cs,
                                                       unsigned long long *total) {
    unsigned tile_id;
    int view, row, col;
    bool ok;
    unsigned long long n = 0;
    if (cone_fp_pixel(g, g.nviews, tile_id, view, row, col, ok) && ok) {
        ConeWalk w;
        if (cone_ray_init(g, cs, view, row, col, w)) {
            bool live = true;
            for (;;) {
                unsigned idx;
                float l;
                cone_step(g, w, live, idx, l);
                if (!live) break;
                ++n;
            }
        }
    }
    for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o);
    if ((threadIdx.x & 63) == 0 && n) atomicAdd(total, n);
}

// Per (view, column) tables of the back projector: 1 / (dx - sx), 1 / (dy - sy)
// (double) and |(dx - sx, dy - sy)|^2 (float) of the column's rays; per view
// the source point.
__global__ void k_cone_vctab(ConeDev g, const float *cs, double2 *inv, float *l2, float4 *src, float2 *pos) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)g.nviews * g.ncols) return;
    const int v = (int)(i / g.ncols), col = (int)(i % g.ncols);
    const float c = cs[2 * v], s = cs[2 * v + 1];
    float sx, sy, sz, dx, dy, dz;
    ray_points(g, c, s, 0, col, sx, sy, sz, dx, dy, dz);   // x and y do not depend on the row
    const double rx = (double)dx - (double)sx, ry = (double)dy - (double)sy;
    inv[i] = make_double2(1.0 / rx, 1.0 / ry);
    l2[i] = (float)(rx * rx + ry * ry);
    pos[i] = make_float2(sx, sy);
    if (col == 0) src[v] = make_float4(sx, sy, sz, 0.0f);
}

// Slab interval of the unit slab [a, a + 1] along one axis for the ray
// s + t r given ir = 1 / r (infinite when r = 0: all or nothing).
__device__ __forceinline__ void cone_slab_inv(double s, double ir, double a, double &lo, double &hi) {
    if (isinf(ir)) {
        const bool in = (s >= a) && (s < a + 1.0);
        lo = in ? lo : 1.0;
        hi = in ? hi : 0.0;
        return;
    }
    const double t0 = (a - s) * ir, t1 = (a + 1.0 - s) * ir;
    lo = fmax(lo, fmin(t0, t1));
    hi = fmin(hi, fmax(t0, t1));
}

// PAR: the parallel beam (rays at constant z, orthographic footprint; the
// rows' z in rowtab[2 r], the columns' start points in vpos).
// RLDS: the rows' 1 / w (nrows doubles) are copied to LDS (dynamic shared
// memory) first.
template <bool PAR, bool RLDS>
__device__ __forceinline__ void cone_bp_voxels(const ConeDev &g, const float *cs, const double *rowtab,
                                               const double2 *__restrict__ vinv, const float *__restrict__ vl2,
                                               const float4 *__restrict__ vsrc, const float2 *__restrict__ vpos,
                                               const int *views, int nv, const float *__restrict__ sino, double *carry,
                                               int first, int last, float *__restrict__ vol, int x, int y, int z0, int nk,
                                               const double *riw, double (*acc)[kBlock]) {
    // Per-lane sums of the kZc voxels in LDS (each lane owns its own slots,
    // so no barrier is needed); a register sums one (column, slice) first.
    // nk <= kZc: the slices from z0.
    // carry: the double sums of the earlier view chunks of a back projection
    // split into several launches (nullptr for a single launch).
    // vol nullptr: the sums stay in acc.
#pragma unroll
    for (int k = 0; k < kZc; ++k)
        acc[k][threadIdx.x] = (carry && !first && k < nk) ? carry[((size_t)(z0 + k) * g.nx + x) * g.ny + y] : 0.0;

    const float cxv = PAR ? g.halfsize : g.nx / 2.0f, cyv = PAR ? g.halfsize : g.ny / 2.0f;
    const float czv = PAR ? g.halfsize : g.nz / 2.0f;
    const float kpar = g.sample / g.pixel;       // parallel: panel pixels per voxel
    const float kcol = g.sdd / g.pixel;          // panel pixels per (voxel offset / voxel depth)
    const float sodv = g.sod / g.sample;         // source distance in voxels
    const float h5 = (float)g.halfdet - 0.5f;
    const float margin = 0.05f;                  // in pixels, covers the float rounding of the bounds

    for (int iv = 0; iv < nv; ++iv) {
        const int v = views[iv];
        const float c = cs[2 * v], s = cs[2 * v + 1];
        const float4 sp = vsrc[v];
        double sx = sp.x, sy = sp.y;
        const double sz = sp.z;
        // Corners of the column in the view's frame (u across the panel,
        // depth from the source): the panel column of a point is
        // u * kcol / depth + h5, the row of height zr is h5 - zr * kcol / depth.
        float cmin = 1e30f, cmax = -1e30f, imin = 1e30f, imax = -1e30f;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float px = (float)(x + (q & 1)) - cxv, py = (float)(y + (q >> 1)) - cyv;
            const float u = c * px + s * py;
            const float id = PAR ? 1.0f : 1.0f / (-s * px + c * py + sodv);
            const float cf = PAR ? u * kpar : u * kcol * id;
            cmin = fminf(cmin, cf);
            cmax = fmaxf(cmax, cf);
            imin = fminf(imin, id);
            imax = fmaxf(imax, id);
        }
        const int c0 = max(0, (int)ceilf(cmin + h5 - margin));
        const int c1 = min(g.ncols - 1, (int)floorf(cmax + h5 + margin));
        for (int col = c0; col <= c1; ++col) {
            const size_t vc = (size_t)v * g.ncols + col;
            const double2 ir = vinv[vc];
            if (PAR) {
                const float2 p0 = vpos[vc];
                sx = p0.x;
                sy = p0.y;
            }
            double lo = 0.0, hi = 1.0;
            cone_slab_inv(sx, ir.x, (double)x, lo, hi);
            cone_slab_inv(sy, ir.y, (double)y, lo, hi);
            if (!(hi > lo)) continue;
            // z-slab parameters relative to lo, so that the float
            // differences below keep full relative precision.
            const float span = (float)(hi - lo);
            const float lxy2 = vl2[vc];
            const double nlo = -lo;
            const float *scol = sino + ((size_t)v * g.nrows) * g.ncols + col;
            if (PAR) {
                // Rays at constant height: row r crosses slice z when
                // z <= z_r < z + 1, over the whole x / y chord.
                const float len = span * sqrtf(lxy2);
#pragma unroll 1
                for (int k = 0; k < nk; ++k) {
                    const int z = z0 + k;
                    const float za = (float)z - czv;
                    const int r0 = max(0, (int)ceilf(h5 - (za + 1.0f) * kpar - margin));
                    const int r1 = min(g.nrows - 1, (int)floorf(h5 - za * kpar + margin));
                    double part = 0.0;
                    for (int r = r0; r <= r1; ++r) {
                        const double zr = rowtab[2 * r];
                        if (zr >= (double)z && zr < (double)z + 1.0)
                            part += (double)scol[(size_t)r * g.ncols] * (double)len;
                    }
                    acc[k][threadIdx.x] += part;
                }
                continue;
            }
#pragma unroll 1
            for (int k = 0; k < nk; ++k) {
                const int z = z0 + k;
                // Rows whose rays can meet slice z inside the column.
                const float za = (float)z - czv, zb = za + 1.0f;
                const float wlo = fminf(za * imin, za * imax) * kcol;
                const float whi = fmaxf(zb * imin, zb * imax) * kcol;
                const int r0 = max(0, (int)ceilf(h5 - whi - margin));
                const int r1 = min(g.nrows - 1, (int)floorf(h5 - wlo + margin));
                const double dz0 = (double)z - sz, dz1 = dz0 + 1.0;
                double part = 0.0;
                for (int r = r0; r <= r1; ++r) {
                    const double iw = RLDS ? riw[r] : rowtab[2 * r + 1];
                    const float ta = (float)fma(dz0, iw, nlo), tb = (float)fma(dz1, iw, nlo);
                    const float a = fmaxf(0.0f, fminf(ta, tb)), e = fminf(span, fmaxf(ta, tb));
                    if (!(e > a)) continue;
                    // w = 1 / iw and the ray length to about one float ulp
                    // (hardware reciprocal and square root).
                    const float wf = __builtin_amdgcn_rcpf((float)iw);
                    const float L = __builtin_amdgcn_sqrtf(lxy2 + wf * wf);
                    const float len = (e - a) * L;
                    // float x float is exact in double: the fused form rounds once
                    part = __builtin_fma((double)scol[(size_t)r * g.ncols], (double)len, part);
                }
                acc[k][threadIdx.x] += part;
            }
        }
    }
    if (vol == nullptr) return;
    for (int k = 0; k < nk; ++k) {
        const size_t i = ((size_t)(z0 + k) * g.nx + x) * g.ny + y;
        if (carry && !last) carry[i] = acc[k][threadIdx.x];
        else vol[i] = (float)acc[k][threadIdx.x];
    }
}

template <bool PAR, bool RLDS>
__global__ __launch_bounds__(kBlock) void k_cone_bp(ConeDev g, const float *cs, const double *rowtab,
                                                    const double2 *__restrict__ vinv, const float *__restrict__ vl2,
                                                    const float4 *__restrict__ vsrc, const float2 *__restrict__ vpos,
                                                    const int *views, int nv, const float *__restrict__ sino,
                                                    double *carry, int first, int last, float *__restrict__ vol) {
    // Workgroup: 16 x 16 voxel columns, wave 8 x 8 of them; kZc slices.
    const int tx = (g.nx + 15) / 16, ty = (g.ny + 15) / 16;
    const unsigned b = xcd_block();
    const int per_z = tx * ty;
    const int zc = (int)(b / per_z), tile = (int)(b % per_z);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int x = (tile / ty) * 16 + (wv >> 1) * 8 + (lane >> 3);
    const int y = (tile % ty) * 16 + (wv & 1) * 8 + (lane & 7);
    const int z0 = zc * kZc;
    extern __shared__ double riw[];
    __shared__ double acc[kZc][kBlock];
    if (RLDS) {
        for (int r = threadIdx.x; r < g.nrows; r += kBlock) riw[r] = rowtab[2 * r + 1];
        __syncthreads();
    }
    if (x >= g.nx || y >= g.ny || z0 >= g.nz) return;
    cone_bp_voxels<PAR, RLDS>(g, cs, rowtab, vinv, vl2, vsrc, vpos, views, nv, sino, carry, first, last, vol, x, y, z0,
                              min(kZc, g.nz - z0), riw, acc);
}

// ---------------------------------------------------------------------------
// Back projection of the cone beam from panel patches.
//
// For a panel column and a voxel column (x, y) the in-plane chord [lo, hi] is
// the same for every row.  At chord parameter t row r is at height w_r t over
// the source (w falls with r), so of a plane dZ over the source the rows
// before some r1 are above it over the whole chord and those behind it are
// below; where (rows / 2) x (chord / source distance) is less than one row, as
// in every usual scanner, at most one row crosses it.  The sum of (row value x
// chord length above the plane) is then
//   B(dZ) = span PS[r1] + cut q_r1,
// with q = sinogram x ray length, PS its running sum over the rows and cut
// the part of the chord on which row r1 is above; a voxel between two planes
// gets B(lower) - B(upper).  A lane so keeps one double per plane of its kNk
// slices and spends some 14 instructions on a plane, where the form that
// clips every candidate ray (k_cone_bp) spends about 40 on a slice (3.3
// candidate rows, each with two double FMAs, a reciprocal, and a load).
//
// A workgroup is 16 x 16 voxel columns by kNk slices.  Per view it takes the
// panel patch its voxels can see (up to some 60 x 70 pixels), one lane per
// column and run of rows: each value is multiplied by its ray's length
// (the hardware's square root, one ulp) and the running sums go to LDS; the
// next view's values are loaded into registers meanwhile.  Summing order and
// everything else is fixed by the geometry.
//
// Bounded by LDS reads (24 bytes per lane, plane and column, 12 clocks of a
// CU per wave: 64% of the clocks) and vector issue (75%); two or three
// workgroups per CU, which the patches' LDS allows.  512^3, 720 views of 1024
// x 768: 508 ms ray by ray, 177 so; 256^3 x 360: 35.5 and 13.0; 128^3 x 180:
// 3.83 and 1.04; 64^3 x 100: 0.91 and 0.33.  Against 64-bit sums of the exact lengths
// both are off by 4.9e-7 of the largest voxel at 128^3.
constexpr int kConeRun = 24, kConeStep = 4;   // rows of a patch column per lane: at most, a multiple of
constexpr double kConeBits = 9.313225746154785e-10;   // 2^-30
constexpr double kConeUlp = 8.881784197001252e-16;    // 2^-50
constexpr int kConeMany = 8;                  // voxels that lost bits, from which on 0 counts as one
constexpr int kConeFew = 512;                 // voxels of a block done again one by one, at most
constexpr int kConeBatch = 5;                 // planes whose LDS reads are issued together (9: 4% slower at C4)
struct ConeView {
    int col0, ncol, r0, nr;       // the patch: panel columns, rows
    int run, cand;                // rows per lane; candidate columns of a voxel column
    float hw, icol;               // half width of a voxel column's shadow, 1 / ncol
};

// A value that all lanes hold, in scalar registers.
__device__ __forceinline__ double uniform(double x) {
    const uint64_t u = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u), hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// View (cos c, sin s) of the block of columns (x0, y0) .. and slices z0 .. z0 + nk.
__device__ __forceinline__ ConeView cone_view(const ConeDev &g, float c, float s, int x0, int y0, int z0, int nk) {
    const float kcol = g.sdd / g.pixel, sodv = g.sod / g.sample, h5 = (float)g.halfdet - 0.5f;
    const float za = (float)z0 - g.nz / 2.0f, zb = za + (float)nk;
    float lo = 1e30f, hi = -1e30f, ax = 0.f, ay = 0.f, rn = 0.f, rf = 1e30f;
    for (int q = 0; q < 4; ++q) {
        const float X = (float)min(g.nx, x0 + (q & 1) * 16) - g.nx / 2.0f, Y = (float)min(g.ny, y0 + (q >> 1) * 16) - g.ny / 2.0f;
        const float rD = 1.0f / (-s * X + c * Y + sodv), u = (c * X + s * Y) * kcol * rD;
        lo = fminf(lo, u);
        hi = fmaxf(hi, u);
        ax = fmaxf(ax, fabsf(c * kcol + s * u));
        ay = fmaxf(ay, fabsf(s * kcol - c * u));
        rn = fmaxf(rn, rD);
        rf = fminf(rf, rD);
    }
    ConeView w;
    // first order in the voxel (1 + 2 rn covers the rest), and the float rounding
    w.hw = 0.5f * (ax + ay) * rn * (1.0f + 2.0f * rn) + 0.01f;
    w.cand = (int)floorf(2.0f * w.hw) + 1;
    const float rlo = h5 - kcol * fmaxf(zb * rn, zb * rf), rhi = h5 - kcol * fminf(za * rn, za * rf);
    w.col0 = max(0, (int)floorf(lo + h5 - w.hw) - 1);
    w.ncol = max(0, min(g.ncols - 1, (int)ceilf(hi + h5 + w.hw) + 1) - w.col0 + 1);
    w.r0 = min(g.nrows, max(0, (int)floorf(rlo) - 2));
    w.nr = max(0, min(g.nrows - 1, (int)ceilf(rhi) + 2) - w.r0 + 1);
    if (w.ncol == 0 || w.nr == 0) w.ncol = w.nr = 0;
    const int seg = kBlock / max(w.ncol, 1);
    w.run = seg > 0 ? ((w.nr + seg - 1) / seg + kConeStep - 1) / kConeStep * kConeStep : INT_MAX;
    if (seg > 0 && w.nr > 0) w.nr = (w.nr + w.run - 1) / w.run * w.run;   // whole runs: rows behind the panel read as 0
    w.icol = 1.0f / (float)max(w.ncol, 1);
    return w;
}

// The largest patch of any block and view: m[0] columns, m[1] rows, m[2] rows
// per lane; m[3] the most rows a block sees over all views.
__global__ __launch_bounds__(kWave) void k_cone_patch(ConeDev g, const float *cs, int nk, int *m) {
    const int tx = (g.nx + 15) / 16, ty = (g.ny + 15) / 16;
    const int b = (int)blockIdx.x, zc = b / (tx * ty), tile = b % (tx * ty);
    int nc = 0, nr = 0, run = 0, r0 = INT_MAX, r1 = 0;
    for (int v = (int)threadIdx.x; v < g.nviews; v += kWave) {
        const ConeView w = cone_view(g, cs[2 * v], cs[2 * v + 1], tile / ty * 16, tile % ty * 16, zc * nk, nk);
        nc = max(nc, w.ncol);
        nr = max(nr, w.nr);
        run = max(run, w.run);
        if (w.nr > 0) {
            r0 = min(r0, w.r0);
            r1 = max(r1, w.r0 + w.nr);
        }
    }
    for (int o = kWave / 2; o > 0; o >>= 1) {
        nc = max(nc, __shfl_xor(nc, o));
        nr = max(nr, __shfl_xor(nr, o));
        run = max(run, __shfl_xor(run, o));
        r0 = min(r0, __shfl_xor(r0, o));
        r1 = max(r1, __shfl_xor(r1, o));
    }
    if (threadIdx.x == 0) {
        atomicMax(m, nc);
        atomicMax(m + 1, nr);
        atomicMax(m + 2, run);
        if (r1 > 0) atomicMax(m + 3, r1 - r0);
    }
}

// LDS of a workgroup: the running sums (column major; one entry before the
// first row and one behind the last), 1 / w and w^2 of the rows its views
// see, 1 / (d - s) per column, the lanes' totals and absolute totals, the
// columns' absolute totals, the views.
constexpr int kConeViews = 36;
__host__ __device__ __forceinline__ int cone_patch_stride(int rows) { return (rows + 3) | 1; }
__host__ __device__ __forceinline__ size_t cone_patch_lds(int cols, int rows, int span) {
    const size_t sums = ((size_t)cols * cone_patch_stride(rows) + 1) & ~(size_t)1;
    const size_t need = 8 * (sums + 2 * (size_t)cols + kBlock + span + 2) + 4 * (size_t)(span + 2 + kBlock + cols) +
                        kConeViews * sizeof(ConeView);
    const size_t again = kZc * kBlock * 8 + kConeFew * 4;   // (the sums of the ray by ray form, the voxels it does)
    return need > again ? need : again;
}

struct ConePatchArgs {
    ConeDev g;
    const float *cs;
    const double *rowtab;
    const double2 *vinv;
    const float *vl2;
    const float4 *vsrc;
    const int *views;
    const float *sino;
    float *vol;
    int nv, cols, rows, span_rows;
};

// The planes' sums A of a block's voxel columns, what they may have held
// (size); true if a sum of this lane was not finite.
// CROSS: the source's height lies within the block's slices.
template <int NK, bool CROSS>
__device__ __forceinline__ bool cone_bp_block(const ConePatchArgs &t, int x0, int y0, int z0, double (&A)[NK + 1],
                                              float &size) {
    const ConeDev &g = t.g;
    const float *cs = t.cs;
    const double *rowtab = t.rowtab;
    const double2 *__restrict__ vinv = t.vinv;
    const float *__restrict__ vl2 = t.vl2;
    const float4 *__restrict__ vsrc = t.vsrc;
    const float *__restrict__ sino = t.sino;
    const int *views = t.views;
    const int nv = t.nv, cols = t.cols, rows = t.rows, span_rows = t.span_rows;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int x = x0 + (wv >> 1) * 8 + (lane >> 3), y = y0 + (wv & 1) * 8 + (lane & 7);
    extern __shared__ double smem[];
    const int stride = cone_patch_stride(rows);
    double *PS = smem;
    double2 *irs = (double2 *)(PS + ((cols * stride + 1) & ~1));
    double *tots = (double *)(irs + cols), *iws = tots + kBlock;
    ConeView *info = (ConeView *)(iws + span_rows + 2);
    float *w2s = (float *)(info + kConeViews), *atots = w2s + span_rows + 2, *acols = atots + kBlock;
    __shared__ int sh_r0, sh_r1;
    const float kcol = g.sdd / g.pixel, kz = g.sample / g.pixel, sodv = g.sod / g.sample, h5 = (float)g.halfdet - 0.5f;
    const float px = (float)x + 0.5f - g.nx / 2.0f, py = (float)y + 0.5f - g.ny / 2.0f;
    const double sz = (double)vsrc[views[0]].z, xd = x, yd = y;   // the source's height is every view's

    // the planes' heights: all over the source (or at it), all under, or both
    const float dz0 = (float)z0 - g.nz / 2.0f;
    const bool over = dz0 >= 0.0f;
    const int kover = __builtin_amdgcn_readfirstlane((int)floorf(-dz0) + 1);   // the first plane over the source
    double mdZ[NK + 1];
#pragma unroll
    for (int k = 0; k <= NK; ++k) {
        A[k] = 0.0;
        mdZ[k] = uniform(-fabs((double)(z0 + k) - sz));
    }
    float raw[kConeRun], l2 = 0.f;
    double2 ir = make_double2(0.0, 0.0);
    const int rowb = g.ncols * 4;
    // this lane's part of view iv's patch, into registers (rows behind its
    // run are other lanes', rows behind the panel read as 0)
    int v0 = 0;
    bool bad = false;   // a sum of this lane was not finite
    size = 0.0f;        // the columns' absolute sums, by the chords
    auto load = [&](int iv) {
        const ConeView w = info[iv];
        const int seg = (int)(((float)tid + 0.5f) * w.icol), col = tid - seg * w.ncol;   // tid / ncol
        const size_t panel = (size_t)g.nrows * g.ncols;
        const int v = __builtin_amdgcn_readfirstlane(views[v0 + iv]);
        const auto rs = __builtin_amdgcn_make_buffer_rsrc((void *)(sino + v * panel), 0, (int)(panel * 4), 0x00020000);
        const int run = __builtin_amdgcn_readfirstlane(w.run);
        const int at = ((w.r0 + seg * run) * g.ncols + w.col0 + col) * 4;
        const bool any = w.ncol > 0 && seg * run < w.nr;
        if (any) {
            l2 = vl2[(size_t)v * g.ncols + w.col0 + col];
#pragma unroll
            for (int i = 0; i < kConeRun; i += kConeStep)
                if (i < run)
#pragma unroll
                    for (int h = i; h < i + kConeStep; ++h)
                        raw[h] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, at + h * rowb, 0, 0));
        }
        if (tid < w.ncol) ir = vinv[(size_t)v * g.ncols + w.col0 + tid];
    };
    for (; v0 < nv; v0 += kConeViews) {
        const int ng = min(kConeViews, nv - v0);
        if (tid == 0) {
            sh_r0 = g.nrows;
            sh_r1 = 0;
        }
        __syncthreads();
        if (tid < ng) {
            const int v = views[v0 + tid];
            const ConeView w = cone_view(g, cs[2 * v], cs[2 * v + 1], x0, y0, z0, NK);
            info[tid] = w;
            if (w.nr > 0) {
                atomicMin(&sh_r0, w.r0);
                atomicMax(&sh_r1, w.r0 + w.nr);
            }
        }
        __syncthreads();
        const int rbase = sh_r0, rspan = sh_r1 - sh_r0;
        for (int i = tid; i < rspan + 2; i += kBlock) {   // entry i: row rbase + i - 1
            const int r = min(max(rbase + i - 1, 0), g.nrows - 1);
            const float wr = (float)rowtab[2 * r];
            iws[i] = rowtab[2 * r + 1];
            w2s[i] = wr * wr;
        }
        load(0);
        __syncthreads();
        for (int iv = 0; iv < ng; ++iv) {
            ConeView w = info[iv];
            w.ncol = __builtin_amdgcn_readfirstlane(w.ncol);   // (0: the view does not see the block)
            w.cand = __builtin_amdgcn_readfirstlane(w.cand);
            w.nr = __builtin_amdgcn_readfirstlane(w.nr);
            w.run = __builtin_amdgcn_readfirstlane(w.run);
            w.r0 = __builtin_amdgcn_readfirstlane(w.r0);
            w.col0 = __builtin_amdgcn_readfirstlane(w.col0);
            const int v = __builtin_amdgcn_readfirstlane(views[v0 + iv]);
            // q = sinogram x ray length, the runs' totals
            const int seg = (int)(((float)tid + 0.5f) * w.icol), col = tid - seg * w.ncol;
            const int r = seg * w.run;
            const bool any = r < w.nr;
            double sum = 0.0;
            float mag = 0.0f;
            if (any) {
                const float *w2 = w2s + (w.r0 - rbase + r + 1);
#pragma unroll
                for (int i = 0; i < kConeRun; i += kConeStep)
                    if (i < w.run)
#pragma unroll
                        for (int h = i; h < i + kConeStep; ++h) {
                            raw[h] *= __builtin_amdgcn_sqrtf(w2[h] + l2);
                            sum += (double)raw[h];
                            mag += fabsf(raw[h]);
                            asm volatile("" : "+v"(raw[h]));   // (converted again below: not 24 doubles kept)
                        }
            }
            bad |= !(fabs(sum) < INFINITY);
            tots[tid] = sum;
            atots[tid] = mag;
            // a ray along an axis: all or nothing on the other, by a huge finite
            // inverse (0 x infinity has no value)
            if (tid < w.ncol) irs[tid] = make_double2(fmin(fmax(ir.x, -1e300), 1e300), fmin(fmax(ir.y, -1e300), 1e300));
            __syncthreads();
            if (any) {
                double run = 0.0;
                for (int i = 0; i < seg; ++i) {
                    run += tots[i * w.ncol + col];
                    mag += atots[i * w.ncol + col];
                }
                double *P = PS + col * stride + 2 + r;   // P[i]: the rows up to r + i
                if (seg == 0) P[-2] = P[-1] = 0.0;
#pragma unroll
                for (int i = 0; i < kConeRun; i += kConeStep)
                    if (i < w.run)
#pragma unroll
                        for (int h = i; h < i + kConeStep; ++h) P[h] = run += (double)raw[h];
                if (r + w.run == w.nr) {
                    P[w.run] = run;
                    acols[col] = fminf(mag, FLT_MAX);   // (times 0: 0)
                }
            }
            __syncthreads();
            if (iv + 1 < ng) load(iv + 1);

            const float c = cs[2 * v], sn = cs[2 * v + 1];
            const float4 sp = vsrc[v];
            const float rD = __builtin_amdgcn_rcpf(-sn * px + c * py + sodv);
            const int c0 = (int)ceilf((c * px + sn * py) * kcol * rD + h5 - w.hw) - w.col0;
            const double *iw0 = iws + (w.r0 - rbase);   // entry i: row r0 + i - 1
            const float h5r = h5 - (float)w.r0;
            for (int j = 0; j < (w.ncol > 0 ? w.cand : 0); ++j) {
                const bool in = (unsigned)(c0 + j) < (unsigned)w.ncol;
                const int lc = in ? c0 + j : 0;
                const double2 irc = irs[lc];
                const double ax = (xd - (double)sp.x) * irc.x, ay = (yd - (double)sp.y) * irc.y;
                const double bx = ax + irc.x, by = ay + irc.y;
                const double lo = fmax(fmax(fmin(ax, bx), fmin(ay, by)), 0.0), hi = fmin(fmin(fmax(ax, bx), fmax(ay, by)), 1.0);
                const float span = (in && hi > lo) ? (float)(hi - lo) : 0.0f;
                if (!__any(span > 0.0f)) continue;
                const float inv = span > 0.0f ? (__builtin_amdgcn_rcpf((float)lo) + __builtin_amdgcn_rcpf((float)hi)) * (0.5f * kz) : 0.0f;
                size = __builtin_fmaf(span, acols[lc], size);
                const double spand = (double)span, nlo = -lo, base = over ? hi : nlo;
                const double *P = PS + lc * stride;
                const float last = (float)(w.nr + 1);
                // the row nearest the plane's at the middle of the chord; planes
                // at the source's height between two rows take the one on their
                // block's side of it
                float pos = __builtin_fmaf(-dz0, inv, h5r + (over ? 1.495f : 1.505f));
#pragma unroll
                for (int k0 = 0; k0 <= NK; k0 += kConeBatch) {   // the planes' LDS reads, a few together
                    double a[kConeBatch], b[kConeBatch], iw[kConeBatch];
#pragma unroll
                    for (int k = k0; k < k0 + kConeBatch && k <= NK; ++k) {
                        const int i = (int)__builtin_amdgcn_fmed3f(pos, 0.0f, last);
                        pos -= inv;
                        a[k - k0] = P[i];
                        b[k - k0] = P[i + 1];
                        iw[k - k0] = iw0[i];
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int k = k0; k < k0 + kConeBatch && k <= NK; ++k) {
                        double from = base;
                        if constexpr (CROSS) {
                            int kz = kover;
                            asm volatile("" : "+v"(kz));   // (compared here: no mask per plane kept in registers)
                            from = k >= kz ? hi : nlo;
                        }
                        const float cut = __builtin_amdgcn_fmed3f((float)__builtin_fma(mdZ[k], iw[k - k0], from), 0.0f, span);
                        // (a row entirely above counts like the rows before it, so that
                        // two planes with no row between them sum alike, to the bit)
                        const double from0 = cut < span ? a[k - k0] : b[k - k0];
                        A[k] = __builtin_fma(spand, from0, A[k]);
                        A[k] = __builtin_fma((double)cut, b[k - k0] - from0, A[k]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            __syncthreads();   // the patch is written again
        }
    }
    return bad;
}

template <int NK>
__global__ __launch_bounds__(kBlock) void k_cone_bp_patch(ConePatchArgs args) {
    const unsigned blk = xcd_block();
    const int ty = (args.g.ny + 15) / 16, txy = (args.g.nx + 15) / 16 * ty;
    const int z0 = (int)(blk / txy) * NK, tile = (int)(blk % txy);
    if (z0 >= args.g.nz) return;
    const int x0 = (tile / ty) * 16, y0 = (tile % ty) * 16;
    double A[NK + 1];
    float size;
    bool bad = 2 * z0 < args.g.nz && 2 * (z0 + NK) > args.g.nz ? cone_bp_block<NK, true>(args, x0, y0, z0, A, size)
                                                               : cone_bp_block<NK, false>(args, x0, y0, z0, A, size);
    // The arguments are read again from here: kept over the views' loop they
    // had scalar registers going to and fro in it (512^3 x 720: 186 ms, now
    // 177; 256^3 x 360: 13.6 and 13.0; 128^3 x 180: 1.055 and 1.038).
    uint64_t at = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(at));
    const ConePatchArgs t = *(const ConePatchArgs *)(const __attribute__((address_space(4))) ConePatchArgs *)at;
    const ConeDev &g = t.g;
    const float *cs = t.cs;
    const double *rowtab = t.rowtab;
    const int *views = t.views;
    const float *sino = t.sino;
    float *vol = t.vol;
    const int nv = t.nv, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int x = x0 + (wv >> 1) * 8 + (lane >> 3), y = y0 + (wv & 1) * 8 + (lane & 7);
    extern __shared__ double smem[];
    __shared__ int sh_again, sh_few;
    __shared__ unsigned sh_least;
    // A voxel is the difference of two planes' sums, which keep some 47 bits of
    // `size`: one that is below 2^-30 of it is done again ray by ray, for a few
    // values far above its own may have been in the sums.  Positive data has it
    // at 2^-6, so there is none; noise about 0 cancels so far in one voxel of
    // some thousands, and where a few values do lie far above the others, the
    // voxels off their rays have it.  0 is exact (no value lies between the two
    // planes) unless the smaller values were lost whole: where the smallest one,
    // over a voxel's width, is below 2^-50 of `size`, or several voxels of the
    // block are small without being 0.  (Looked up here, in blocks that hold
    // zeros, and not kept in the views' loop, which every call pays for.)
    if (tid == 0) {
        sh_again = sh_few = 0;
        sh_least = UINT_MAX;
    }
    __syncthreads();
    const double small = (double)size * kConeBits;
    int few = 0;
    bool none = false;
#pragma unroll
    for (int k = 0; k < NK; ++k) {
        const double d = fabs(A[k] - A[k + 1]);
        const bool lower = x < g.nx && y < g.ny && z0 + k < g.nz && d < small;
        few += lower && d != 0.0;
        none |= lower && d == 0.0;
    }
    if (few > 0) atomicAdd(&sh_few, few);
    none = __syncthreads_or(none);
    bool lost = sh_few >= kConeMany;
    if (none && !lost) {
        // The smallest non-zero value of the patches: a wave a view, eight rows'
        // loads together (the last row's again behind it; one at a time, 48^3 x
        // 120 took 445 us, so 407, without the look 392).
        unsigned least = UINT_MAX;   // its bits 2 x - 1 (0: the largest)
        for (int iv = wv; iv < nv; iv += kBlock / kWave) {
            const int v = views[iv];
            const ConeView w = cone_view(g, cs[2 * v], cs[2 * v + 1], x0, y0, z0, NK);
            const int nr = __builtin_amdgcn_readfirstlane(min(w.nr, g.nrows - w.r0));
            const float *from = sino + ((size_t)v * g.nrows + w.r0) * g.ncols + w.col0;
            for (int col = lane; col < w.ncol; col += kWave)
                for (int r = 0; r < nr; r += 8) {
                    float q[8];
#pragma unroll
                    for (int h = 0; h < 8; ++h) q[h] = from[(size_t)min(r + h, nr - 1) * g.ncols + col];
#pragma unroll
                    for (int h = 0; h < 8; ++h) least = min(least, (__builtin_bit_cast(unsigned, q[h]) << 1) - 1u);
                }
        }
        atomicMin(&sh_least, least);
        __syncthreads();
        lost = (double)__builtin_bit_cast(float, (sh_least + 1u) >> 1) < (double)size * kConeUlp;
    }
    int *list = (int *)(smem + kZc * kBlock);
#pragma unroll
    for (int k = 0; k < NK; ++k)
        if (x < g.nx && y < g.ny && z0 + k < g.nz) {
            const double d = A[k] - A[k + 1];
            if (fabs(d) < small && (d != 0.0 || lost)) {
                const int n = atomicAdd(&sh_again, 1);
                if (n < kConeFew) list[n] = k * kBlock + tid;
            } else {
                vol[((size_t)(z0 + k) * g.nx + x) * g.ny + y] = (float)d;
            }
        }
    bad = __syncthreads_or(bad);
    const int again = sh_again;
    double(*acc)[kBlock] = (double(*)[kBlock])smem;
    if (bad || again > kConeFew) {
        // The whole block (a value that is not finite reached every row behind
        // it through the running sums).
        const int zend = min(z0 + NK, g.nz);
        for (int z = z0; z < zend; z += kZc) {
            if (x >= g.nx || y >= g.ny) break;
            cone_bp_voxels<false, false>(g, cs, rowtab, t.vinv, t.vl2, t.vsrc, nullptr, views, nv, sino, nullptr, 1, 1, vol, x, y,
                                         z, min(kZc, zend - z), nullptr, acc);
        }
        return;
    }
    // A wave a voxel, its lanes some of the views each: one of noise costs a
    // block some microseconds, where the whole block would take three times as
    // long as all before.
    for (int i = wv; i < again; i += kBlock / kWave) {
        const int id = __builtin_amdgcn_readfirstlane(list[i]), w = id % kBlock / kWave, l = id % kWave;
        const int vx = x0 + (w >> 1) * 8 + (l >> 3), vy = y0 + (w & 1) * 8 + (l & 7), vz = z0 + id / kBlock;
        const int from = (int)((int64_t)lane * nv / kWave), to = (int)((int64_t)(lane + 1) * nv / kWave);
        cone_bp_voxels<false, false>(g, cs, rowtab, t.vinv, t.vl2, t.vsrc, nullptr, views + from, to - from, sino, nullptr, 1, 1,
                                     nullptr, vx, vy, vz, 1, nullptr, acc);
        double sum = acc[0][tid];
        for (int o = kWave / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
        if (lane == 0) vol[((size_t)vz * g.nx + vx) * g.ny + vy] = (float)sum;
    }
}

unsigned grid8(size_t blocks) { return (unsigned)((blocks + 7) / 8 * 8); }

}  // namespace

void validate_cone(const mi_cone_geometry &g) {
    MI_REQUIRE(g.nx > 0 && g.ny > 0 && g.nz > 0 && g.n_views > 0 && g.n_rows > 0 && g.n_cols > 0, MI_E_ARG,
               "cone geometry sizes must be positive");
    MI_REQUIRE((int64_t)g.nx * g.ny * g.nz < ((int64_t)1 << 31), MI_E_LIMIT, "volume beyond 2^31 voxels");
    // The forward walk forms a voxel's offset as ((z nx + x) ny) + y with
    // 24-bit multiplies: z nx + x and ny must stay below 2^24.
    MI_REQUIRE((int64_t)g.nz * g.nx <= ((int64_t)1 << 24) && g.ny < (1 << 24), MI_E_LIMIT,
               "cone volume needs nz * nx <= 2^24 and ny < 2^24");
    MI_REQUIRE((int64_t)g.n_views * g.n_rows * g.n_cols < ((int64_t)1 << 40), MI_E_LIMIT, "sinogram too large");
    MI_REQUIRE(std::isfinite(g.sample_mm) && std::isfinite(g.pixel_mm) && g.sample_mm > 0 && g.pixel_mm > 0,
               MI_E_ARG, "sample_mm and pixel_mm must be positive");
    MI_REQUIRE(std::isfinite(g.sdd_mm) && g.sod_mm > 0 && g.sdd_mm > g.sod_mm, MI_E_ARG, "need sdd > sod > 0");
    MI_REQUIRE(g.beam == MI_CONE_BEAM || g.beam == MI_CONE_PARALLEL, MI_E_ARG, "unknown cone-geometry beam");
    // The source circle must lie outside the volume (the back projector's
    // corner projection assumes every voxel is in front of the source).
    const double half = 0.5 * g.sample_mm * std::sqrt((double)g.nx * g.nx + (double)g.ny * g.ny);
    MI_REQUIRE(g.beam == MI_CONE_PARALLEL || g.sod_mm > half, MI_E_ARG, "the source orbit must lie outside the volume");
}

ConeTables &cone_tables(mi_context *ctx, const mi_cone_geometry &g) {
    validate_cone(g);
    if (ctx->cone && std::memcmp(&ctx->cone->g, &g, sizeof(g)) == 0) return *ctx->cone;
    auto t = std::make_shared<ConeTables>();
    t->g = g;
    t->d = ConeDev{g.nx, g.ny, g.nz, g.n_views, g.n_rows, g.n_cols, g.n_rows / 2,
                   g.sample_mm, g.pixel_mm, g.sod_mm, g.sdd_mm, g.beam == MI_CONE_PARALLEL ? 1 : 0,
                   (float)(g.nx / 2.0)};
    std::vector<float> cs(2 * (size_t)g.n_views);
    for (int a = 0; a < g.n_views; ++a) {
        // theta = (float)alpha / NPROJ * 2 * PI, industry3d/src/tracing.cpp:58.
        float th = (float)a / (float)g.n_views;
        th = th * 2.0f;
        th = (float)((double)th * 3.1415926535897932385);
        cs[2 * a] = cosf(th);
        cs[2 * a + 1] = sinf(th);
    }
    const float sz = (float)((double)(0.0f / g.sample_mm) + g.nz / 2.0);
    std::vector<double> rows(2 * (size_t)g.n_rows);
    for (int r = 0; r < g.n_rows; ++r) {
        if (t->d.parallel) {
            // the row's constant z: (HALFDET - r - 0.5) PIXELSIZE / SAMPLESIZE + HALFSIZE in float
            float Z = (float)((double)(t->d.halfdet - r) - 0.5);
            Z *= g.pixel_mm;
            rows[2 * r] = (double)(Z / g.sample_mm + t->d.halfsize);
            rows[2 * r + 1] = 0.0;
            continue;
        }
        const double w = (double)cone_det_z(t->d, r) - (double)sz;
        MI_REQUIRE(w != 0.0, MI_E_ARG, "a detector row lies in the plane of the source orbit");
        rows[2 * r] = w;
        rows[2 * r + 1] = 1.0 / w;
    }
    std::vector<int> all(g.n_views);
    for (int a = 0; a < g.n_views; ++a) all[a] = a;
    t->all.alloc(all.size());
    MI_HIP(hipMemcpyAsync(t->all.p, all.data(), all.size() * sizeof(int), hipMemcpyHostToDevice, ctx->stream));
    t->cs.alloc(cs.size());
    t->rows.alloc(rows.size());
    MI_HIP(hipMemcpyAsync(t->cs.p, cs.data(), cs.size() * sizeof(float), hipMemcpyHostToDevice, ctx->stream));
    MI_HIP(hipMemcpyAsync(t->rows.p, rows.data(), rows.size() * sizeof(double), hipMemcpyHostToDevice,
                          ctx->stream));
    const size_t nvc = (size_t)g.n_views * g.n_cols;
    t->vinv.alloc(nvc);
    t->vl2.alloc(nvc);
    t->vsrc.alloc(g.n_views);
    t->vpos.alloc(nvc);
    hipLaunchKernelGGL(k_cone_vctab, dim3((unsigned)((nvc + kBlock - 1) / kBlock)), dim3(kBlock), 0, ctx->stream, t->d,
                       t->cs.p, t->vinv.p, t->vl2.p, t->vsrc.p, t->vpos.p);
    MI_HIP(hipGetLastError());
    if (!t->d.parallel) {
        // At most one row may cross a plane within a voxel column's chord
        // (sqrt 2 voxels at the least distance from the source).
        const double near = g.sod_mm / (double)g.sample_mm - 0.5 * std::hypot((double)g.nx, (double)g.ny);
        const double far = std::max(t->d.halfdet, g.n_rows - t->d.halfdet) + 1.0;
        if (near > 1.0 && far * std::sqrt(2.0) / near + 0.05 < 1.0) {
            DevBuf<int> m(8);
            int h[8];
            MI_HIP(hipMemsetAsync(m.p, 0, m.bytes(), ctx->stream));
            for (int i = 0; i < 2; ++i) {
                const size_t nb = (size_t)((g.nx + 15) / 16) * ((g.ny + 15) / 16) * ((g.nz + kConeNk[i] - 1) / kConeNk[i]);
                hipLaunchKernelGGL(k_cone_patch, dim3((unsigned)nb), dim3(kWave), 0, ctx->stream, t->d, t->cs.p, kConeNk[i],
                                   m.p + 4 * i);
                MI_HIP(hipGetLastError());
            }
            MI_HIP(hipMemcpyAsync(h, m.p, sizeof(h), hipMemcpyDeviceToHost, ctx->stream));
            MI_HIP(hipStreamSynchronize(ctx->stream));
            for (int i = 0; i < 2; ++i)
                if (h[4 * i] > 0 && h[4 * i + 2] <= kConeRun && ((size_t)g.n_rows + kConeRun) * g.n_cols < (size_t)1 << 29 &&
                    cone_patch_lds(h[4 * i], h[4 * i + 1], h[4 * i + 3]) <= ((size_t)63 << 10)) {
                    t->patch_cols[i] = h[4 * i];
                    t->patch_rows[i] = h[4 * i + 1];
                    t->patch_span[i] = h[4 * i + 3];
                }
        }
    }
    MI_HIP(hipStreamSynchronize(ctx->stream));
    ctx->cone = t;
    return *t;
}

void cone_trace(hipStream_t st, const ConeTables &t, int view, int row, int col, int64_t *ind, float *len, int cap,
                int *numb) {
    hipLaunchKernelGGL(k_cone_trace, dim3(1), dim3(64), 0, st, t.d, t.cs.p, view, row, col, ind, len, cap, numb);
    MI_HIP(hipGetLastError());
}

static size_t cone_fp_blocks(const ConeDev &d, int nv) {
    return (size_t)((d.ncols + kConeTile - 1) / kConeTile) * ((d.nrows + kConeTile - 1) / kConeTile) * nv;
}

size_t cone_fp_views(hipStream_t st, const ConeTables &t, const int *views, int nv, int mode, const float *vol,
                     const float *meas, float *out, double *part) {
    const size_t nb = cone_fp_blocks(t.d, nv);
    const dim3 grid(grid8(nb)), block(kBlock);
    switch (mode) {
        case CFP_WRITE:
            launch(k_cone_fp<CFP_WRITE>, grid, block, 0u, st, t.d, t.cs.p, views, nv, vol, meas, out, part);
            break;
        case CFP_RESID:
            launch(k_cone_fp<CFP_RESID>, grid, block, 0u, st, t.d, t.cs.p, views, nv, vol, meas, out, part);
            break;
        default:
            launch(k_cone_fp<CFP_SQ>, grid, block, 0u, st, t.d, t.cs.p, views, nv, vol, meas, out, part);
    }
    MI_HIP(hipGetLastError());
    return nb;
}

// The allocation-free back projection's carry (mi_cone_backproject_dev_noalloc):
// one copy per device, for the life of the process.
constexpr size_t kScratchCarry = (size_t)8 << 20;   // doubles (64 MiB): volumes up to 8 Mi voxels
static __device__ __align__(256) double scratch[kScratchCarry];

namespace {
constexpr int kMaxDevices = 64;
std::once_flag g_scratch_once[kMaxDevices];
double *g_scratch_ptr[kMaxDevices];
hipError_t g_scratch_err[kMaxDevices];
}  // namespace

void cone_scratch_init(int device) {
    MI_REQUIRE(device >= 0 && device < kMaxDevices, MI_E_LIMIT, "device index beyond the scratch table");
    // The array's name is a host-side stand-in: its device address (one per
    // device) comes from the runtime, with that device current.
    std::call_once(g_scratch_once[device], [device] {
        g_scratch_err[device] = hipGetSymbolAddress((void **)&g_scratch_ptr[device], HIP_SYMBOL(scratch));
    });
    MI_HIP(g_scratch_err[device]);
}

int64_t cone_scratch_voxels() { return (int64_t)kScratchCarry; }

void cone_bp_views(hipStream_t st, const ConeTables &t, const int *views, int nv, const float *sino, float *vol,
                   int device_scratch) {
    const int chunks = (nv + kBpViewChunk - 1) / kBpViewChunk;
    const size_t nvox = (size_t)t.d.nx * t.d.ny * t.d.nz;
    if (chunks > 1 && device_scratch >= 0) {
        MI_REQUIRE(nvox <= kScratchCarry, MI_E_LIMIT,
                   "volume of " + std::to_string(nvox) + " voxels exceeds the allocation-free back projection's " +
                       std::to_string(kScratchCarry) + "-voxel scratch");
        MI_REQUIRE(g_scratch_ptr[device_scratch], MI_E_STATE, "device scratch not initialised");
    }
    auto grid = [&](int nk) { return (size_t)((t.d.nx + 15) / 16) * ((t.d.ny + 15) / 16) * ((t.d.nz + nk - 1) / nk); };
    // The patch form where the geometry has it, all views in one launch (the
    // sums stay in registers: 5 launches of 36 views and their carry volume
    // were 1.31 ms at 128^3 x 180 views, one is 1.14).  16 slices a workgroup,
    // 8 where that leaves fewer workgroups than two per CU or 16 slices' patch
    // does not fit: 128^3 x 180 views (512 workgroups of 16) 0.94 ms with 16
    // and 1.22 with 8, 512^3 x 720 152 and 214, 64^3 x 100 (64 workgroups of
    // 16) 0.40 and 0.30 (all before the voxels were tested for lost bits: 1.04,
    // 177 and 0.33 with it).
    int patch = t.patch_cols[0] > 0 ? 0 : -1;
    if (t.patch_cols[1] > 0 && (patch < 0 || grid(kConeNk[0]) < 512)) patch = 1;
    if (patch >= 0) {
        const int pc = t.patch_cols[patch], pr = t.patch_rows[patch], ps = t.patch_span[patch];
        const ConePatchArgs args{t.d,      t.cs.p, t.rows.p, t.vinv.p, t.vl2.p, t.vsrc.p,
                                 views,    sino,   vol,      nv,       pc,      pr,       ps};
        launch(patch == 0 ? k_cone_bp_patch<kConeNk[0]> : k_cone_bp_patch<kConeNk[1]>, dim3(grid8(grid(kConeNk[patch]))),
               dim3(kBlock), (uint32_t)cone_patch_lds(pc, pr, ps), st, args);
        MI_HIP(hipGetLastError());
        return;
    }
    const size_t blocks = grid(kZc);
    // Views in chunks whose sinogram rows stay cached while every workgroup
    // sweeps them; double sums carried between chunks (a buffer allocated
    // here, or the device's fixed scratch array).
    DevBuf<double> own(chunks > 1 && device_scratch < 0 ? nvox : 0);
    double *carry = chunks > 1 && device_scratch >= 0 ? g_scratch_ptr[device_scratch] : own.p;
    for (int c = 0; c < chunks; ++c) {
        const int v0 = c * kBpViewChunk, n = std::min(kBpViewChunk, nv - v0);
        if (t.d.parallel)
            launch(k_cone_bp<true, false>, dim3(grid8(blocks)), dim3(kBlock), 0u, st, t.d, t.cs.p,
                               t.rows.p, t.vinv.p, t.vl2.p, t.vsrc.p, t.vpos.p, views + v0, n, sino, carry, c == 0,
                               c == chunks - 1, vol);
        else if (t.d.nrows <= kBpRowLds)
            launch(k_cone_bp<false, true>, dim3(grid8(blocks)), dim3(kBlock),
                               (uint32_t)(t.d.nrows * sizeof(double)), st, t.d, t.cs.p, t.rows.p, t.vinv.p, t.vl2.p,
                               t.vsrc.p, t.vpos.p, views + v0, n, sino, carry, c == 0, c == chunks - 1, vol);
        else
            launch(k_cone_bp<false, false>, dim3(grid8(blocks)), dim3(kBlock), 0u, st, t.d, t.cs.p,
                               t.rows.p, t.vinv.p, t.vl2.p, t.vsrc.p, t.vpos.p, views + v0, n, sino, carry, c == 0,
                               c == chunks - 1, vol);
        MI_HIP(hipGetLastError());
    }
    if (own.p) MI_HIP(hipStreamSynchronize(st));   // before the carry buffer is freed
}

void cone_forward(hipStream_t st, const ConeTables &t, const float *vol, float *sino) {
    cone_fp_views(st, t, t.all.p, t.d.nviews, CFP_WRITE, vol, nullptr, sino, nullptr);
}

void cone_backproject(hipStream_t st, const ConeTables &t, const float *sino, float *vol) {
    cone_bp_views(st, t, t.all.p, t.d.nviews, sino, vol);
}

double cone_fp_bytes(const ConeTables &t) {
    const double rays = (double)t.d.nviews * t.d.nrows * t.d.ncols;
    const double vox = (double)t.d.nx * t.d.ny * t.d.nz;
    return (double)t.nnz * 8.0 + rays * 4.0 + vox * 4.0;
}

double cone_bp_bytes(const ConeTables &t) { return cone_fp_bytes(t); }

int64_t cone_nnz(hipStream_t st, ConeTables &t) {
    if (t.nnz >= 0) return t.nnz;
    DevBuf<unsigned long long> n(1);
    MI_HIP(hipMemsetAsync(n.p, 0, sizeof(unsigned long long), st));
    hipLaunchKernelGGL(k_cone_count, dim3(grid8(cone_fp_blocks(t.d, t.d.nviews))), dim3(kBlock), 0, st, t.d, t.cs.p,
                       n.p);
    MI_HIP(hipGetLastError());
    unsigned long long h = 0;
    MI_HIP(hipMemcpyAsync(&h, n.p, sizeof(h), hipMemcpyDeviceToHost, st));
    MI_HIP(hipStreamSynchronize(st));
    t.nnz = (int64_t)h;
    return t.nnz;
}

}  // namespace mi
