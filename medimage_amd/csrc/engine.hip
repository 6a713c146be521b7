// Kernels of the batched ordered-subset AT engine (gfx950).
//
// One launch per phase serves every unit of a batch; units with lines and
// units with matrices have projection kernels, and launches, of their own.
// The global block index is mapped to (unit, local block) through the
// BlockMap passed by value, each of the 8 XCDs owning a contiguous eighth of
// each unit's blocks (unit_block).  K, the number of jobs of a unit, selects a
// code path compiled for that K; a launch uses the kernel compiled for K <= 1,
// <= 4 or <= 8 that covers its units, so it keeps the register budget of that
// case.
//
// FP32 fan beams project along the rays' lines (Lines, runtime.hpp;
// line_fp_unit, line_bp_unit, k_line_project): no matrix is read, a ray's
// lengths follow from its position in each line of pixels.  The other fan
// beams' forward projection is the checkpointed walk (walk_otf): the tracer
// re-run from stored per-segment states, a block holding 32 neighbouring rays
// x 8 segments.  Their back projection (and the forward projection of other
// geometries) reads the sliced matrices (Sell, runtime.hpp): a lane owns one
// pixel column (back) or one segment of one ray (forward) and walks it in
// entry order with a Kahan sum, four entries per 16-byte load, a wave's loads
// contiguous; neighbouring lanes own neighbouring rays / pixels, so one gather
// instruction touches few cache lines.  The back projection stages each 16 x
// 16 pixel block's residual values in LDS first where they fit (bp_unit).
// Images are stored in 4 x 8 tiles (tile_index).  Partial sums of an item are
// combined in a fixed order.
#include "engine.hpp"
#include "tracers.hpp"

#include <cmath>
#include <type_traits>

namespace mi {

namespace {

// Global address space.  The unit table is read from device memory, so the
// compiler cannot infer that its pointers are global and would emit flat
// loads (64-bit addresses, counted against lgkmcnt as well as vmcnt, which
// serialises them with every scalar and LDS wait).  Every access of the
// engine goes through these pointers instead.
#define GL __attribute__((address_space(1)))

template <typename T>
struct UG {
    const GL int64_t *fs_slice0, *fs_base;
    const GL int32_t *fs_T;
    const GL uint32_t *fs_idx, *fs_first;
    const GL int16_t *fs_d16;
    const GL T *fs_len;
    const GL int64_t *bs_slice0, *bs_base;
    const GL int32_t *bs_T;
    const GL uint32_t *bs_idx, *bs_first;
    const GL int16_t *bs_d16;
    const GL T *bs_len;
    const GL uint16_t *bs_slot16;
    const GL int32_t *bs_vlo, *bs_voff;
    const GL int64_t *bs_vtab0;
    const GL double *ot_lam, *ot_ax, *ot_ay, *ot_stx, *ot_sty;
    const GL int32_t *ot_cx, *ot_cy, *ot_sg, *ot_cnt;
    const GL int64_t *ln_slice0;
    const GL double *ln_mb, *ln_len;
    const GL double *ln_inv;
    const GL int32_t *ln_drop, *ln_skip, *ln_rng;
    const GL double *ln_mx, *ln_my;
    const GL float *ln_ix, *ln_iy;
    const GL int64_t *ln_win0;
    const GL int32_t *ln_views;
    const GL int64_t *sub_row0;
    GL T *g, *r, *u, *v, *d, *w, *ul, *dl;
    GL float *px, *py;
    GL char *qx, *qy;
    int64_t npix_t, nrows, part_off, cap;
    int nx, ny, tny, K, fs_P, bs_P, job0, nbins, ln_arc, ln_vstride;
    float ln_sod, ln_k, ln_pix;
    template <typename Desc>   // UnitDesc<T>, of any address space
    __device__ __forceinline__ explicit UG(Desc &D)
        : fs_slice0((const GL int64_t *)D.fs_slice0), fs_base((const GL int64_t *)D.fs_base),
          fs_T((const GL int32_t *)D.fs_T), fs_idx((const GL uint32_t *)D.fs_idx),
          fs_first((const GL uint32_t *)D.fs_first), fs_d16((const GL int16_t *)D.fs_d16),
          fs_len((const GL T *)D.fs_len), bs_slice0((const GL int64_t *)D.bs_slice0),
          bs_base((const GL int64_t *)D.bs_base), bs_T((const GL int32_t *)D.bs_T),
          bs_idx((const GL uint32_t *)D.bs_idx), bs_first((const GL uint32_t *)D.bs_first),
          bs_d16((const GL int16_t *)D.bs_d16), bs_len((const GL T *)D.bs_len),
          bs_slot16((const GL uint16_t *)D.bs_slot16), bs_vlo((const GL int32_t *)D.bs_vlo),
          bs_voff((const GL int32_t *)D.bs_voff), bs_vtab0((const GL int64_t *)D.bs_vtab0),
          ot_lam((const GL double *)D.ot_lam), ot_ax((const GL double *)D.ot_ax), ot_ay((const GL double *)D.ot_ay),
          ot_stx((const GL double *)D.ot_stx), ot_sty((const GL double *)D.ot_sty),
          ot_cx((const GL int32_t *)D.ot_cx), ot_cy((const GL int32_t *)D.ot_cy),
          ot_sg((const GL int32_t *)D.ot_sg), ot_cnt((const GL int32_t *)D.ot_cnt),
          ln_slice0((const GL int64_t *)D.ln_slice0), ln_mb((const GL double *)D.ln_mb),
          ln_len((const GL double *)D.ln_len), ln_inv((const GL double *)D.ln_inv),
          ln_drop((const GL int32_t *)D.ln_drop), ln_skip((const GL int32_t *)D.ln_skip), ln_rng((const GL int32_t *)D.ln_rng), ln_mx((const GL double *)D.ln_mx),
          ln_my((const GL double *)D.ln_my), ln_ix((const GL float *)D.ln_ix), ln_iy((const GL float *)D.ln_iy),
          ln_win0((const GL int64_t *)D.ln_win0), ln_views((const GL int32_t *)D.ln_views),
          sub_row0((const GL int64_t *)D.sub_row0), g((GL T *)D.g), r((GL T *)D.r), u((GL T *)D.u),
          v((GL T *)D.v), d((GL T *)D.d), w((GL T *)D.w), ul((GL T *)D.ul), dl((GL T *)D.dl), px((GL float *)D.px), py((GL float *)D.py), qx((GL char *)D.qx), qy((GL char *)D.qy),
          npix_t(D.npix_t), nrows(D.nrows),
          part_off(D.part_off), cap(D.cap), nx(D.nx), ny(D.ny), tny(D.tny), K(D.K), fs_P(D.fs_P), bs_P(D.bs_P),
          job0(D.job0), nbins(D.nbins), ln_arc(D.ln_arc), ln_vstride(D.ln_vstride), ln_sod(D.ln_sod), ln_k(D.ln_k),
          ln_pix(D.ln_pix) {}
    // Tiled index of pixel (i, j), or -1 outside the image.
    __device__ __forceinline__ int64_t at(int i, int j) const {
        return (i < 0 || j < 0 || i >= nx || j >= ny) ? -1 : tile_index(i, j, tny);
    }
};

template <typename T>
__device__ __forceinline__ const GL JobParams &jpar(const EngArgs<T> &a, int js) {
    return ((const GL JobParams *)a.jp)[js];
}
template <typename T>
__device__ __forceinline__ GL Scalars &jsc(const EngArgs<T> &a, int js) {
    return ((GL Scalars *)a.sc)[js];
}

#ifndef MI_NT_FP
#define MI_NT_FP 1      // non-temporal matrix streams in the forward projector
#endif
#ifndef MI_NT_BP
#define MI_NT_BP 1      // ... and in the back projector
#endif
// Staged back projection: the walk's first stream loads issued with the
// residual copies, before their wait (0: never, 1: K = 1 only, 2: every K).
// Measured on the 64-job batch: with every K the K <= 4 staged launch took
// 678 us against 617 us unprimed; K = 1 only: 622 us.
#ifndef MI_BP_PRIME
#define MI_BP_PRIME 1
#endif
#ifndef MI_STEPS
#define MI_STEPS 8      // steps of a projector lane in flight (K <= 2; 4 above)
#endif

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Matrix streams are read once per launch; non-temporal loads keep them from
// evicting the image / residual lines that the gathers reuse from L2.
template <bool NT, typename V>
__device__ __forceinline__ V stream_ld(const GL V *p) {
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}

// K consecutive values at p (p is aligned to K * sizeof(T)).
template <typename T, int K>
__device__ __forceinline__ void loadk(const GL T *__restrict__ p, T (&o)[K]) {
    constexpr int B = K * (int)sizeof(T);
    if constexpr (B >= 16) {
#pragma unroll
        for (int c = 0; c < B / 16; ++c) {
            const u32x4 a = ((const GL u32x4 *)p)[c];
            __builtin_memcpy(&o[c * (16 / (int)sizeof(T))], &a, 16);
        }
    } else if constexpr (B == 8) {
        const uint64_t a = *(const GL uint64_t *)p;
        __builtin_memcpy(&o[0], &a, 8);
    } else {
        o[0] = p[0];
    }
}

// Gathers through a raw buffer resource: a 32-bit byte offset per lane against
// a base held in scalar registers (the image is < 4 GiB).
#ifndef MI_BUF_GATHER
#define MI_BUF_GATHER 1
#endif
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, 0x00020000);
}

template <typename T, int K>
__device__ __forceinline__ void loadk_buf(__amdgpu_buffer_rsrc_t rs, uint32_t off, T (&o)[K]) {
    constexpr int B = K * (int)sizeof(T);
    if constexpr (B >= 16) {
#pragma unroll
        for (int c = 0; c < B / 16; ++c) {
            const u32x4 a = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(off + 16 * c), 0, 0);
            __builtin_memcpy(&o[c * (16 / (int)sizeof(T))], &a, 16);
        }
    } else if constexpr (B == 8) {
        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
        const u32x2 a = __builtin_amdgcn_raw_buffer_load_b64(rs, (int)off, 0, 0);
        __builtin_memcpy(&o[0], &a, 8);
    } else {
        const uint32_t a = __builtin_amdgcn_raw_buffer_load_b32(rs, (int)off, 0, 0);
        __builtin_memcpy(&o[0], &a, 4);
    }
}

template <typename T, int K>
__device__ __forceinline__ void storek(GL T *__restrict__ p, const T (&o)[K]) {
    constexpr int B = K * (int)sizeof(T);
    if constexpr (B >= 16) {
#pragma unroll
        for (int c = 0; c < B / 16; ++c) {
            u32x4 a;
            __builtin_memcpy(&a, &o[c * (16 / (int)sizeof(T))], 16);
            ((GL u32x4 *)p)[c] = a;
        }
    } else if constexpr (B == 8) {
        uint64_t a;
        __builtin_memcpy(&a, &o[0], 8);
        *(GL uint64_t *)p = a;
    } else {
        p[0] = o[0];
    }
}

template <typename T, int K>
__device__ __forceinline__ void zerok(T (&o)[K]) {
#pragma unroll
    for (int j = 0; j < K; ++j) o[j] = T(0);
}

// Sums v[j] over aligned groups of P lanes (fixed butterfly).
template <int K>
__device__ __forceinline__ void group_sums(double (&v)[K], int P) {
    for (int o = P >> 1; o > 0; o >>= 1)
#pragma unroll
        for (int j = 0; j < K; ++j) v[j] += __shfl_xor(v[j], o, kWave);
}

// This workgroup's unit and block of it.  Each XCD (workgroups go to the 8
// XCDs in turn) takes an eighth of every unit's blocks, a contiguous one, unit
// by unit: units differ tenfold in the cost of a block, and with the whole
// launch cut into eight runs of blocks some XCDs had the costly units and the
// others waited (64 slices of 17 geometries, K = 1 to 8: 2385 AT iterations/s,
// now 3400; eight jobs of two geometries 27.5 and 25.8 ms).  A launch of one
// unit is cut as before.  False for the padding.
__device__ __forceinline__ bool unit_block(const BlockMap &m, int &ui, int &lb) {
    const int x = (int)(blockIdx.x & 7), p = (int)(blockIdx.x >> 3) * 8;
    if (p >= m.start[m.nunits]) return false;
    int lo = 0, hi = m.nunits;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (m.start[mid] <= p) lo = mid;
        else hi = mid;
    }
    ui = lo;
    lb = (x * (m.start[lo + 1] - m.start[lo]) + (p - m.start[lo])) / 8;
    return lb < m.count[lo];
}

template <typename T>
__device__ __forceinline__ bool job_live(const EngArgs<T> &a, int js) {
    return jpar(a, js).active && !jsc(a, js).done;
}

template <typename T>
__device__ __forceinline__ bool unit_idle(const EngArgs<T> &a, const UG<T> &U) {
    for (int j = 0; j < U.K; ++j)
        if (job_live(a, U.job0 + j)) return false;
    return true;
}

template <typename T>
__device__ __forceinline__ GL double *part_at(const EngArgs<T> &a, const UG<T> &U, int slot, int j) {
    return (GL double *)a.part + U.part_off + ((int64_t)slot * U.K + j) * U.cap;
}

// Sum (or max) of one value per thread (of the block's first kBlock) for each
// of K jobs; thread j < K stores job j's block total at part_at(slot, j)[lb].
// Fixed order.
template <typename T, int K, bool MAX>
__device__ __forceinline__ void block_store(const EngArgs<T> &a, const UG<T> &U, int slot, int lb,
                                            const double (&m)[K], double *lds) {
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    if (wv < kBlock / kWave)
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const double t = MAX ? wave_max(m[j]) : group_sum<kWave>(m[j]);
            if (lane == 0) lds[wv * K + j] = t;
        }
    __syncthreads();
    if (threadIdx.x < K) {
        double t = 0.0;
        for (int w = 0; w < kBlock / kWave; ++w) t = MAX ? fmax(t, lds[w * K + threadIdx.x]) : t + lds[w * K + threadIdx.x];
        part_at(a, U, slot, threadIdx.x)[lb] = t;
    }
}

// ---------------------------------------------------------------------------
// One projector lane: its entries t = 0 .. n-1 (sell_pos), Kahan-summed in
// entry order (zero-length padding skipped), gathering K interleaved values of
// `x` per entry.  Index stream: absolute (ip) or, when D16, 16-bit
// differences (dp) accumulated from the lane's first index.  ip / dp / lp
// point at the lane's first group; a group of 4 steps is one 16-byte length
// load and one 16-byte (absolute) or 8-byte (differences) index load.
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

#define LDSP __attribute__((address_space(3)))
enum IdxMode { IM_ABS32 = 0, IM_DELTA16 = 1, IM_SLOT16 = 2 };

// Stream registers of one pipeline stage of walk: GR groups of kGroup
// entries (index word and length) per lane.
template <typename T, int K>
struct Stage {
    static constexpr int GR = (K <= 2) ? MI_STEPS / kGroup : 1;   // groups per pipeline stage
    uint32_t sv[GR][kGroup];
    T lv[GR][kGroup];
};

// Issues the stream loads of groups g0 .. g0 + GR - 1 of a lane into b.
template <typename T, int K, bool NT, int IM>
__device__ __forceinline__ void stage_fetch(Stage<T, K> &b, const GL uint32_t *__restrict__ ip,
                                            const GL int16_t *__restrict__ dp, const GL T *__restrict__ lp, int g0) {
    constexpr bool D16 = IM != IM_ABS32;
    constexpr int64_t kStride = kGroup * kWave;   // entries between a lane's groups
#pragma unroll
    for (int r = 0; r < Stage<T, K>::GR; ++r) {
        const int64_t o = (int64_t)(g0 + r) * kStride;
        if constexpr (IM == IM_SLOT16) {
            const u32x2 a = stream_ld<NT>((const GL u32x2 *)(dp + o));
            b.sv[r][0] = a.x & 0xffffu;
            b.sv[r][1] = a.x >> 16;
            b.sv[r][2] = a.y & 0xffffu;
            b.sv[r][3] = a.y >> 16;
        } else if constexpr (D16) {
            const u32x2 a = stream_ld<NT>((const GL u32x2 *)(dp + o));
            b.sv[r][0] = (uint32_t)(int32_t)(int16_t)(a.x & 0xffffu);
            b.sv[r][1] = (uint32_t)(int32_t)(int16_t)(a.x >> 16);
            b.sv[r][2] = (uint32_t)(int32_t)(int16_t)(a.y & 0xffffu);
            b.sv[r][3] = (uint32_t)(int32_t)(int16_t)(a.y >> 16);
        } else {
            const u32x4 a = stream_ld<NT>((const GL u32x4 *)(ip + o));
            b.sv[r][0] = a.x; b.sv[r][1] = a.y; b.sv[r][2] = a.z; b.sv[r][3] = a.w;
        }
        if constexpr (sizeof(T) == 4) {
            const u32x4 a = stream_ld<NT>((const GL u32x4 *)(lp + o));
            __builtin_memcpy(&b.lv[r][0], &a, 16);
        } else {
            const u32x4 a = stream_ld<NT>((const GL u32x4 *)(lp + o));
            const u32x4 c = stream_ld<NT>((const GL u32x4 *)(lp + o) + 1);
            __builtin_memcpy(&b.lv[r][0], &a, 16);
            __builtin_memcpy(&b.lv[r][2], &c, 16);
        }
    }
}

// The first stage of a walk over n entries (none when the walk has no full
// stage); a walk with PRIMED set starts from it.
template <typename T, int K, bool NT, int IM>
__device__ __forceinline__ void walk_prime(Stage<T, K> &b, const GL uint32_t *ip, const GL int16_t *dp,
                                           const GL T *lp, int n) {
    if (n / kGroup / Stage<T, K>::GR > 0) stage_fetch<T, K, NT, IM>(b, ip, dp, lp, 0);
}

// IM: absolute 32-bit indices (ip), 16-bit differences (dp, from `cur`), or
// 16-bit LDS slots (dp read unsigned).  LDSG: gather from `lx` (LDS) instead
// of the global array x.  b holds the stage in flight; with PRIMED the caller
// has issued the first one (walk_prime).
template <typename T, int K, bool NT, int IM, bool LDSG = false, bool PRIMED = false>
__device__ __forceinline__ void walk(const GL uint32_t *__restrict__ ip, const GL int16_t *__restrict__ dp,
                                     uint32_t cur, const GL T *__restrict__ lp, int n, const GL T *__restrict__ x,
                                     uint32_t xbytes, Acc<T> (&acc)[K], Stage<T, K> &b,
                                     const LDSP T *lx = nullptr) {
    constexpr bool D16 = IM != IM_ABS32;
    constexpr int GR = Stage<T, K>::GR;
    constexpr int64_t kStride = kGroup * kWave;             // entries between a lane's groups
#if MI_BUF_GATHER
    const __amdgpu_buffer_rsrc_t xr = make_rsrc((const void *)x, xbytes);
#else
    (void)xbytes;
#endif
    auto fetch = [&](int g0) { stage_fetch<T, K, NT, IM>(b, ip, dp, lp, g0); };
    auto gather = [&](uint32_t id, T (&o)[K]) {
        if constexpr (LDSG) {
#pragma unroll
            for (int j = 0; j < K; ++j) o[j] = lx[id * K + j];
        } else {
#if MI_BUF_GATHER
            loadk_buf<T, K>(xr, id * (uint32_t)(K * sizeof(T)), o);
#else
            loadk<T, K>(x + (uint32_t)(id * K), o);
#endif
        }
    };
    const int ng = n / kGroup, full = ng / GR;
    // Software pipeline: the next stage's stream loads are issued after the
    // current stage's gathers (the barriers keep that order) and before they
    // are consumed, so a lane waits for one memory round trip per stage.
    if (!PRIMED && full > 0) fetch(0);
    int g = 0;
    for (int c = 0; c < full; ++c, g += GR) {
        uint32_t id[GR][kGroup];
        T ln[GR][kGroup], xv[GR][kGroup][K];
#pragma unroll
        for (int r = 0; r < GR; ++r)
#pragma unroll
            for (int q = 0; q < kGroup; ++q) {
                if constexpr (IM == IM_DELTA16) {
                    cur += b.sv[r][q];
                    id[r][q] = cur;
                } else {
                    id[r][q] = b.sv[r][q];
                }
                ln[r][q] = b.lv[r][q];
            }
#pragma unroll
        for (int r = 0; r < GR; ++r)
#pragma unroll
            for (int q = 0; q < kGroup; ++q) gather(id[r][q], xv[r][q]);
        __builtin_amdgcn_sched_barrier(0);
        fetch(c + 1 < full ? g + GR : g);   // the last stage re-reads its own groups
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < GR; ++r)
#pragma unroll
            for (int q = 0; q < kGroup; ++q)
#pragma unroll
                for (int j = 0; j < K; ++j) acc[j].add_prod_if(xv[r][q][j], ln[r][q], ln[r][q] != T(0));
    }
    for (; g < ng; ++g) {
        const int64_t o = (int64_t)g * kStride;
        uint32_t id[kGroup];
        T ln[kGroup], xv[kGroup][K];
        if constexpr (IM == IM_SLOT16) {
            const u32x2 a = stream_ld<NT>((const GL u32x2 *)(dp + o));
            const uint32_t w[2] = {a.x, a.y};
#pragma unroll
            for (int q = 0; q < kGroup; ++q) id[q] = (w[q >> 1] >> (16 * (q & 1))) & 0xffffu;
        } else if constexpr (D16) {
            const u32x2 a = stream_ld<NT>((const GL u32x2 *)(dp + o));
            const uint32_t w[2] = {a.x, a.y};
#pragma unroll
            for (int q = 0; q < kGroup; ++q) {
                cur += (uint32_t)(int32_t)(int16_t)((w[q >> 1] >> (16 * (q & 1))) & 0xffffu);
                id[q] = cur;
            }
        } else {
            const u32x4 a = stream_ld<NT>((const GL u32x4 *)(ip + o));
            id[0] = a.x; id[1] = a.y; id[2] = a.z; id[3] = a.w;
        }
#pragma unroll
        for (int q = 0; q < kGroup; ++q) ln[q] = lp[o + q];
#pragma unroll
        for (int q = 0; q < kGroup; ++q) gather(id[q], xv[q]);
#pragma unroll
        for (int q = 0; q < kGroup; ++q)
#pragma unroll
            for (int j = 0; j < K; ++j) acc[j].add_prod_if(xv[q][j], ln[q], ln[q] != T(0));
    }
}

// Walks lane `lane` of slice sl of one sliced matrix in whichever index form
// it is stored.
template <typename T, int K, bool NT>
__device__ __forceinline__ void walk_slice(const GL int64_t *base, const GL int32_t *Tn, const GL uint32_t *idx,
                                           const GL uint32_t *first, const GL int16_t *d16, const GL T *len,
                                           int64_t sl, int lane, const GL T *x, int64_t xn, Acc<T> (&acc)[K]) {
    const int64_t p0 = sell_pos(base[sl], 0, lane);
    const int n = Tn[sl];
    const uint32_t xb = (uint32_t)(xn * K * (int64_t)sizeof(T));
    Stage<T, K> b;
    if (d16) walk<T, K, NT, IM_DELTA16>(nullptr, d16 + p0, first[sl * kWave + lane], len + p0, n, x, xb, acc, b);
    else walk<T, K, NT, IM_ABS32>(idx + p0, nullptr, 0u, len + p0, n, x, xb, acc, b);
}

// One lane of the checkpointed forward walk: n Siddon steps from the stored
// tracer state, each step's pixel gathered from the tiled image x and its
// length (rounded to T as the stored matrix rounds it) Kahan-summed in step
// order.  The step is siddon_step (tracers.hpp) written with selects instead
// of a branch: the same comparisons and the same additions on the taken side,
// so lam / ax / ay and the lengths are bit-identical.  The pixel position is
// carried as byte offsets into the tiled layout, X = 4 E cx and Y = E cy
// (E bytes per pixel), so the tiled offset is
//   E tile_index(cx, cy) = (cx >> 2) (32 tny - 16) E + X + (cy >> 2) 12 E + Y.
// Every step of a lane is summed, zero-length crossings included (as the
// oracle sums every matrix entry).  Steps go in groups of OS, software
// pipelined: the next group is traced and its gathers issued before this
// group's gathers are consumed.
template <typename T, int K>
__device__ __forceinline__ void walk_otf(const UG<T> &U, int64_t q, const GL T *__restrict__ x, Acc<T> (&acc)[K]) {
#ifndef MI_OTF_OS8
#define MI_OTF_OS8 2   // steps in flight at K = 8 (4: 116 VGPRs, slower at every image size)
#endif
    constexpr int OS = (K <= 2) ? 8 : (K == 4 ? 4 : MI_OTF_OS8);
    constexpr uint32_t E = K * sizeof(T), LE = __builtin_ctz(E);
    double lam = U.ot_lam[q], ax = U.ot_ax[q], ay = U.ot_ay[q];
    const double stx = U.ot_stx[q], sty = U.ot_sty[q];
    const int sgb = U.ot_sg[q];
    uint32_t X = (uint32_t)U.ot_cx[q] * (4 * E), Y = (uint32_t)U.ot_cy[q] * E;
    const uint32_t dX = (sgb & 1) ? 4 * E : 0u - 4 * E, dY = (sgb & 2) ? E : 0u - E;
    const uint32_t rowE = (uint32_t)(U.tny * (kTileH * kTileW) - 16) * E;
    const int n = U.ot_cnt[q];
#if MI_BUF_GATHER
    const __amdgpu_buffer_rsrc_t xr = make_rsrc((const void *)x, (uint32_t)(U.npix_t * (int64_t)E));
#endif
    auto step = [&](uint32_t &off, T &ln) {
        const bool bx = ax <= ay;
        const double nxt = bx ? ax : ay;
        ln = (T)(nxt - lam);
        lam = nxt;
        off = (uint32_t)__umul24(X >> (4 + LE), rowE) + X + (uint32_t)__umul24(Y >> (2 + LE), 12 * E) + Y;
        double nax = ax + stx, nay = ay + sty;
        // both sums exist on every lane: keeps the selects below from being
        // turned back into a divergent branch
        asm volatile("" : "+v"(nax), "+v"(nay));
        ax = bx ? nax : ax;
        ay = bx ? ay : nay;
        X += bx ? dX : 0u;
        Y += bx ? 0u : dY;
    };
    auto gather = [&](uint32_t off, T (&o)[K]) {
#if MI_BUF_GATHER
        loadk_buf<T, K>(xr, off, o);
#else
        loadk<T, K>((const GL T *)((const GL char *)x + off), o);
#endif
    };
    auto stage = [&](T (&ln)[OS], T (&xv)[OS][K]) {
        uint32_t off[OS];
#pragma unroll
        for (int k = 0; k < OS; ++k) step(off[k], ln[k]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < OS; ++k) gather(off[k], xv[k]);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto consume = [&](const T (&ln)[OS], const T (&xv)[OS][K]) {
#pragma unroll
        for (int k = 0; k < OS; ++k)
#pragma unroll
            for (int j = 0; j < K; ++j) acc[j].add_prod(xv[k][j], ln[k]);
    };
    const int ng = n / OS;
    T la[OS], lb[OS], xa[OS][K], xb[OS][K];
    int g = 0;
    if (ng > 0) {
        stage(la, xa);
        for (g = 1; g + 1 < ng; g += 2) {
            stage(lb, xb);
            consume(la, xa);
            stage(la, xa);
            consume(lb, xb);
        }
        if (g < ng) {
            stage(lb, xb);
            consume(la, xa);
            consume(lb, xb);
        } else {
            consume(la, xa);
        }
    }
    // the last n % OS steps: traced and gathered together, one round trip
    const int rem = n - ng * OS;
    if (rem > 0) {
        uint32_t off[OS - 1];
        T ln[OS - 1], xv[OS - 1][K];
#pragma unroll
        for (int k = 0; k < OS - 1; ++k)
            if (k < rem) step(off[k], ln[k]);
#pragma unroll
        for (int k = 0; k < OS - 1; ++k)
            if (k < rem) gather(off[k], xv[k]);
#pragma unroll
        for (int k = 0; k < OS - 1; ++k)
            if (k < rem)
#pragma unroll
                for (int j = 0; j < K; ++j) acc[j].add_prod(xv[k][j], ln[k]);
    }
}

// Forward projection of subset s: a block is 4 slices (one per wave).
// RESID: r = g - A u (stored), partial sum r^2; else partial sum (A d)^2.
static_assert(kOtfWaves == 4, "the forward walk's cross-wave combination is written for 4 waves");

// FM: 1 when every unit of the launch has the checkpointed walk (the sliced
// branch is not compiled), 3 when either form may occur.
template <typename T, int K, bool RESID, int FM>
__device__ __forceinline__ void fp_unit(const EngArgs<T> &a, const UG<T> &U, int s, int lb, double *lds,
                                        double *ldr /* kBlock / kOtfPerWave * K */) {
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    const int P = U.fs_P, C = kWave / P;
    const int64_t sl0 = U.fs_slice0[s], li = (int64_t)lb * (kBlock / kWave) + wv;
    double m[K];
#pragma unroll
    for (int j = 0; j < K; ++j) m[j] = 0.0;
    if (li < U.fs_slice0[s + 1] - sl0) {
        const int64_t sl = sl0 + li;
        Acc<T> acc[K];
        double tot[K];
        int64_t row;
        bool owner;
        if (FM == 1 || U.ot_cnt) {
            // the block is kOtfRays rays x kOtfSeg segments (runtime.hpp);
            // a ray's segment sums combine in a fixed tree: inside the wave
            // (lanes a, a + kOtfRays, ...), then over the block's waves
            walk_otf<T, K>(U, sl * kWave + lane, RESID ? U.u : U.d, acc);
#pragma unroll
            for (int j = 0; j < K; ++j) tot[j] = acc[j].value();
            for (int o = kOtfRays; o < kWave; o <<= 1)
#pragma unroll
                for (int j = 0; j < K; ++j) tot[j] += __shfl_xor(tot[j], o, kWave);
            if (lane < kOtfRays)
#pragma unroll
                for (int j = 0; j < K; ++j) ldr[(wv * kOtfRays + lane) * K + j] = tot[j];
            __syncthreads();
            if (wv == 0 && lane < kOtfRays)
#pragma unroll
                for (int j = 0; j < K; ++j) {
                    const double *q = ldr + lane * K + j;
                    tot[j] = (q[0] + q[kOtfRays * K]) + (q[2 * kOtfRays * K] + q[3 * kOtfRays * K]);
                }
            row = U.sub_row0[s] + (int64_t)lb * kOtfRays + lane;
            owner = wv == 0 && lane < kOtfRays;
        } else if constexpr (FM != 1) {
            walk_slice<T, K, MI_NT_FP>(U.fs_base, U.fs_T, U.fs_idx, U.fs_first, U.fs_d16, U.fs_len, sl, lane,
                                       RESID ? U.u : U.d, U.npix_t, acc);
#pragma unroll
            for (int j = 0; j < K; ++j) tot[j] = acc[j].value();
            group_sums<K>(tot, P);
            row = U.sub_row0[s] + li * C + lane / P;
            owner = lane % P == 0;
        }
        if (owner && row < U.sub_row0[s + 1]) {
            if (RESID) {
                T gg[K], o[K];
                loadk<T, K>(U.g + row * K, gg);
#pragma unroll
                for (int j = 0; j < K; ++j) {
                    o[j] = (T)((double)gg[j] - tot[j]);
                    m[j] = (double)o[j] * (double)o[j];
                }
                storek<T, K>(U.r + row * K, o);
            } else {
#pragma unroll
                for (int j = 0; j < K; ++j) m[j] = tot[j] * tot[j];
            }
        }
    }
    block_store<T, K, false>(a, U, RESID ? SL_DF : SL_AD, lb, m, lds);
}

// Forward projection along the lines (Lines, runtime.hpp), FP32.
//
// One workgroup is one group of kLineRays neighbouring rays; its kLineWaves
// waves cut the lines the group crosses into as many runs, one lane per ray.
// At line a of the dominant axis a ray covers at most two neighbouring pixels
// of that line, so a step is one 2K-value load from the projection image that
// holds the line contiguously and the two products
//   w u[j] + (1 - w) u[j - 1],   w = min(1, frac(hi) / |m|),
// with hi the upper end of the covered interval, j = floor(hi).  Weights and
// products are double: a pixel that the ray does not meet has weight 0 or 1 - w
// = 0 exactly and adds nothing, however large it is (as a difference in FP32 it
// left 2^-24 of itself in the ray).  hi advances
// by m, one double add, and is biased by 2^20 + 2^19 so that its low word is
// frac(hi) 2^32 and its high word j plus a constant (rounded to 2^-33 pixel a
// step, under 2^-24 over a run of 512 lines).  Positions outside the image
// read the zero padding.  The run's sum is double; a ray's runs are added in
// order, times the ray's length per line.  The line in which the tracer leaves
// out a piece (Lines) is not part of the runs: its other pixel is added last
// (line_kept).
//
// What bounds it: the load, 17 accesses of the CU's L1 a line (four lanes an
// access), beside 11 VALU instructions, eight of them on doubles at half rate; a
// line brings the two pixels' entries
// (1.4 entries of the matrix on average), where the checkpointed walk spends 26
// VALU instructions and such a load on each entry.  512 x 512 pixels, 60 views
// of 736 bins: 18.8 us (residual) and 18.4 us, against 32.4 and 32.1 us of the
// walk (17.4 and 17.0 with the interpolation in FP32).  Four lines in flight keep
// eight waves a SIMD; eight of them and four waves: 20.2 / 19.9.  The run length
// is a multiple of 8 whatever K is, so a ray's sum does not depend on K.
constexpr int kLineWaves = 8, kLineBlock = kLineWaves * kWave;
constexpr double kLineBias = 1572864.0;                    // 2^20 + 2^19
constexpr int kLineHi0 = (0x413 << 20) + (1 << 19);        // high word of kLineBias

template <int B, typename V>
__device__ __forceinline__ void load_bytes(__amdgpu_buffer_rsrc_t rs, uint32_t off, int line, V &o) {
    static_assert(sizeof(V) == B, "");
    if constexpr (B == 8) {
        const u32x2 a = __builtin_amdgcn_raw_buffer_load_b64(rs, (int)off, line, 0);
        __builtin_memcpy(&o, &a, 8);
    } else {
#pragma unroll
        for (int c = 0; c < B / 16; ++c) {
            const u32x4 a = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(off + 16 * c), line, 0);
            __builtin_memcpy((char *)&o + 16 * c, &a, 16);
        }
    }
}

// How a projection image is held.  u is projected with its remainder
// (axpy_unit), to 40 bits: as doubles for up to two jobs, whose pair is one load
// as the FP32 pair is (one job; two jobs two), for four and eight as FP32, rounded
// towards zero, and the 16 bits of the mantissa behind it: six bytes a value,
// three loads a line of four jobs where doubles take four and FP32 alone two.
// The value is the same in either form.  d, and an image given in FP32, is FP32.
enum LineForm { LF_F32, LF_F64, LF_SPLIT };
template <int K, bool RESID>
constexpr LineForm line_form() { return !RESID ? LF_F32 : K <= 2 ? LF_F64 : LF_SPLIT; }
// The double of the two parts: the FP32 part's low 29 bits are zero.
__device__ __forceinline__ double line_join(float f, uint32_t lo13 /* the 16 bits, 13 up */) {
    const double d = (double)f;
    return __hiloint2double(__double2hiint(d), (int)((uint32_t)__double2loint(d) | lo13));
}
__device__ __forceinline__ void line_split(double v, float &f, uint32_t &lo16) {
    f = (float)v;
    lo16 = 0;
    if (!(fabs((double)f) < INFINITY) || fabsf(f) < 2.0f * 1.17549435e-38f) return;   // (no bits behind these)
    if (fabs((double)f) > fabs(v)) f = __uint_as_float(__float_as_uint(f) - 1);
    lo16 = (uint32_t)__double2loint(v) >> 13 & 0xffff;
}

struct LineImg {
    const GL float *f;       // LF_F32, LF_SPLIT
    const GL void *q;        // LF_F64: the doubles, LF_SPLIT: the remainders
    template <LineForm F>
    __device__ __forceinline__ double at(int64_t i) const {
        if constexpr (F == LF_F32) return (double)f[i];
        else if constexpr (F == LF_F64) return ((const GL double *)q)[i];
        else return line_join(f[i], (uint32_t)((const GL uint16_t *)q)[i] << 13);
    }
};
// What one line brings: the values of both pixels (j - 1, then j), K each.
template <int K, LineForm F>
struct LinePair {
    float f[F == LF_F64 ? 1 : 2 * K];
    double d[F == LF_F64 ? 2 * K : 1];
    uint32_t lo[F == LF_SPLIT ? K : 1];
    __device__ __forceinline__ double at(int i) const {
        if constexpr (F == LF_F64) {
            double x = d[i];
            asm volatile("" : "+v"(x));
            return x;
        } else {
            float x = f[i];
            asm volatile("" : "+v"(x));   // (converted where it is used, not all values before)
            if constexpr (F == LF_F32) return (double)x;
            uint32_t l = lo[i >> 1];
            asm volatile("" : "+v"(l));
            return line_join(x, i & 1 ? l >> 3 & 0x1fffe000u : (l & 0xffffu) << 13);
        }
    }
};

// Pixel (i, j) of the unit's projection images: d, or u and its remainder.
template <typename T>
__device__ __forceinline__ void proj_at(const UG<T> &U, int i, int j, int64_t &x, int64_t &y) {
    x = ((int64_t)i * line_stride(U.ny) + j + kLinePad) * U.K;
    y = ((int64_t)j * line_stride(U.nx) + i + kLinePad) * U.K;
}
template <typename T, int K>
__device__ __forceinline__ void put_proj_d(const UG<T> &U, int i, int j, const float (&d)[K]) {
    int64_t x, y;
    proj_at(U, i, j, x, y);
    storek<float, K>(U.px + x, d);
    storek<float, K>(U.py + y, d);
}
template <typename T, int K>
__device__ __forceinline__ void put_proj_u(const UG<T> &U, int i, int j, const T (&u)[K], const T (&ul)[K]) {
    int64_t x, y;
    proj_at(U, i, j, x, y);
    float f[K];
    uint32_t lo[K];
#pragma unroll
    for (int k = 0; k < K; ++k) line_split((double)u[k] + (double)ul[k], f[k], lo[k]);
    if constexpr (line_form<K, true>() == LF_F64) {
        double v[K];
#pragma unroll
        for (int k = 0; k < K; ++k) v[k] = line_join(f[k], lo[k] << 13);
        storek<double, K>((GL double *)U.qx + x, v);
        storek<double, K>((GL double *)U.qy + y, v);
    } else {
        uint16_t l[K];
#pragma unroll
        for (int k = 0; k < K; ++k) l[k] = (uint16_t)lo[k];
        storek<float, K>(U.px + x, f);
        storek<float, K>(U.py + y, f);
        storek<uint16_t, K>((GL uint16_t *)U.qx + x, l);
        storek<uint16_t, K>((GL uint16_t *)U.qy + y, l);
    }
}

// Adds this lane's ray over lines c0 .. c0 + n - 1 (n a multiple of 8), without
// line `skip`, to acc.
template <int K, LineForm F>
__device__ __forceinline__ void line_run(const LineImg &img, int nb, int c0, int n, double m, double b0, double inv, int skip,
                                         double (&acc)[K]) {
    constexpr int OS = K <= 2 ? (F == LF_F64 && K == 2 ? 2 : 4) : (K == 4 ? (F == LF_SPLIT ? 4 : 2) : (F == LF_SPLIT ? 2 : 1));
    constexpr int E = K * (F == LF_F64 ? 8 : 4);   // bytes of a pixel
    const uint32_t lineb = (uint32_t)line_stride(nb) * E;
    const int64_t first = (int64_t)c0 * line_stride(nb) * K;
    const __amdgpu_buffer_rsrc_t rs =
        F == LF_F64 ? make_rsrc((const void *)((const GL double *)img.q + first), n * lineb)
                    : make_rsrc((const void *)(img.f + first), n * lineb);
    const __amdgpu_buffer_rsrc_t rl = make_rsrc((const void *)((const GL uint16_t *)img.q + first), n * lineb / 2);
    double hi = b0 + 0.5 * fabs(m) + m * c0 + kLineBias;
    const double sc = inv * 2.3283064365386963e-10;   // 2^-32
    uint32_t at = 0;
    skip -= c0;
    auto stage = [&](uint32_t (&f)[OS], LinePair<K, F> (&x)[OS]) {
        uint32_t off[OS];
#pragma unroll
        for (int k = 0; k < OS; ++k) {
            const int h = __double2hiint(hi);
            f[k] = (uint32_t)__double2loint(hi);
            const int j = max(kLineHi0 - 1, min(h, kLineHi0 + nb + 1));   // zeros beyond
            off[k] = (uint32_t)(j - (kLineHi0 - 1)) * E;                  // pixel j - 1, behind two of padding
            hi += m;
        }
        if (__any((unsigned)skip < (unsigned)OS))
#pragma unroll
            for (int k = 0; k < OS; ++k) off[k] = skip == k ? 0u : off[k];   // zeros
        skip -= OS;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < OS; ++k) {
            const uint32_t line = at + k * lineb;
            if constexpr (F == LF_F64) load_bytes<16 * K>(rs, off[k], (int)line, x[k].d);
            else load_bytes<8 * K>(rs, off[k], (int)line, x[k].f);
            if constexpr (F == LF_SPLIT) load_bytes<4 * K>(rl, off[k] / 2, (int)(line / 2), x[k].lo);
        }
        at += OS * lineb;
        __builtin_amdgcn_sched_barrier(0);
    };
    auto consume = [&](const uint32_t (&f)[OS], const LinePair<K, F> (&x)[OS]) {
#pragma unroll
        for (int k = 0; k < OS; ++k) {
            uint32_t fr = f[k];
            asm volatile("" : "+v"(fr));
            const double w = fmin(fmax((double)fr * sc, 0.0), 1.0), w0 = 1.0 - w;
#pragma unroll
            for (int j = 0; j < K; ++j) acc[j] = __builtin_fma(w, x[k].at(K + j), __builtin_fma(w0, x[k].at(j), acc[j]));
        }
    };
    uint32_t wa[OS], wb[OS];
    LinePair<K, F> xa[OS], xb[OS];
    const int ng = n / OS;
    stage(wa, xa);
    int g = 1;
    for (; g + 1 < ng; g += 2) {
        stage(wb, xb);
        consume(wa, xa);
        stage(wa, xa);
        consume(wb, xb);
    }
    if (g < ng) {
        stage(wb, xb);
        consume(wa, xa);
        consume(wb, xb);
    } else {
        consume(wa, xa);
    }
}

// Pixels j - 1 and j of line a that the ray (m, b0, inv) meets, and j's share.
__device__ __forceinline__ int line_at(double m, double b0, double inv, int a, int nb, double &w) {
    const double pos = b0 + 0.5 * fabs(m) + m * a, jf = floor(pos);
    w = fmin(1.0, (pos - jf) * inv);
    return (int)fmin(fmax(jf, -1.0), (double)(nb + 1));
}

// Value k of the K interleaved ones of the ray's left-out line, over the ray's
// length per line: the pixel of the line that is not `drop`.  img: px or py, by
// the ray's axis (yd: columns), lines of nb pixels.
template <LineForm F>
__device__ __forceinline__ double line_kept(const LineImg &img, int nb, int ny, bool yd, double m, double b0, double inv,
                                            int drop, int K, int k) {
    const int i = drop / ny, jy = drop - i * ny, a = yd ? jy : i, gone = yd ? i : jy;
    double w;
    const int j = line_at(m, b0, inv, a, nb, w);
    const int64_t e = ((int64_t)a * line_stride(nb) + j - 1 + kLinePad) * K + k;
    const double x0 = img.at<F>(e), x1 = img.at<F>(e + K);
    return j == gone ? (1.0 - w) * x0 : j - 1 == gone ? w * x1 : (1.0 - w) * x0 + w * x1;
}

// The sum over lines r0 .. r1 - 1 again where it is not finite: some pixel beside the
// ray, or its left-out one, may not be (0 times it is not 0).  Only what the
// ray crosses counts.
template <LineForm F>
__device__ __forceinline__ double line_ray_again(const LineImg &img, int nb, int ny, bool yd, double m, double b0, double inv,
                                                 int r0, int r1, int drop, int K, int k) {
    double tot = 0.0;
    for (int a = r0; a < r1; ++a) {
        double w;
        const int j = line_at(m, b0, inv, a, nb, w);
        for (int h = 0; h < 2; ++h) {   // pixels j - 1 and j of the line (both may be padding)
            const int jj = j - 1 + h;
            const double part = h ? w : 1.0 - w;
            const bool gone = drop >= 0 && drop == (yd ? jj * ny + a : a * ny + jj) && jj >= 0 && jj < nb;
            if (!gone && part > 1e-6) tot += part * img.at<F>(((int64_t)a * line_stride(nb) + jj + kLinePad) * K + k);
        }
    }
    return tot;
}

// RESID: r = g - A u, stored times the ray's length per line (what the back
// projection weighs), partial sum r^2; else partial sum (A d)^2.
template <int K, bool RESID>
__device__ __forceinline__ void line_fp_unit(const EngArgs<float> &a, const UG<float> &U, int s, int lb, double *lds) {
    const int lane = threadIdx.x & (kWave - 1), wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int64_t g0 = U.ln_slice0[s] / 4;
    if (lb >= U.ln_slice0[s + 1] / 4 - g0) return;
    const int per = (U.nbins + kLineRays - 1) / kLineRays;
    const int view = lb / per, bin = (lb - view * per) * kLineRays + lane;
    const int64_t row = U.sub_row0[s] + (int64_t)view * U.nbins + bin;
    const GL int32_t *rng = U.ln_rng + 4 * (g0 + lb);
    constexpr LineForm F = line_form<K, RESID>();
    const LineImg ix{U.px, U.qx}, iy{U.py, U.qy};
    double m = 0.0, b0 = 0.0, inv = 0.0;
    int skip = -1;
    const bool valid = bin < U.nbins;
    if (valid) {
        m = U.ln_mb[2 * row];
        b0 = U.ln_mb[2 * row + 1];
        inv = U.ln_inv[row];
        skip = U.ln_skip[row];
    }
    double acc[K];
#pragma unroll
    for (int j = 0; j < K; ++j) acc[j] = 0.0;
#pragma unroll
    for (int ax = 0; ax < 2; ++ax) {
        const int r0 = rng[2 * ax], r1 = rng[2 * ax + 1];
        if (r0 >= r1) continue;
        // runs of a multiple of 8 lines; one reaching past r1 reads zeros
        // there (its rays have left the image)
        const int run = ((r1 - r0 + kLineWaves - 1) / kLineWaves + 7) & ~7, c0 = r0 + wv * run;
        if (c0 >= r1) continue;
        const bool mine = valid && (inv < 0.0) == (ax == 1);
        line_run<K, F>(ax ? iy : ix, ax ? U.nx : U.ny, c0, min(run, (r1 - c0 + 7) & ~7),
                    mine ? m : 0.0, mine ? b0 : -64.0, mine ? fabs(inv) : 0.0, mine ? skip : -1, acc);
    }
    // thread (job k, ray): the ray's runs in order
#pragma unroll
    for (int j = 0; j < K; ++j) lds[(wv * K + j) * kLineRays + lane] = acc[j];
    __syncthreads();
    if (wv >= K) return;
    double tot = 0.0;
#pragma unroll
    for (int w = 0; w < kLineWaves; ++w) tot += lds[(w * K + wv) * kLineRays + lane];
    double mm = 0.0;
    if (valid) {
        const double len = U.ln_len[row];
        const bool yd = inv < 0.0;
        const LineImg &img = yd ? iy : ix;
        const int nb = yd ? U.nx : U.ny, drop = skip >= 0 ? U.ln_drop[row] : -1;
        if (skip >= 0) tot += line_kept<F>(img, nb, U.ny, yd, m, b0, fabs(inv), drop, K, wv);
        if (!(fabs(tot) < INFINITY))
            tot = line_ray_again<F>(img, nb, U.ny, yd, m, b0, fabs(inv), rng[2 * yd], min(rng[2 * yd + 1], yd ? U.ny : U.nx),
                                 drop, K, wv);
        tot *= len;
        if (RESID) {
            const double res = (double)U.g[row * K + wv] - tot;
            U.r[row * K + wv] = (float)(res * len);
            const float o = (float)res;
            mm = (double)o * (double)o;
        } else {
            mm = tot * tot;
        }
    }
    mm = group_sum<kWave>(mm);
    if (lane == 0) part_at(a, U, RESID ? SL_DF : SL_AD, wv)[lb] = mm;
}

// One image with its lines' zeros around it, row by row (px) and column by
// column (py), from row-major pixels.
__global__ __launch_bounds__(kBlock) void k_line_planes(const float *__restrict__ img, int nx, int ny,
                                                        float *__restrict__ px, float *__restrict__ py) {
    const int64_t ex = line_elems(nx, ny), ey = line_elems(ny, nx);
    const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (e < ex) {
        const int64_t i = e / line_stride(ny), j = e % line_stride(ny) - kLinePad;
        px[e] = i < nx && j >= 0 && j < ny ? img[i * ny + j] : 0.0f;
    } else if (e < ex + ey) {
        const int64_t j = (e - ex) / line_stride(nx), i = (e - ex) % line_stride(nx) - kLinePad;
        py[e - ex] = j < ny && i >= 0 && i < nx ? img[i * ny + j] : 0.0f;
    }
}

// sino = A img over every view: the forward projection above without a
// residual, for one image.  512 x 512 pixels, 720 views of 736 bins: a
// whole call from and to host arrays 382 us, 1593 with a wave per ray that
// reads the matrix (1332 of it, 2.7 GB); relative error against 64 bits 2.6e-8
// and 3.2e-8.
__global__ __launch_bounds__(kLineBlock) void k_line_project(
    const float *px, const float *py, int nx, int ny, int nbins, int64_t groups, const double2 *__restrict__ mb,
    const double *__restrict__ rinv, const double *__restrict__ rlen, const int32_t *__restrict__ rdrop,
    const int32_t *__restrict__ rskip, const int4 *__restrict__ rng, float *__restrict__ sino) {
    __shared__ double lds[kLineWaves][kLineRays];
    const int lane = threadIdx.x & (kWave - 1), wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int64_t lb = xcd_block();
    if (lb >= groups) return;
    const int per = (nbins + kLineRays - 1) / kLineRays;
    const int64_t view = lb / per;
    const int bin = (int)(lb - view * per) * kLineRays + lane;
    const int64_t row = view * nbins + bin;
    const bool valid = bin < nbins;
    const LineImg ix{(const GL float *)px, nullptr}, iy{(const GL float *)py, nullptr};
    double m = 0.0, b0 = 0.0, inv = 0.0, acc[1] = {0.0};
    int skip = -1;
    if (valid) {
        m = mb[row].x;
        b0 = mb[row].y;
        inv = rinv[row];
        skip = rskip[row];
    }
    const int4 r = rng[lb];
#pragma unroll
    for (int ax = 0; ax < 2; ++ax) {
        const int r0 = ax ? r.z : r.x, r1 = ax ? r.w : r.y;
        if (r0 >= r1) continue;
        const int run = ((r1 - r0 + kLineWaves - 1) / kLineWaves + 7) & ~7, c0 = r0 + wv * run;
        if (c0 >= r1) continue;
        const bool mine = valid && (inv < 0.0) == (ax == 1);
        line_run<1, LF_F32>(ax ? iy : ix, ax ? nx : ny, c0, min(run, (r1 - c0 + 7) & ~7),
                    mine ? m : 0.0, mine ? b0 : -64.0, mine ? fabs(inv) : 0.0, mine ? skip : -1, acc);
    }
    lds[wv][lane] = acc[0];
    __syncthreads();
    if (wv != 0 || !valid) return;
    double tot = 0.0;
#pragma unroll
    for (int w = 0; w < kLineWaves; ++w) tot += lds[w][lane];
    const bool yd = inv < 0.0;
    const LineImg &img = yd ? iy : ix;
    const int nb = yd ? nx : ny, drop = skip >= 0 ? rdrop[row] : -1;
    if (skip >= 0) tot += line_kept<LF_F32>(img, nb, ny, yd, m, b0, fabs(inv), drop, 1, 0);
    if (!(fabs(tot) < INFINITY))
        tot = line_ray_again<LF_F32>(img, nb, ny, yd, m, b0, fabs(inv), yd ? r.z : r.x, min(yd ? r.w : r.y, yd ? ny : nx), drop, 1, 0);
    sino[row] = (float)(tot * rlen[row]);
}

// K interleaved values at pixel (i, j), or `pad` outside the image.
template <typename T, int K>
__device__ __forceinline__ void ldn(const UG<T> &U, const GL T *arr, int i, int j, T (&o)[K], T pad) {
    const int64_t q = U.at(i, j);
    if (q < 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) o[k] = pad;
    } else {
        loadk<T, K>(arr + q * K, o);
    }
}

// The back projection's 16 x 16 pixel square (rows i0 .. i0 + 15, columns
// j0 .. j0 + 15) and its one-pixel halo, 18 x 18 pixels of K values, for the
// regulariser of its epilogue: staged through LDS once instead of eight
// neighbour loads per pixel.
constexpr int kSqW = kBpBlockTC * kTileW + 2, kSqN = kSqW * kSqW;
static_assert(kBpBlockTR * kTileH == kBpBlockTC * kTileW, "the back-projection block is square");
__device__ __forceinline__ int sq_at(int r, int c) { return (r + 1) * kSqW + c + 1; }

// L[sq_at(r, c) * K + k] = arr at (i0 + r, j0 + c), `pad` outside the image.
// Thread (w, lane) stages pixel (tile row w, tile column lane / 32, tile
// position lane % 32) of the square; threads 0 .. 67 the halo.
template <typename T, int K>
__device__ __forceinline__ void put_square(const UG<T> &U, const GL T *arr, int i0, int j0, T pad, LDSP T *L) {
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave, w = lane & 31;
    const int r = wv * kTileH + ((w >> 2) & 3), c = (lane >> 5) * kTileW + ((w >> 4) << 2) + (w & 3);
    T x[K];
    ldn<T, K>(U, arr, i0 + r, j0 + c, x, pad);
#pragma unroll
    for (int k = 0; k < K; ++k) L[sq_at(r, c) * K + k] = x[k];
    constexpr int E = kSqW - 2, kHalo = 2 * kSqW + 2 * E;   // 68
    if (threadIdx.x < kHalo) {
        const int e = threadIdx.x;
        const int hr = e < kSqW ? -1 : (e < 2 * kSqW ? E : (e - 2 * kSqW) % E);
        const int hc = e < 2 * kSqW ? e % kSqW - 1 : (e < 2 * kSqW + E ? -1 : E);
        ldn<T, K>(U, arr, i0 + hr, j0 + hc, x, pad);
#pragma unroll
        for (int k = 0; k < K; ++k) L[sq_at(hr, hc) * K + k] = x[k];
    }
}
// The same; every thread calls it; ends with a barrier.
template <typename T, int K>
__device__ __forceinline__ void stage_square(const UG<T> &U, const GL T *arr, int i0, int j0, T pad, LDSP T *L) {
    put_square<T, K>(U, arr, i0, j0, pad, L);
    __syncthreads();
}

// The same square as stage_square, in the same layout, moved by direct
// global-to-LDS loads (positions outside the image get `pad` by LDS stores).
// Nothing waits here: the caller waits for every load (s_waitcnt 0) and
// synchronises the block before reading L.
template <typename T, int K>
__device__ __forceinline__ void dma_square(const UG<T> &U, const GL T *arr, int i0, int j0, T pad, LDSP T *L) {
    constexpr int DW = (int)(sizeof(T) / 4), PD = K * DW, N = kSqN * PD;   // dwords per pixel, per square
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    uint32_t pw[DW];
    __builtin_memcpy(pw, &pad, sizeof(T));
    const GL uint32_t *src = (const GL uint32_t *)arr;
    LDSP uint32_t *dst = (LDSP uint32_t *)L;
    for (int b = wv * kWave; b < N; b += kBlock) {
        const int t = b + lane;
        if (t < N) {
            const int p = t / PD, e = t - p * PD;
            const int i = i0 + p / kSqW - 1, j = j0 + p % kSqW - 1;
            if (i >= 0 && j >= 0 && i < U.nx && j < U.ny)
                __builtin_amdgcn_global_load_lds((const GL void *)(src + tile_index(i, j, U.tny) * PD + e),
                                                 (LDSP void *)(dst + b), 4, 0, 0);
            else
                dst[t] = (DW == 1 || (e & 1) == 0) ? pw[0] : pw[DW - 1];
        }
    }
}

// GoldenC image-gradient regulariser of K interleaved jobs at square pixel
// (r, c): u zero padded, v one padded (origin/GoldenC/src/main.c:112-125).
template <typename T, int K>
__device__ __forceinline__ void gc_reg(const LDSP T *Lu, const LDSP T *Lv, int r, int c, const double (&eps)[K],
                                       double (&out)[K]) {
    const LDSP T *u = Lu + sq_at(r, c) * K, *v = Lv + sq_at(r, c) * K;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const double Z = u[k], Zd = u[kSqW * K + k], Zr = u[K + k], Zu = u[-kSqW * K + k], Zl = u[-K + k];
        const double Pp = v[k], Pu = v[-kSqW * K + k], Pl = v[-K + k];
        out[k] = +(Pp * Pp) * (Zd - Z) + (Pp * Pp) * (Zr - Z) - (Pu * Pu) * (Z - Zu) - (Pl * Pl) * (Z - Zl) +
                 0.01 * (eps[k] * eps[k]) * (Zd + Zr - 4 * Z + Zu + Zl);
    }
}

// Gather back projection of subset s over 4 slices of tiled pixels, fused
// with d = S * A_s^T r + alpha * R(u, v); partial sum d^2.
// Back projection of subset s over one 16 x 16 block of pixels (bp_item;
// wave w holds tile row w of the block).  LDS: the block first copies the
// residual values of every (view, bin) its entries use into `ldr` (slots of
// the block's table, `vlo` / `voff`), then gathers from there.
template <typename T, int K, bool LDS, bool SQ>
__device__ __forceinline__ void bp_unit(const EngArgs<T> &a, const UG<T> &U, int s, int lb, double *lds,
                                        LDSP T *ldr, int sq_off) {
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    const int64_t sl0 = U.bs_slice0[s], li = (int64_t)lb * (kBlock / kWave) + wv, sl = sl0 + li;
    const bool has = li < U.bs_slice0[s + 1] - sl0;
    const int tnx = (U.nx + kTileH - 1) / kTileH;
    const int nbc = (U.tny + kBpBlockTC - 1) / kBpBlockTC;
    const int i0 = (lb / nbc) * (kBpBlockTR * kTileH), j0 = (lb % nbc) * (kBpBlockTC * kTileW);
    double m[K];
#pragma unroll
    for (int j = 0; j < K; ++j) m[j] = 0.0;
    // u and v of the square for the regulariser: with SQ in their own LDS
    // region at sq_off, loaded now, behind the walk; otherwise after the
    // walk, in the LDS the residual slots used.
    LDSP T *Lu = ldr + (SQ ? sq_off : 0), *Lv = Lu + kSqN * K;
    if constexpr (SQ) {
        dma_square<T, K>(U, U.u, i0, j0, T(0), Lu);
        dma_square<T, K>(U, U.v, i0, j0, T(1), Lv);
    }
    Stage<T, K> st;
    int64_t p0 = 0;
    int n = 0;
    if (LDS) {
        if (has) {
            p0 = sell_pos(U.bs_base[sl], 0, lane);
            n = U.bs_T[sl];
        }
        const int nv = (int)((U.sub_row0[s + 1] - U.sub_row0[s]) / U.nbins);
        const int64_t nblk = bp_blocks_of(tnx, U.tny);
        const GL int32_t *vlo = U.bs_vlo + U.bs_vtab0[s] + (int64_t)lb * nv;
        // the same offsets as voff_at (runtime.hpp)
        const GL int32_t *voff = U.bs_voff + (U.bs_vtab0[s] + (int64_t)s * nblk + (int64_t)lb * (nv + 1));
        // Wave w copies views w, w + 4, ...: a view's slots are c consecutive
        // residual rows (K values each), so the copy is one contiguous run of
        // dwords, moved by direct global-to-LDS loads (no register round
        // trip; every load of the block in flight until the one wait).
        // The views' slot offsets and first rows are read 64 views at a time,
        // one view per lane, and taken from the lanes in turn, so that no
        // load waits between the direct loads.
        constexpr int NW = kBlock / kWave, DW = (int)(sizeof(T) / 4) * K;
        for (int vb = wv; vb < nv; vb += NW * kWave) {
            const int vl = vb + NW * lane;
            int o_l = 0, c_l = 0, row_l = 0;   // row within the subset's residual rows
            if (vl < nv) {
                o_l = voff[vl];
                c_l = voff[vl + 1] - o_l;
                row_l = vl * U.nbins + vlo[vl];
            }
            const int nb = min(kWave, (nv - vb + NW - 1) / NW);
            const GL uint32_t *r0 = (const GL uint32_t *)(U.r + U.sub_row0[s] * K);
            for (int i = 0; i < nb; ++i) {
                const int o = __builtin_amdgcn_readlane(o_l, i), nd = __builtin_amdgcn_readlane(c_l, i) * DW;
                const GL uint32_t *src = r0 + (int64_t)__builtin_amdgcn_readlane(row_l, i) * DW;
                LDSP uint32_t *dst = (LDSP uint32_t *)(ldr + (int64_t)o * K);
                for (int e0 = 0; e0 < nd; e0 += kWave)
                    if (e0 + lane < nd)
                        __builtin_amdgcn_global_load_lds((const GL void *)(src + e0 + lane), (LDSP void *)(dst + e0), 4,
                                                         0, 0);
            }
        }
        // The walk's first stream loads go out with the copies, so that the
        // one wait covers both.
        if (has && (MI_BP_PRIME == 2 || (MI_BP_PRIME == 1 && K == 1)))
            walk_prime<T, K, MI_NT_BP, IM_SLOT16>(st, nullptr, (const GL int16_t *)(U.bs_slot16 + p0),
                                                  U.bs_len + p0, n);
        __builtin_amdgcn_s_waitcnt(0);   // the block's direct loads have landed in LDS
        __syncthreads();
    }
    double tot[K];
#pragma unroll
    for (int j = 0; j < K; ++j) tot[j] = 0.0;
    if (has) {
        Acc<T> acc[K];
        if (LDS) {
            if (MI_BP_PRIME == 2 || (MI_BP_PRIME == 1 && K == 1))
                walk<T, K, MI_NT_BP, IM_SLOT16, true, true>(nullptr, (const GL int16_t *)(U.bs_slot16 + p0), 0u,
                                                            U.bs_len + p0, n, U.r, 0u, acc, st, ldr);
            else
                walk<T, K, MI_NT_BP, IM_SLOT16, true, false>(nullptr, (const GL int16_t *)(U.bs_slot16 + p0), 0u,
                                                             U.bs_len + p0, n, U.r, 0u, acc, st, ldr);
        } else {
            walk_slice<T, K, MI_NT_BP>(U.bs_base, U.bs_T, U.bs_idx, U.bs_first, U.bs_d16, U.bs_len, sl, lane, U.r,
                                       U.nrows, acc);
        }
#pragma unroll
        for (int j = 0; j < K; ++j) tot[j] = acc[j].value();
    }
    if constexpr (!SQ) {
        __syncthreads();   // every wave has finished its walk
        stage_square<T, K>(U, U.u, i0, j0, T(0), Lu);
        stage_square<T, K>(U, U.v, i0, j0, T(1), Lv);
    } else if constexpr (!LDS) {
        __builtin_amdgcn_s_waitcnt(0);   // the squares' direct loads
        __syncthreads();
    }
    if (has) {
        const int64_t q = bp_item(lb, wv, lane, tnx, U.tny);
        if (q >= 0) {
            int i, j;
            tile_coords(q, U.tny, i, j);
            T dv[K];
            if (i < U.nx && j < U.ny) {
                double eps[K], reg[K];
#pragma unroll
                for (int k = 0; k < K; ++k) eps[k] = jpar(a, U.job0 + k).eps;
                gc_reg<T, K>(Lu, Lv, i - i0, j - j0, eps, reg);
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const double d = (double)a.S * tot[k] + jpar(a, U.job0 + k).alpha * reg[k];
                    dv[k] = (T)d;
                    m[k] = (double)dv[k] * (double)dv[k];
                }
            } else {
                zerok<T, K>(dv);
            }
            storek<T, K>(U.d + q * K, dv);
        }
    }
    block_store<T, K, false>(a, U, SL_DD, lb, m, lds);
}

// Back projection along the lines (Lines, runtime.hpp), FP32: a lane is a
// pixel, a workgroup its 16 x 16 block as in bp_unit.  No matrix is read.  Per
// view the pixel's position on the detector (float) gives the few
// bins whose rays can meet it, a superset; for each the exact length follows
// from the ray's line in double,
//   min(1, max(0, ((1 + |m|) / 2 - |b0 + m a - j - 1/2|) / |m|)),
// times the residual, which holds the ray's length per line.  Weight, product
// and sum are double; 1 / |m| is rounded to FP32, once, as a stored length is (as
// a double it costs 8 more bytes of LDS a slot).  A sum that is not finite is taken again over the rays
// that cross the pixel (line_bp_again).
//
// A block's views come in windows of 64, sorted by axis and by candidates
// (LineView, prepared with the geometry).  As many views as half of the
// launch's LDS slots hold, and their rays, are copied there by direct
// global-to-LDS loads, which run while the lanes work on the other half's
// views.
// Where the image has few blocks, 2 or 4 groups of 256 lanes share a block's
// views (view by view in turn) and their sums are added in order.  The order
// of a pixel's sum depends on the geometry only, not on K or on the LDS slots.
//
// What bounds it: VALU at K = 1, some 32 instructions a view and pixel, half of
// them on doubles at half rate (a quarter of the
// issue slots go to LDS latency at four waves a SIMD), LDS reads at K = 4 (36
// bytes a candidate).  512 x 512 pixels, 60
// views: 40.1 us, against 35.4 of the staged matrix form (bp_unit, 179 MB a
// launch) and 37.6 with weights and a view's products in FP32.
// It needs no matrix at all: an 874 x 874 slice of 576 views is ready in 2 ms
// (95 ms with the matrix), in 0.2 GB instead of 4.
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
static_assert(sizeof(LineView) == 2 * sizeof(i32x4), "a view is two 16-byte loads");

// Position on the detector of a pixel in units of bins, less bin0.  Flat:
// (Xk, Yk) = (X, Y) / k and sodk = sod / k.  Arc: X, Y, sod, and the arc
// tangent of Abramowitz & Stegun 4.4.47 (within 1.2e-5).
__device__ __forceinline__ float line_bin_flat(float X, float Y, float Xk, float Yk, float c, float s, float sodk) {
    const float D = __builtin_fmaf(c, Yk, __builtin_fmaf(-s, Xk, sodk));
    return __builtin_fmaf(s, Y, c * X) * __builtin_amdgcn_rcpf(D);
}
__device__ __forceinline__ float line_bin_arc(float X, float Y, float c, float s, float sod, float k) {
    const float q = __builtin_fmaf(c, Y, -s * X), e = __builtin_fmaf(-s, Y, __builtin_fmaf(-c, X, sod));
    const float t = q * __builtin_amdgcn_rcpf(e), y = t * t;
    const float f = __builtin_fmaf(
        y, __builtin_fmaf(y, __builtin_fmaf(y, __builtin_fmaf(y, .0208351f, -.0851330f), .1801410f), -.3302995f),
        .9998660f);
    return -k * t * f;
}

// One half of the LDS slots: each array holds `cap` of them.
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
template <int K>
struct LineHalf {
    const LDSP f64x2 *mb;    // m, b0
    const LDSP float *inv;   // 1 / |m|
    const LDSP float *r;     // K residuals
    const LDSP int32_t *drop;
};
constexpr int line_slot_bytes(int K) { return 16 + 4 + 4 * K + 4; }

// What a lane's pixel brings.
struct LinePix {
    float X, Y, Xk, Yk, sodk, sod, k;
    int id;                  // x ny + y
};
__device__ __forceinline__ LinePix line_pix(const UG<float> &U, int i, int j) {
    LinePix p;
    p.X = (i + 0.5f - 0.5f * U.nx) * U.ln_pix;
    p.Y = (j + 0.5f - 0.5f * U.ny) * U.ln_pix;
    p.k = U.ln_k;
    p.sod = U.ln_sod;
    p.Xk = p.X / p.k;
    p.Yk = p.Y / p.k;
    p.sodk = p.sod / p.k;
    p.id = i * U.ny + j;
    return p;
}

// The ray's share of pixel b - 1/2 of line a.
__device__ __forceinline__ double line_weight(double m, double b0, float inv, double a, double b) {
    const double D = __builtin_fma(m, a, b0) - b;
    return fmin(fmax((__builtin_fma(fabs(m), 0.5, 0.5) - fabs(D)) * (double)inv, 0.0), 1.0);
}

// C candidates of one view (0: `cand` of them, two at a time) added to tot;
// slot: the first one's, in the half.
template <int K, bool EDGE, int C>
__device__ __forceinline__ void line_bp_view(const LineHalf<K> &h, uint32_t slot, int cand, int id, double a, double b,
                                             double (&tot)[K]) {
    constexpr int CC = C ? C : 2;
    for (int q = 0; q < (C ? C : cand); q += CC, slot += CC) {
        double t[CC];
#pragma unroll
        for (int n = 0; n < CC; ++n) {
            const f64x2 mb = h.mb[slot + n];
            t[n] = line_weight(mb.x, mb.y, h.inv[slot + n], a, b);
            if (EDGE) t[n] = h.drop[slot + n] == id ? 0.0 : t[n];
        }
        const LDSP float *r = h.r + slot * K;
#pragma unroll
        for (int k = 0; k < K; ++k)
#pragma unroll
            for (int n = 0; n < CC; ++n) tot[k] = __builtin_fma(t[n], (double)r[n * K + k], tot[k]);
    }
}

// This group's views k, k + P, ... below k1 of a half, all of one class.  The
// next view's numbers are read (one address for the wave) while this one's
// rays are.  off0: the half's first slot in the window.
template <int K, bool ARC, bool EDGE, int C>
__device__ __forceinline__ void line_bp_run(const LDSP unsigned char *views, int k, int k1, int P, const LineHalf<K> &h,
                                            float off0, const LinePix &p, double a, double b, double (&tot)[K]) {
    auto get = [&](int n, f32x4 &w, float &end, int &meta) {
        const LDSP unsigned char *v = views + n * (int)sizeof(LineView);
        w = *(const LDSP f32x4 *)v;   // c, s, lob, first
        end = *(const LDSP float *)(v + 16);
        if constexpr (C == 0) meta = *(const LDSP int *)(v + 20);
    };
    f32x4 w, nw;
    float end, nend;
    int meta = 0, nmeta = 0;
    get(k, w, end, meta);
    while (k < k1) {
        k += P;
        get(k < k1 ? k : k - P, nw, nend, nmeta);
        const float u = ARC ? line_bin_arc(p.X, p.Y, w.x, w.y, p.sod, p.k)
                            : line_bin_flat(p.X, p.Y, p.Xk, p.Yk, w.x, w.y, p.sodk);
        const uint32_t slot = (uint32_t)(__builtin_amdgcn_fmed3f(u + w.z, w.w, end) - off0);
        line_bp_view<K, EDGE, C>(h, slot, C ? C : __builtin_amdgcn_readfirstlane(line_cand(meta)), p.id, a, b, tot);
        w = nw;
        end = nend;
        meta = nmeta;
    }
}

// Job k's sum of one pixel again, straight from memory, over the rays that
// cross the pixel: where it is not finite a residual beside the pixel may not
// be (0 times it is not 0).  tab: the block's first window, windows `step`
// table entries apart.
template <bool ARC>
__device__ __forceinline__ double line_bp_again(const UG<float> &U, const GL char *tab, int64_t step, int s, int i, int j,
                                                int K, int k) {
    const LinePix p = line_pix(U, i, j);
    const int64_t row0 = U.sub_row0[s];
    const int nv = (int)((U.sub_row0[s + 1] - row0) / U.nbins);
    const double x = i, y = j;
    double tot = 0.0;
    for (int v = 0; v < nv; ++v) {
        const GL LineView &w = ((const GL LineView *)tab)[v / kLineViews * step + v % kLineViews];
        const float u = ARC ? line_bin_arc(p.X, p.Y, w.c, w.s, p.sod, p.k)
                            : line_bin_flat(p.X, p.Y, p.Xk, p.Yk, w.c, w.s, p.sodk);
        const int slot = (int)__builtin_amdgcn_fmed3f(u + w.lob, w.first, w.end);
        const bool yd = line_axis(w.meta);
        for (int n = slot; n < slot + line_cand(w.meta); ++n) {
            const int64_t e = w.src + n, row = row0 + w.row + n;
            const GL double *mb = (yd ? U.ln_my : U.ln_mx) + 2 * e;
            const double t = line_weight(mb[0], mb[1], (yd ? U.ln_iy : U.ln_ix)[e], yd ? y : x, (yd ? x : y) + 0.5);
            if (t > 1e-6 && U.ln_drop[row] != p.id) tot += t * (double)U.r[row * K + k];
        }
    }
    return tot;
}

// d = S A_s^T r + alpha R(u, v) for the block's pixels; partial sum d^2.
// P groups of 256 lanes; cap: slots of one half.
template <int K, int P>
__device__ __forceinline__ void line_bp_unit(const EngArgs<float> &a, const UG<float> &U, const UnitDesc<float> *unit, int s, int lb,
                                             int cap,
                                             double *lds, LDSP unsigned char *raw) {
    const int lane = threadIdx.x & (kWave - 1), wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int grp = wv / (kBlock / kWave);   // this wave's group
    const int tnx = (U.nx + kTileH - 1) / kTileH, nbc = (U.tny + kBpBlockTC - 1) / kBpBlockTC;
    const int i0 = (lb / nbc) * (kBpBlockTR * kTileH), j0 = (lb % nbc) * (kBpBlockTC * kTileW);
    const int64_t q = bp_item(lb, wv % (kBlock / kWave), lane, tnx, U.tny);
    int i = U.nx, j = U.ny;
    if (q >= 0) tile_coords(q, U.tny, i, j);
    const bool real = i < U.nx && j < U.ny;
    // LDS: two halves (each views, mb, inv, r, drop), used again behind the views
    constexpr int VB = kLineViews * (int)sizeof(LineView);
    const int half = VB + cap * line_slot_bytes(K);
    double tot[K];
#pragma unroll
    for (int k = 0; k < K; ++k) tot[k] = 0.0;
    const int64_t row0 = U.sub_row0[s];
    const int nv = (int)((U.sub_row0[s + 1] - row0) / U.nbins);
    const int64_t nblk = bp_blocks_of(tnx, U.tny);
    if (j0 < U.ny) {   // else: only padding of the tile rows
        const LinePix p = line_pix(U, i, j);
        const double id = i, jd = j;
        const int nwin = (nv + kLineViews - 1) / kLineViews;
        const bool edge = i0 == 0 || j0 == 0 || i0 + 16 >= U.nx || j0 + 16 >= U.ny;

        // A window: lane l holds view l (its second half: end, meta, src, row;
        // and first), and the views up to the end of each class.
        struct Window {
            const GL char *tab;   // its views
            i32x4 b;
            float first;
            int n;
        };
        auto load = [&](int w) {
            Window W;
            W.tab = (const GL char *)U.ln_views + ((U.ln_win0[s] + w) * nblk + lb) * (U.ln_vstride * (int64_t)sizeof(LineView));
            W.n = min(kLineViews, nv - w * kLineViews);
            W.b = i32x4{0, 0, 0, 0};
            W.first = 0.0f;
            if (lane < W.n) {
                W.b = *(const GL i32x4 *)(W.tab + lane * sizeof(LineView) + 16);
                W.first = *(const GL float *)(W.tab + lane * sizeof(LineView) + 12);
            }
            return W;
        };
        auto fit = [&](const Window &W, int off) {   // as many views as a half holds (the slots' ends only grow)
            return (int)__popcll(__ballot(lane < W.n && line_stop(W.b.y) - off <= cap));
        };
        // copies views k0 .. k1 - 1 of a window and their rays to a half
        auto copy = [&](const Window &W, int k0, int k1, int off0, LDSP unsigned char *to) {
            if (wv == 0)
                for (int e = lane; e < (k1 - k0) * 2; e += kWave)
                    __builtin_amdgcn_global_load_lds((const GL void *)(W.tab + k0 * sizeof(LineView) + e * 16u),
                                                     (LDSP void *)(to + (e - lane) * 16), 16, 0, 0);
            to += VB;
            for (int k = k0 + wv; k < k1; k += P * (kBlock / kWave)) {
                const int first = (int)__uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(W.first), k));
                const int meta = __builtin_amdgcn_readlane(W.b.y, k);
                const int n = line_stop(meta) - first, at = first - off0;
                const int64_t src = __builtin_amdgcn_readlane(W.b.z, k) + first;
                const int64_t row = row0 + __builtin_amdgcn_readlane(W.b.w, k) + first;
                const bool yd = line_axis(meta);
                const GL char *mb = (const GL char *)(yd ? U.ln_my : U.ln_mx) + src * 16;
                const GL char *iv = (const GL char *)(yd ? U.ln_iy : U.ln_ix) + src * 4;
                const GL char *rr = (const GL char *)U.r + row * (4 * K), *dr = (const GL char *)U.ln_drop + row * 4;
                LDSP unsigned char *o = to + at * 16;
                for (int e = lane; e < n; e += kWave)
                    __builtin_amdgcn_global_load_lds((const GL void *)(mb + e * 16u), (LDSP void *)(o + (e - lane) * 16), 16,
                                                     0, 0);
                o = to + cap * 16 + at * 4;
                for (int e = lane; e < n; e += kWave)
                    __builtin_amdgcn_global_load_lds((const GL void *)(iv + e * 4u), (LDSP void *)(o + (e - lane) * 4), 4, 0,
                                                     0);
                o = to + cap * 20 + at * (4 * K);
                for (int e = lane; e < n * K; e += kWave)
                    __builtin_amdgcn_global_load_lds((const GL void *)(rr + e * 4u), (LDSP void *)(o + (e - lane) * 4), 4, 0,
                                                     0);
                if (edge) {
                    o = to + cap * (20 + 4 * K) + at * 4;
                    for (int e = lane; e < n; e += kWave)
                        __builtin_amdgcn_global_load_lds((const GL void *)(dr + e * 4u), (LDSP void *)(o + (e - lane) * 4),
                                                         4, 0, 0);
                }
            }
        };
        // The round at hand: views k0 .. k1 - 1 of window w, slots from off0;
        // W: the window of the round behind it, N: the window behind W.
        int w = 0, k0 = 0, off0 = 0, par = 0;
        Window W = load(0), N = load(nwin > 1 ? 1 : 0);
        int k1 = fit(W, 0);
        copy(W, k0, k1, off0, raw);
        while (w < nwin) {
            // the classes of this round's views: along x with 2, 3, more candidates, along y likewise
            int upto[6];
            const int cls = line_class(W.b.y);
#pragma unroll
            for (int c = 0; c < 6; ++c)
                upto[c] = min(k1, (int)__popcll(__ballot(lane < W.n && cls <= c)));
            int nw = w, nk0 = k1, noff = line_stop(__builtin_amdgcn_readlane(W.b.y, k1 - 1)), nk1 = 0;
            if (nk0 >= W.n) {
                ++nw;
                nk0 = noff = 0;
                W = N;
                if (nw + 1 < nwin) N = load(nw + 1);
            }
            if (nw < nwin) nk1 = fit(W, noff);
            __builtin_amdgcn_s_waitcnt(0);   // this round's copies have landed
            __syncthreads();                 // ... everybody's, and the other half is free
            if (nw < nwin) copy(W, nk0, nk1, noff, raw + (par ^ 1) * half);
            const LDSP unsigned char *vt = raw + par * half, *b = vt + VB;
            vt -= k0 * (int)sizeof(LineView);
            const LineHalf<K> h{(const LDSP f64x2 *)b, (const LDSP float *)(b + cap * 16),
                                (const LDSP float *)(b + cap * 20), (const LDSP int32_t *)(b + cap * (20 + 4 * K))};
            auto run = [&](auto arc, auto ed) {
                auto one = [&](auto c, int e) {
                    constexpr int C = decltype(c)::value;
                    const int c0 = max(k0, e ? upto[e - 1] : 0);
                    const int k = c0 + (grp - c0 % P + P) % P;   // the window's views go to the groups in turn
                    if (k < upto[e])
                        line_bp_run<K, decltype(arc)::value, decltype(ed)::value, C>(
                            vt, k, upto[e], P, h, (float)off0, p, e < 3 ? id : jd, (e < 3 ? jd : id) + 0.5, tot);
                };
                using std::integral_constant;
#pragma unroll
                for (int e = 0; e < 6; e += 3) {
                    one(integral_constant<int, 2>{}, e);
                    one(integral_constant<int, 3>{}, e + 1);
                    one(integral_constant<int, 0>{}, e + 2);
                }
            };
            if (U.ln_arc) {
                if (edge) run(std::true_type{}, std::true_type{});
                else run(std::true_type{}, std::false_type{});
            } else {
                if (edge) run(std::false_type{}, std::true_type{});
                else run(std::false_type{}, std::false_type{});
            }
            w = nw;
            k0 = nk0;
            k1 = nk1;
            off0 = noff;
            par ^= 1;
        }
        __syncthreads();   // the slots' LDS is used again
    }
    if constexpr (P > 1) {   // the groups' sums, in order
        LDSP double *part = (LDSP double *)raw;
        if (grp > 0)
#pragma unroll
            for (int k = 0; k < K; ++k) part[((grp - 1) * K + k) * kBlock + threadIdx.x % kBlock] = tot[k];
        __syncthreads();
        if (grp == 0)
#pragma unroll
            for (int g = 1; g < P; ++g)
#pragma unroll
                for (int k = 0; k < K; ++k) tot[k] += part[((g - 1) * K + k) * kBlock + threadIdx.x];
        __syncthreads();
    }
    // The unit's numbers again: kept over the views, they would not fit the
    // scalar registers (512 x 512, 60 views, one job: 41.7 us, so 39.4; 874 x
    // 874, 72 views 112 and 102).
    uint64_t at = (uint64_t)unit;
    asm volatile("" : "+s"(at));
    const UG<float> V(*(const __attribute__((address_space(4))) UnitDesc<float> *)at);
    if (grp == 0 && real)
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (!(fabs(tot[k]) < INFINITY)) {
                const GL char *tab =
                    (const GL char *)V.ln_views + (V.ln_win0[s] * nblk + lb) * (V.ln_vstride * (int64_t)sizeof(LineView));
                tot[k] = V.ln_arc ? line_bp_again<true>(V, tab, nblk * V.ln_vstride, s, i, j, K, k)
                                  : line_bp_again<false>(V, tab, nblk * V.ln_vstride, s, i, j, K, k);
            }
    LDSP float *Lu = (LDSP float *)raw, *Lv = Lu + kSqN * K;
    if (grp == 0) {
        put_square<float, K>(V, V.u, i0, j0, 0.0f, Lu);
        put_square<float, K>(V, V.v, i0, j0, 1.0f, Lv);
    }
    __syncthreads();
    double m[K];
#pragma unroll
    for (int k = 0; k < K; ++k) m[k] = 0.0;
    if (grp == 0 && q >= 0) {
        float dv[K], dl[K];
        zerok<float, K>(dv);
        zerok<float, K>(dl);
        if (real) {
            double eps[K], reg[K];
#pragma unroll
            for (int k = 0; k < K; ++k) eps[k] = jpar(a, V.job0 + k).eps;
            gc_reg<float, K>(Lu, Lv, i - i0, j - j0, eps, reg);
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const double d = (double)a.S * tot[k] + jpar(a, V.job0 + k).alpha * reg[k];
                dv[k] = (float)d;
                dl[k] = (float)(d - (double)dv[k]);
                m[k] = (double)dv[k] * (double)dv[k];
            }
            put_proj_d<float, K>(V, i, j, dv);
        }
        storek<float, K>(V.d + q * K, dv);
        storek<float, K>(V.dl + q * K, dl);
    }
    block_store<float, K, false>(a, V, SL_DD, lb, m, lds);
}

// Stencil kernels: one thread per tiled position q (256 per block); the
// padding positions of the tiles do no work.

// Stencil strips.  Tile rows hold a multiple of kStripTiles tiles, so the 256
// tiled positions of stencil block lb are the 4 x 64 pixels of one strip
// (rows i0 .. i0 + 3, columns j0 .. j0 + 63).  A stencil stages the strip of
// each array it reads around, with a one-pixel halo (6 x 66 pixels, K values
// each), through LDS once, and reads the neighbours from there.
constexpr int kStripW = kStripTiles * kTileW, kHaloW = kStripW + 2, kHaloN = (kTileH + 2) * kHaloW;
static_assert(kPixBlock == kStripTiles * kTileH * kTileW, "a stencil block is one strip");

struct Strip {
    int64_t q;        // this thread's tiled position
    int i0, j0;       // strip origin
    int li, lj;       // this thread's pixel, relative to the origin
    bool real;        // the pixel lies in the image
};
template <typename T>
__device__ __forceinline__ Strip strip_of(const UG<T> &U, int lb) {
    const int t0 = lb * kStripTiles;
    Strip s;
    s.q = (int64_t)lb * kPixBlock + threadIdx.x;
    s.i0 = (t0 / U.tny) * kTileH;
    s.j0 = (t0 % U.tny) * kTileW;
    int i, j;
    tile_coords(s.q, U.tny, i, j);
    s.li = i - s.i0;
    s.lj = j - s.j0;
    s.real = i < U.nx && j < U.ny;
    return s;
}
__device__ __forceinline__ int halo_at(int li, int lj) { return (li + 1) * kHaloW + lj + 1; }

// L[halo_at(r, c) * K + k] = arr at pixel (i0 + r, j0 + c) for the strip and
// its halo, `pad` outside the image.  Every thread calls it; ends with a
// barrier.
template <typename T, int K>
__device__ __forceinline__ void stage_strip(const UG<T> &U, const GL T *arr, const Strip &s, T pad, T *L) {
    T x[K];
    if (s.real) {
        loadk<T, K>(arr + s.q * K, x);
    } else {
#pragma unroll
        for (int k = 0; k < K; ++k) x[k] = pad;
    }
#pragma unroll
    for (int k = 0; k < K; ++k) L[halo_at(s.li, s.lj) * K + k] = x[k];
    // the halo: rows -1 and 4 (66 pixels each, corners included), columns
    // -1 and 64 of rows 0 .. 3
    constexpr int kHalo = 2 * kHaloW + 2 * kTileH;
    static_assert(kHalo <= kBlock, "one halo pixel per thread");
    if (threadIdx.x < kHalo) {
        const int e = threadIdx.x, f = e - 2 * kHaloW;
        const int li = e < 2 * kHaloW ? (e < kHaloW ? -1 : kTileH) : f % kTileH;
        const int lj = e < 2 * kHaloW ? e % kHaloW - 1 : (f < kTileH ? -1 : kStripW);
        ldn<T, K>(U, arr, s.i0 + li, s.j0 + lj, x, pad);
#pragma unroll
        for (int k = 0; k < K; ++k) L[halo_at(li, lj) * K + k] = x[k];
    }
    __syncthreads();
}

// The staged values at offset (di, dj) from this thread's pixel.
template <typename T, int K>
__device__ __forceinline__ void ldl(const T *L, const Strip &s, int di, int dj, T (&o)[K]) {
    const T *p = L + halo_at(s.li + di, s.lj + dj) * K;
#pragma unroll
    for (int k = 0; k < K; ++k) o[k] = p[k];
}

// nV(d) = sum (v^2 + 0.01 eps^2)((d - d_up)^2 + (d - d_left)^2), d zero
// padded (origin/GoldenC/src/main.c:152-158).
template <typename T, int K>
__device__ __forceinline__ void nv_unit(const EngArgs<T> &a, const UG<T> &U, int lb, double *lds, T *L) {
    const Strip st = strip_of(U, lb);
    stage_strip<T, K>(U, U.d, st, T(0), L);
    double m[K];
#pragma unroll
    for (int j = 0; j < K; ++j) m[j] = 0.0;
    if (st.real) {
        T dq[K], du[K], dl[K], vv[K];
        ldl<T, K>(L, st, 0, 0, dq);
        ldl<T, K>(L, st, -1, 0, du);
        ldl<T, K>(L, st, 0, -1, dl);
        loadk<T, K>(U.v + st.q * K, vv);
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const double eps = jpar(a, U.job0 + j).eps;
            const double e2 = 0.01 * (eps * eps);
            const double z = (double)dq[j];
            const double A = z - (double)du[j], B = z - (double)dl[j];
            const double w = (double)vv[j];
            m[j] = (w * w + e2) * (A * A + B * B);
        }
    }
    block_store<T, K, false>(a, U, SL_NV, lb, m, lds);
}

__device__ __forceinline__ bool real_pixel(int64_t q, int64_t npix_t, int tny, int nx, int ny, int &i, int &j) {
    if (q >= npix_t) return false;
    tile_coords(q, tny, i, j);
    return i < nx && j < ny;
}

// u = clamp(u + c d, lower, upper) for live jobs.
//
// Units with lines keep what the rounding of u and d to FP32 leaves over (ul;
// dl until here), and project u with its remainder: the iteration hardly damps an image's finest structure, so the roundings
// of its updates add up, and on one input in ten the exact line search makes any
// difference grow 1.5 to 2 times a pass, most of all that of a rounded u in its
// projections.  512 x 512 pixels, 720 views, 12 subsets, 20 passes, 48 inputs:
// error of u against 64 bits 2.8e-7 to 2.4e-6 with u rounded at every step, 2.5e-8
// to 9.1e-8 so (the result's own rounding is 2.5e-8).
template <typename T, int K>
__device__ __forceinline__ void axpy_unit(const EngArgs<T> &a, const UG<T> &U, int lb) {
    const int64_t q = (int64_t)lb * kPixBlock + threadIdx.x;
    int i, j;
    if (!real_pixel(q, U.npix_t, U.tny, U.nx, U.ny, i, j)) return;
    T uu[K], dd[K], ul[K], dl[K];
    loadk<T, K>(U.u + q * K, uu);
    loadk<T, K>(U.d + q * K, dd);
    zerok<T, K>(ul);
    zerok<T, K>(dl);
    if (U.ul) {
        loadk<T, K>(U.ul + q * K, ul);
        loadk<T, K>(U.dl + q * K, dl);
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int js = U.job0 + k;
        if (!job_live(a, js)) continue;
        const GL JobParams &P = jpar(a, js);
        double yn = ((double)uu[k] + (double)ul[k]) + jsc(a, js).c * ((double)dd[k] + (double)dl[k]);
        if (yn < P.lower) yn = P.lower;
        if (yn > P.upper) yn = P.upper;
        uu[k] = (T)yn;
        ul[k] = fabs((double)uu[k]) < INFINITY ? (T)(yn - (double)uu[k]) : T(0);
    }
    storek<T, K>(U.u + q * K, uu);
    if (!U.ul) return;
    storek<T, K>(U.ul + q * K, ul);
    put_proj_u<T, K>(U, i, j, uu, ul);
}

template <typename T>
__device__ __forceinline__ void cswap(T &x, T &y) {
    const T lo = x < y ? x : y, hi = x < y ? y : x;
    x = lo;
    y = hi;
}

template <typename T>
__device__ __forceinline__ bool median_due(const EngArgs<T> &a, int js) {
    const GL JobParams &P = jpar(a, js);
    return job_live(a, js) && P.median_every > 0 && (jsc(a, js).iters + 1) % P.median_every == 0;
}

// w = 3x3 median of u (zero padding, origin/GoldenC/src/main.c:366-390) for
// jobs whose median is due this pass, else w = u.
template <typename T, int K>
__device__ __forceinline__ void median_unit(const EngArgs<T> &a, const UG<T> &U, int lb, T *L) {
    const Strip st = strip_of(U, lb);
    stage_strip<T, K>(U, U.u, st, T(0), L);
    if (!st.real) return;
    const int64_t q = st.q;
    T nb[9][K];
    int n = 0;
#pragma unroll
    for (int di = -1; di <= 1; ++di)
#pragma unroll
        for (int dj = -1; dj <= 1; ++dj, ++n) ldl<T, K>(L, st, di, dj, nb[n]);
    T out[K];
#pragma unroll
    for (int j = 0; j < K; ++j) {
        if (!median_due(a, U.job0 + j)) {
            out[j] = nb[4][j];
            continue;
        }
        T t[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) t[k] = nb[k][j];
        // Paeth's 19-exchange median-of-9 network (exact selection).
        cswap(t[1], t[2]); cswap(t[4], t[5]); cswap(t[7], t[8]);
        cswap(t[0], t[1]); cswap(t[3], t[4]); cswap(t[6], t[7]);
        cswap(t[1], t[2]); cswap(t[4], t[5]); cswap(t[7], t[8]);
        cswap(t[0], t[3]); cswap(t[5], t[8]); cswap(t[4], t[7]);
        cswap(t[3], t[6]); cswap(t[1], t[4]); cswap(t[2], t[5]);
        cswap(t[4], t[7]); cswap(t[4], t[2]); cswap(t[6], t[4]);
        cswap(t[4], t[2]);
        out[j] = t[4];
    }
    storek<T, K>(U.w + q * K, out);
}

template <typename T, int K>
__device__ __forceinline__ void copy_wu_unit(const EngArgs<T> &a, const UG<T> &U, int lb) {
    const int64_t q = (int64_t)lb * kPixBlock + threadIdx.x;
    int i, j;
    if (!real_pixel(q, U.npix_t, U.tny, U.nx, U.ny, i, j)) return;
    T t[K];
    loadk<T, K>(U.w + q * K, t);
    storek<T, K>(U.u + q * K, t);
    if (U.ul) {   // a median is one of the FP32 values
        T ul[K];
        loadk<T, K>(U.ul + q * K, ul);
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (median_due(a, U.job0 + k)) ul[k] = T(0);
        storek<T, K>(U.ul + q * K, ul);
        put_proj_u<T, K>(U, i, j, t, ul);
    }
}

template <typename T>
__device__ __forceinline__ bool edge_live(const EngArgs<T> &a, int js, int it) {
    return job_live(a, js) && !jsc(a, js).edge_done && it < jpar(a, js).iter_edge;
}

// Edge step, origin/GoldenC/src/main.c:294-305: w = -grad_v, partials
// ||w||^2 and sum n w^2 (f = u zero padded, v one padded).
template <typename T, int K>
__device__ __forceinline__ void edge_grad_unit(const EngArgs<T> &a, const UG<T> &U, int lb, int it,
                                               double *lds, T *L) {
    const Strip st = strip_of(U, lb);
    T *Lu = L, *Lv = L + kHaloN * K;
    stage_strip<T, K>(U, U.u, st, T(0), Lu);
    stage_strip<T, K>(U, U.v, st, T(1), Lv);
    const int64_t q = st.q;
    double m0[K], m1[K];
#pragma unroll
    for (int j = 0; j < K; ++j) m0[j] = m1[j] = 0.0;
    if (st.real) {
        T fd[K], fu[K], fr[K], fl[K], vc[K], vd[K], vu[K], vr[K], vl[K];
        ldl<T, K>(Lu, st, 1, 0, fd);
        ldl<T, K>(Lu, st, -1, 0, fu);
        ldl<T, K>(Lu, st, 0, 1, fr);
        ldl<T, K>(Lu, st, 0, -1, fl);
        ldl<T, K>(Lv, st, 0, 0, vc);
        ldl<T, K>(Lv, st, 1, 0, vd);
        ldl<T, K>(Lv, st, -1, 0, vu);
        ldl<T, K>(Lv, st, 0, 1, vr);
        ldl<T, K>(Lv, st, 0, -1, vl);
        T out[K];
        zerok<T, K>(out);
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const int js = U.job0 + j;
            if (!edge_live(a, js, it)) continue;
            const GL JobParams &P = jpar(a, js);
            const double dxf = 0.5 * ((double)fd[j] - (double)fu[j]);
            const double dyf = 0.5 * ((double)fr[j] - (double)fl[j]);
            const double n = dxf * dxf + dyf * dyf;
            const double t = (double)vc[j];
            const double lap = 0.25 * ((double)vd[j] + (double)vr[j] - 4 * t + (double)vu[j] + (double)vl[j]);
            const double gr = P.alpha * t * n - P.beta * P.eps * lap + P.beta * (t - 1) / (4 * P.eps);
            const T dt = (T)(-gr);
            out[j] = dt;
            const double dd = (double)dt * (double)dt;
            m0[j] = dd;
            m1[j] = n * dd;
        }
        storek<T, K>(U.w + q * K, out);
    }
    block_store<T, K, false>(a, U, SL_E0, lb, m0, lds);
    __syncthreads();
    block_store<T, K, false>(a, U, SL_E1, lb, m1, lds);
}

// main.c:311-329: |central gradient of w|^2.
template <typename T, int K>
__device__ __forceinline__ void edge_nabla_unit(const EngArgs<T> &a, const UG<T> &U, int lb, int it,
                                                double *lds, T *L) {
    const Strip st = strip_of(U, lb);
    stage_strip<T, K>(U, U.w, st, T(0), L);
    double m[K];
#pragma unroll
    for (int j = 0; j < K; ++j) m[j] = 0.0;
    if (st.real) {
        T d1[K], d2[K], d3[K], d4[K];
        ldl<T, K>(L, st, 1, 0, d1);
        ldl<T, K>(L, st, -1, 0, d2);
        ldl<T, K>(L, st, 0, 1, d3);
        ldl<T, K>(L, st, 0, -1, d4);
#pragma unroll
        for (int j = 0; j < K; ++j) {
            if (!edge_live(a, U.job0 + j, it)) continue;
            const double A = 0.5 * ((double)d1[j] - (double)d2[j]);
            const double B = 0.5 * ((double)d3[j] - (double)d4[j]);
            m[j] = A * A + B * B;
        }
    }
    block_store<T, K, false>(a, U, SL_E2, lb, m, lds);
}

// main.c:332-354: v = clamp(v + c w, 0, 1); partial max |c w|.
template <typename T, int K>
__device__ __forceinline__ void edge_update_unit(const EngArgs<T> &a, const UG<T> &U, int lb, int it,
                                                 double *lds) {
    const int64_t q = (int64_t)lb * kPixBlock + threadIdx.x;
    double m[K];
#pragma unroll
    for (int j = 0; j < K; ++j) m[j] = 0.0;
    int pi, pj;
    if (real_pixel(q, U.npix_t, U.tny, U.nx, U.ny, pi, pj)) {
        T vv[K], ww[K];
        loadk<T, K>(U.v + q * K, vv);
        loadk<T, K>(U.w + q * K, ww);
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const int js = U.job0 + j;
            if (!edge_live(a, js, it)) continue;
            const double cd = jsc(a, js).e_c * (double)ww[j];
            double x = (double)vv[j] + cd;
            m[j] = fabs(cd);
            if (x > 1) x = 1;
            if (x < 0) x = 0;
            vv[j] = (T)x;
        }
        storek<T, K>(U.v + q * K, vv);
    }
    block_store<T, K, true>(a, U, SL_E3, lb, m, lds);
}

// ---------------------------------------------------------------------------
// Kernels: block -> (unit, local block) and dispatch on K.

#define MI_KSWITCH(KMAX, CALL)                  \
    if constexpr (KMAX == 1) {                  \
        constexpr int K = 1;                    \
        CALL;                                   \
    } else if constexpr (KMAX == 4) {           \
        switch (U.K) {                          \
            case 1: { constexpr int K = 1; CALL; break; } \
            case 2: { constexpr int K = 2; CALL; break; } \
            default: { constexpr int K = 4; CALL; break; } \
        }                                       \
    } else {                                    \
        switch (U.K) {                          \
            case 1: { constexpr int K = 1; CALL; break; } \
            case 2: { constexpr int K = 2; CALL; break; } \
            case 4: { constexpr int K = 4; CALL; break; } \
            default: { constexpr int K = 8; CALL; break; } \
        }                                       \
    }

template <typename T, int KMAX, bool RESID, int FM>
__global__ __launch_bounds__(kBlock) void k_eng_fp(EngArgs<T> a, BlockMap m, int s) {
    __shared__ double lds[kBlock / kWave * kMaxK];
    __shared__ double ldr[kBlock / kOtfPerWave * KMAX];
    int ui, lb;
    if (!unit_block(m, ui, lb)) return;
    const UG<T> U(a.units[ui]);
    if (unit_idle(a, U)) return;
    MI_KSWITCH(KMAX, (fp_unit<T, K, RESID, FM>(a, U, s, lb, lds, ldr)))
}

template <int KMAX, bool RESID>
__global__ __launch_bounds__(kLineBlock) void k_line_fp(EngArgs<float> a, BlockMap m, int s) {
    __shared__ double lds[kLineWaves * KMAX * kLineRays];
    int ui, lb;
    if (!unit_block(m, ui, lb)) return;
    const UG<float> U(a.units[ui]);
    if (unit_idle(a, U)) return;
    MI_KSWITCH(KMAX, (line_fp_unit<K, RESID>(a, U, s, lb, lds)))
}

// The bounds keep the waves a SIMD that the LDS slots leave room for (six at K =
// 1, five at K = 4, four at K = 8): unbounded, a few more registers cost one.
template <int KMAX, int P>
__global__ __launch_bounds__(P * kBlock, KMAX == 1 ? 6 : KMAX == 4 ? 5 : 4) void k_line_bp(EngArgs<float> a, BlockMap m, int s, int cap) {
    __shared__ double lds[kBlock / kWave * kMaxK];
    extern __shared__ __align__(16) unsigned char ldr_raw[];
    int ui, lb;
    if (!unit_block(m, ui, lb)) return;
    const UG<float> U(a.units[ui]);
    if (unit_idle(a, U)) return;
    MI_KSWITCH(KMAX, (line_bp_unit<K, P>(a, U, a.units + ui, s, lb, cap, lds, (LDSP unsigned char *)ldr_raw)))
}

template <typename T, int KMAX, bool LDS, bool SQ>
__global__ __launch_bounds__(kBlock) void k_eng_bp(EngArgs<T> a, BlockMap m, int s, int sq_off) {
    __shared__ double lds[kBlock / kWave * kMaxK];
    extern __shared__ __align__(16) unsigned char ldr_raw[];   // LDS: the block's residual slots
    int ui, lb;
    if (!unit_block(m, ui, lb)) return;
    const UG<T> U(a.units[ui]);
    if (unit_idle(a, U)) return;
    MI_KSWITCH(KMAX, (bp_unit<T, K, LDS, SQ>(a, U, s, lb, lds, (LDSP T *)ldr_raw, sq_off)))
}

// Fixed-order block reduction of n partials (sum or max), 256 threads.
__device__ __forceinline__ double fin_reduce(const GL double *p, int64_t n, bool mx, double *lds) {
    double acc = 0.0;
    for (int64_t base = 0; base < n; base += (int64_t)kBlock * 8) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int64_t i = base + u * kBlock + threadIdx.x;
            v[u] = (i < n) ? p[i] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) acc = mx ? fmax(acc, v[u]) : acc + v[u];
    }
    acc = mx ? wave_max(acc) : group_sum<kWave>(acc);
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    if (lane == 0) lds[wv] = acc;
    __syncthreads();
    double t = 0.0;
    for (int w = 0; w < kBlock / kWave; ++w) t = mx ? fmax(t, lds[w]) : t + lds[w];
    __syncthreads();
    return t;
}

// Fixed-order block sums of up to four partial arrays at once (all their
// loads in flight together), 256 threads; out[i] = sum of p[i][0 .. n[i]).
template <int NA>
__device__ __forceinline__ void fin_reduce_n(const GL double *const (&p)[NA], const int64_t (&n)[NA],
                                             double (&out)[NA], double *lds) {
    double acc[NA];
#pragma unroll
    for (int q = 0; q < NA; ++q) acc[q] = 0.0;
    int64_t nmax = 0;
#pragma unroll
    for (int q = 0; q < NA; ++q) nmax = n[q] > nmax ? n[q] : nmax;
    for (int64_t base = 0; base < nmax; base += (int64_t)kBlock * 4) {
        double v[NA][4];
#pragma unroll
        for (int q = 0; q < NA; ++q)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int64_t i = base + u * kBlock + threadIdx.x;
                v[q][u] = (i < n[q]) ? p[q][i] : 0.0;
            }
#pragma unroll
        for (int q = 0; q < NA; ++q)
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[q] += v[q][u];
    }
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
#pragma unroll
    for (int q = 0; q < NA; ++q) {
        acc[q] = group_sum<kWave>(acc[q]);
        if (lane == 0) lds[q * (kBlock / kWave) + wv] = acc[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NA; ++q) {
        double t = 0.0;
        for (int w = 0; w < kBlock / kWave; ++w) t += lds[q * (kBlock / kWave) + w];
        out[q] = t;
    }
    __syncthreads();
}

__host__ __device__ __forceinline__ int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// The subset step's sums of job j of unit U (fixed order over the blocks of
// the forward walks, back projection and nV) and its line search
// c = <d,d> / (S |A_s d|^2 + alpha nV(d)).  All threads of the block.
template <typename T>
__device__ __forceinline__ void fin_step(const EngArgs<T> &a, const UG<T> &U, int j, int s, double *lds) {
    const int js = U.job0 + j;
    if (!job_live(a, js)) return;
    GL Scalars *sc = &jsc(a, js);
    const GL JobParams &P = jpar(a, js);
    const GL int64_t *fs0 = U.ln_slice0 ? U.ln_slice0 : U.fs_slice0;
    const int64_t nr = cdiv(fs0[s + 1] - fs0[s], kBlock / kWave);
    const int64_t nb = cdiv(U.bs_slice0[s + 1] - U.bs_slice0[s], kBlock / kWave);
    const int64_t npx = cdiv(U.npix_t, kPixBlock);
    const GL double *const p[4] = {part_at(a, U, SL_DD, j), part_at(a, U, SL_AD, j), part_at(a, U, SL_NV, j),
                                   part_at(a, U, SL_DF, j)};
    const int64_t n[4] = {nb, nr, npx, nr};
    double r[4];
    fin_reduce_n<4>(p, n, r, lds);
    const double dd = r[0], ad2 = r[1], nv = r[2], df = r[3];
    if (threadIdx.x == 0) {
        sc->df_pass += df;
        sc->dd = dd;
        sc->ad2 = ad2;
        sc->nv = nv;
        const double den = (double)a.S * ad2 + P.alpha * nv;
        sc->c = (den > 0) ? dd / den : 0.0;
    }
}

// Finalize op `op` of job j of unit U (every thread of the block calls it).
template <typename T>
__device__ __forceinline__ void fin_job(const EngArgs<T> &a, const UG<T> &U, int j, int op, int s, double *lds) {
    const int js = U.job0 + j;
    if (!job_live(a, js)) return;
    GL Scalars *sc = &jsc(a, js);
    const GL JobParams &P = jpar(a, js);
    const int64_t npx = cdiv(U.npix_t, kPixBlock);
    switch (op) {
        case EF_EDGE_C: {
            if (sc->edge_done || s >= P.iter_edge) return;
            const GL double *const p[3] = {part_at(a, U, SL_E0, j), part_at(a, U, SL_E1, j),
                                           part_at(a, U, SL_E2, j)};
            const int64_t n[3] = {npx, npx, npx};
            double r[3];
            fin_reduce_n<3>(p, n, r, lds);
            const double nd = r[0], nd2 = r[1], nnd = r[2];
            if (threadIdx.x == 0) {
                // origin/GoldenC/src/main.c:329
                sc->e_nd = nd;
                sc->e_nd2 = nd2;
                sc->e_nnd = nnd;
                sc->e_c = nd / (P.alpha * nd2 + P.beta * P.eps * nnd + (P.beta / (4 * P.eps)) * nd);
            }
            break;
        }
        case EF_EDGE_DONE:
        case EF_EDGE_END: {
            // every wave has read the flag before EF_END below clears it
            // (without the reduction no barrier stands between the two)
            const bool stopped = sc->edge_done;
            __syncthreads();
            if (!stopped && s < P.iter_edge) {
                const double mx = fin_reduce(part_at(a, U, SL_E3, j), npx, true, lds);
                if (threadIdx.x == 0) {
                    sc->e_maxcd = mx;
                    if (mx < 1e-5) sc->edge_done = 1;   // main.c:351
                }
            }
            if (op == EF_EDGE_DONE) break;
            [[fallthrough]];
        }
        default: {  // EF_END
            if (threadIdx.x != 0) return;
            const double df = sc->df_pass;
            if (sc->iters > 0) {
                const double diff = fabs(df - sc->df_prev);
                sc->rel = sc->df_prev > 0 ? diff / sc->df_prev : 0.0;
                if (diff < P.rel_tol * sc->df_prev) sc->converged = 1;
            }
            sc->df_prev = df;
            sc->df_pass = 0.0;
            sc->edge_done = 0;
            sc->iters += 1;
            if (sc->converged || (P.max_iters > 0 && sc->iters >= P.max_iters)) sc->done = 1;
            break;
        }
    }
}

// One block per job slot (units listed in m; m.nunits * kMaxK blocks).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_eng_fin(EngArgs<T> a, int op, int s) {
    __shared__ double lds[4 * (kBlock / kWave)];
    const int ui = blockIdx.x / kMaxK, j = blockIdx.x % kMaxK;
    const UG<T> U(a.units[ui]);
    if (j >= U.K) return;
    if (op == EF_STEP) fin_step(a, U, j, s, lds);
    else fin_job(a, U, j, op, s, lds);
}

enum PixOp { PX_AXPY = 0, PX_MEDIAN, PX_COPY_WU, PX_EDGE_GRAD, PX_EDGE_NABLA, PX_EDGE_UPDATE, PX_NV };

template <typename T, int KMAX, int OP>
__global__ __launch_bounds__(kBlock) void k_eng_pix(EngArgs<T> a, BlockMap m, int it) {
    __shared__ double lds[kBlock / kWave * kMaxK];
    // strips of the arrays the stencil reads around (u and v for the edge
    // gradient, one array for the median, nV and the gradient of the edge
    // direction)
    constexpr int kStrips = OP == PX_EDGE_GRAD ? 2 : (OP == PX_MEDIAN || OP == PX_EDGE_NABLA || OP == PX_NV ? 1 : 0);
    __shared__ __align__(16) T L[kStrips ? kStrips * kHaloN * KMAX : 1];
    int ui, lb;
    if (!unit_block(m, ui, lb)) return;
    const UG<T> U(a.units[ui]);
    if (unit_idle(a, U)) return;
    if constexpr (OP == PX_AXPY) { MI_KSWITCH(KMAX, (axpy_unit<T, K>(a, U, lb))) }
    else if constexpr (OP == PX_MEDIAN) { MI_KSWITCH(KMAX, (median_unit<T, K>(a, U, lb, L))) }
    else if constexpr (OP == PX_NV) { MI_KSWITCH(KMAX, (nv_unit<T, K>(a, U, lb, lds, L))) }
    else if constexpr (OP == PX_COPY_WU) { MI_KSWITCH(KMAX, (copy_wu_unit<T, K>(a, U, lb))) }
    else if constexpr (OP == PX_EDGE_GRAD) { MI_KSWITCH(KMAX, (edge_grad_unit<T, K>(a, U, lb, it, lds, L))) }
    else if constexpr (OP == PX_EDGE_NABLA) { MI_KSWITCH(KMAX, (edge_nabla_unit<T, K>(a, U, lb, it, lds, L))) }
    else { MI_KSWITCH(KMAX, (edge_update_unit<T, K>(a, U, lb, it, lds))) }
}

template <typename T>
__global__ void k_put_rows(T *dst, int K, int slot, int64_t n, const int64_t *perm, const T *src) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i * K + slot] = src[perm[i]];
}
// Row-major image <-> slot of a tiled interleaved image.
template <typename T>
__global__ void k_put_img(T *dst, int K, int slot, int nx, int ny, int tny, const T *src, T fillv) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= (int64_t)nx * ny) return;
    const int64_t q = tile_index((int)(p / ny), (int)(p % ny), tny);
    dst[q * K + slot] = src ? src[p] : fillv;
}
template <typename T>
__global__ void k_get_img(T *dst, const T *src, int K, int slot, int nx, int ny, int tny) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= (int64_t)nx * ny) return;
    dst[p] = src[tile_index((int)(p / ny), (int)(p % ny), tny) * K + slot];
}
template <typename T>
__global__ void k_move(T *dst, int Kd, int sd, const T *src, int Ks, int ss, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i * Kd + sd] = src[i * Ks + ss];
}

// u and its remainder into the projection images (put_proj_u): one thread per
// pixel and job, row by row (px, qx) and column by column (py, qy).
template <typename T>
__global__ void k_spread(const T *u, const T *ul, float *px, float *py, void *qx, void *qy, int K, int nx, int ny, int tny) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (int64_t)nx * ny * K) return;
    const int64_t p = e / K;
    const int k = (int)(e - p * K);
    const int i = (int)(p / ny), j = (int)(p % ny);
    const int jt = (int)(p / nx), it = (int)(p % nx);
    const int64_t q = tile_index(i, j, tny) * K + k, qt = tile_index(it, jt, tny) * K + k;
    const int64_t x = ((int64_t)i * line_stride(ny) + j + kLinePad) * K + k;
    const int64_t y = ((int64_t)jt * line_stride(nx) + it + kLinePad) * K + k;
    float f, ft;
    uint32_t lo, lot;
    line_split((double)u[q] + (double)ul[q], f, lo);
    line_split((double)u[qt] + (double)ul[qt], ft, lot);
    if (K <= 2) {
        ((double *)qx)[x] = line_join(f, lo << 13);
        ((double *)qy)[y] = line_join(ft, lot << 13);
    } else {
        px[x] = f;
        py[y] = ft;
        ((uint16_t *)qx)[x] = (uint16_t)lo;
        ((uint16_t *)qy)[y] = (uint16_t)lot;
    }
}

// Plain streaming copy, 16 bytes per thread per step (the reference kernel
// against which memory counters are read).
__global__ __launch_bounds__(kBlock) void k_copy16(const u32x4 *__restrict__ src, u32x4 *__restrict__ dst,
                                                   int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock)
        dst[i] = src[i];
}

unsigned grid8(int blocks) {
    if (blocks < 1) blocks = 1;
    return (unsigned)((blocks + 7) / 8 * 8);
}
unsigned grid_of(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

}  // namespace

// ---------------------------------------------------------------------------

template <typename T>
void eng_fp_resid(hipStream_t st, const EngArgs<T> &a, const BlockMap &m, int s, int kmax, bool all_walk) {
    const unsigned grid = grid8(m.start[m.nunits]);
    if (all_walk) {
        if (kmax == 1) launch(k_eng_fp<T, 1, true, 1>, dim3(grid), dim3(kBlock), (uint32_t)(0), st, a, m, s);
        else if (kmax <= 4) launch(k_eng_fp<T, 4, true, 1>, dim3(grid), dim3(kBlock), (uint32_t)(0), st, a, m, s);
        else launch(k_eng_fp<T, kMaxK, true, 1>, dim3(grid), dim3(kBlock), (uint32_t)(0), st, a, m, s);
    } else {
        if (kmax == 1) launch(k_eng_fp<T, 1, true, 3>, dim3(grid), dim3(kBlock), (uint32_t)(0), st, a, m, s);
        else if (kmax <= 4) launch(k_eng_fp<T, 4, true, 3>, dim3(grid), dim3(kBlock), (uint32_t)(0), st, a, m, s);
        else launch(k_eng_fp<T, kMaxK, true, 3>, dim3(grid), dim3(kBlock), (uint32_t)(0), st, a, m, s);
    }
    MI_HIP(hipGetLastError());
}

// Dynamic LDS of a back-projection launch.  The u / v squares of the
// regulariser either take a region of their own behind the residual slots,
// loaded while the slots are (the kernel's SQ form, squares at element sq_off),
// or reuse the slots' LDS after the walk.  The staged form takes its own
// region when both fit the launch's LDS and that kernel keeps as many blocks
// per CU (its registers and LDS, by the occupancy calculator, up to the
// blocks per CU the grid has); the global-gather form holds only the squares.
template <typename T, int KM, bool LDS>
void bp_launch(hipStream_t st, unsigned grid, const EngArgs<T> &a, const BlockMap &m, int s, size_t slot_bytes,
               int sq_mode) {
    const size_t sq = (size_t)2 * kSqN * KM * sizeof(T), at = (slot_bytes + 15) & ~(size_t)15;
    const uint32_t own = (uint32_t)(at + sq), shared = (uint32_t)std::max(slot_bytes, sq);
    const int sq_off = (int)(at / sizeof(T));
    if constexpr (!LDS) {
        launch(k_eng_bp<T, KM, false, true>, dim3(grid), dim3(kBlock), own, st, a, m, s, sq_off);
    } else {
        bool sep = false;
        if (at + sq > kBpLdsLaunch) {
            sep = false;
        } else if (sq_mode >= 0) {
            sep = sq_mode == 1;
        } else {
            int nb_own = 0, nb_shared = 0;
            MI_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb_own, (const void *)k_eng_bp<T, KM, true, true>,
                                                                kBlock, own));
            MI_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &nb_shared, (const void *)k_eng_bp<T, KM, true, false>, kBlock, shared));
            int dev = 0, ncu = 1;
            MI_HIP(hipGetDevice(&dev));
            MI_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
            const int used = (int)((grid + ncu - 1) / ncu);   // blocks per CU the launch can place
            sep = std::min(nb_own, used) >= std::min(nb_shared, used);
        }
        if (sep) launch(k_eng_bp<T, KM, true, true>, dim3(grid), dim3(kBlock), own, st, a, m, s, sq_off);
        else launch(k_eng_bp<T, KM, true, false>, dim3(grid), dim3(kBlock), shared, st, a, m, s, 0);
    }
}

template <typename T>
void eng_bp_grad(hipStream_t st, const EngArgs<T> &a, const BlockMap &m, int s, int kmax, size_t lds_bytes,
                 int sq_mode) {
    const unsigned grid = grid8(m.start[m.nunits]);
    if (lds_bytes) {
        if (kmax == 1) bp_launch<T, 1, true>(st, grid, a, m, s, lds_bytes, sq_mode);
        else if (kmax <= 4) bp_launch<T, 4, true>(st, grid, a, m, s, lds_bytes, sq_mode);
        else bp_launch<T, kMaxK, true>(st, grid, a, m, s, lds_bytes, sq_mode);
    } else {
        if (kmax == 1) bp_launch<T, 1, false>(st, grid, a, m, s, 0, sq_mode);
        else if (kmax <= 4) bp_launch<T, 4, false>(st, grid, a, m, s, 0, sq_mode);
        else bp_launch<T, kMaxK, false>(st, grid, a, m, s, 0, sq_mode);
    }
    MI_HIP(hipGetLastError());
}

template <typename T>
void eng_fp_sq(hipStream_t st, const EngArgs<T> &a, const BlockMap &rows, int s, int kmax, bool all_walk) {
    const unsigned grid = grid8(rows.start[rows.nunits]);
    if (all_walk) {
        if (kmax == 1) launch(k_eng_fp<T, 1, false, 1>, dim3(grid), dim3(kBlock), (uint32_t)(0), st, a, rows, s);
        else if (kmax <= 4) launch(k_eng_fp<T, 4, false, 1>, dim3(grid), dim3(kBlock), (uint32_t)(0), st, a, rows, s);
        else launch(k_eng_fp<T, kMaxK, false, 1>, dim3(grid), dim3(kBlock), (uint32_t)(0), st, a, rows, s);
    } else {
        if (kmax == 1) launch(k_eng_fp<T, 1, false, 3>, dim3(grid), dim3(kBlock), (uint32_t)(0), st, a, rows, s);
        else if (kmax <= 4) launch(k_eng_fp<T, 4, false, 3>, dim3(grid), dim3(kBlock), (uint32_t)(0), st, a, rows, s);
        else launch(k_eng_fp<T, kMaxK, false, 3>, dim3(grid), dim3(kBlock), (uint32_t)(0), st, a, rows, s);
    }
    MI_HIP(hipGetLastError());
}

void eng_line_fp(hipStream_t st, const EngArgs<float> &a, const BlockMap &m, int s, int kmax, bool resid) {
    const dim3 grid(grid8(m.start[m.nunits])), block(kLineBlock);
    if (resid) {
        if (kmax == 1) launch(k_line_fp<1, true>, grid, block, 0u, st, a, m, s);
        else if (kmax <= 4) launch(k_line_fp<4, true>, grid, block, 0u, st, a, m, s);
        else launch(k_line_fp<kMaxK, true>, grid, block, 0u, st, a, m, s);
    } else {
        if (kmax == 1) launch(k_line_fp<1, false>, grid, block, 0u, st, a, m, s);
        else if (kmax <= 4) launch(k_line_fp<4, false>, grid, block, 0u, st, a, m, s);
        else launch(k_line_fp<kMaxK, false>, grid, block, 0u, st, a, m, s);
    }
    MI_HIP(hipGetLastError());
}

// LDS slots of a half: fewer rounds with more of them, so the workgroups that
// a CU gets share its LDS, up to six of them (874 x 874, 72 views: 97.9 us; four
// 109.4, eight 99.6).
constexpr int kLineResident = 6;
template <int KM, int P>
static void line_bp_launch(hipStream_t st, const EngArgs<float> &a, const BlockMap &m, int s) {
    const int blocks = m.start[m.nunits];
    constexpr int per = 2 * line_slot_bytes(KM), fix = 2 * kLineViews * (int)sizeof(LineView);
    const int res = std::min(kLineResident, (blocks + 255) / 256);
    const int lim = (int)std::min<size_t>(kBpLdsLaunch, ((size_t)160 << 10) / res - 1024);
    const int cap = std::max(kLineSlots, std::min(1024, (lim - fix) / per & ~3));
    const size_t lds = std::max({(size_t)cap * per + fix, (size_t)2 * kSqN * KM * sizeof(float),
                                 (size_t)(P - 1) * KM * kBlock * sizeof(double)});
    launch(k_line_bp<KM, P>, dim3(grid8(blocks)), dim3(P * kBlock), (uint32_t)lds, st, a, m, s, cap);
}
static_assert(kLineSlots * 2 * line_slot_bytes(kMaxK) + 2 * kLineViews * sizeof(LineView) <= kBpLdsLaunch,
              "the slots of eight jobs fit a launch");

void eng_line_bp(hipStream_t st, const EngArgs<float> &a, const BlockMap &m, int s, int kmax, int groups) {
    auto go = [&](auto km) {
        constexpr int KM = decltype(km)::value;
        if (groups == 4) line_bp_launch<KM, 4>(st, a, m, s);
        else if (groups == 2) line_bp_launch<KM, 2>(st, a, m, s);
        else line_bp_launch<KM, 1>(st, a, m, s);
    };
    if (kmax == 1) go(std::integral_constant<int, 1>{});
    else if (kmax <= 4) go(std::integral_constant<int, 4>{});
    else go(std::integral_constant<int, kMaxK>{});
    MI_HIP(hipGetLastError());
}

void line_project(hipStream_t st, const Matrix &m, const float *img, float *px, float *py, float *sino) {
    const mi_geometry &g = m.g;
    const Lines &q = m.lines;
    const int64_t groups = q.slice0.back() / 4;
    k_line_planes<<<grid_of(line_elems(g.nx, g.ny) + line_elems(g.ny, g.nx)), kBlock, 0, st>>>(img, g.nx, g.ny, px, py);
    MI_HIP(hipGetLastError());
    k_line_project<<<grid8((int)groups), kLineBlock, 0, st>>>(px, py, g.nx, g.ny, g.n_bins, groups, q.mb.p, q.inv.p, q.len.p,
                                                              q.drop.p, q.skip.p, q.rng.p, sino);
    MI_HIP(hipGetLastError());
}

template <typename T>
void eng_spread(hipStream_t st, const T *u, const T *ul, float *px, float *py, void *qx, void *qy, int K, int nx, int ny,
                int tny) {
    k_spread<T><<<grid_of((int64_t)nx * ny * K), kBlock, 0, st>>>(u, ul, px, py, qx, qy, K, nx, ny, tny);
    MI_HIP(hipGetLastError());
}

template <typename T, int OP>
static void launch_pix(hipStream_t st, const EngArgs<T> &a, const BlockMap &m, int it, int kmax) {
    const unsigned grid = grid8(m.start[m.nunits]);
    if (kmax == 1) k_eng_pix<T, 1, OP><<<grid, kBlock, 0, st>>>(a, m, it);
    else if (kmax <= 4) k_eng_pix<T, 4, OP><<<grid, kBlock, 0, st>>>(a, m, it);
    else k_eng_pix<T, kMaxK, OP><<<grid, kBlock, 0, st>>>(a, m, it);
    MI_HIP(hipGetLastError());
}

template <typename T>
void eng_nv(hipStream_t st, const EngArgs<T> &a, const BlockMap &pix, int kmax) {
    launch_pix<T, PX_NV>(st, a, pix, 0, kmax);
}

template <typename T>
void eng_axpy(hipStream_t st, const EngArgs<T> &a, const BlockMap &pix, int kmax) {
    launch_pix<T, PX_AXPY>(st, a, pix, 0, kmax);
}

template <typename T>
void eng_median(hipStream_t st, const EngArgs<T> &a, const BlockMap &pix, int kmax) {
    launch_pix<T, PX_MEDIAN>(st, a, pix, 0, kmax);
    launch_pix<T, PX_COPY_WU>(st, a, pix, 0, kmax);
}

template <typename T>
void eng_edge_iter(hipStream_t st, const EngArgs<T> &a, const BlockMap &pix, int it, int kmax, bool last) {
    launch_pix<T, PX_EDGE_GRAD>(st, a, pix, it, kmax);
    launch_pix<T, PX_EDGE_NABLA>(st, a, pix, it, kmax);
    eng_finalize<T>(st, a, EF_EDGE_C, it);
    launch_pix<T, PX_EDGE_UPDATE>(st, a, pix, it, kmax);
    eng_finalize<T>(st, a, last ? EF_EDGE_END : EF_EDGE_DONE, it);
}

template <typename T>
void eng_finalize(hipStream_t st, const EngArgs<T> &a, int op, int s) {
    if (a.nunits <= 0) return;
    k_eng_fin<T><<<(unsigned)(a.nunits * kMaxK), kBlock, 0, st>>>(a, op, s);
    MI_HIP(hipGetLastError());
}

template <typename T>
void eng_put_rows(hipStream_t st, T *dst, int K, int slot, int64_t n, const int64_t *perm, const T *src) {
    if (n <= 0) return;
    k_put_rows<T><<<grid_of(n), kBlock, 0, st>>>(dst, K, slot, n, perm, src);
    MI_HIP(hipGetLastError());
}
template <typename T>
void eng_put_img(hipStream_t st, T *dst, int K, int slot, int nx, int ny, int tny, const T *src, T fillv) {
    const int64_t n = (int64_t)nx * ny;
    if (n <= 0) return;
    k_put_img<T><<<grid_of(n), kBlock, 0, st>>>(dst, K, slot, nx, ny, tny, src, fillv);
    MI_HIP(hipGetLastError());
}
template <typename T>
void eng_get_img(hipStream_t st, T *dst, const T *src, int K, int slot, int nx, int ny, int tny) {
    const int64_t n = (int64_t)nx * ny;
    if (n <= 0) return;
    k_get_img<T><<<grid_of(n), kBlock, 0, st>>>(dst, src, K, slot, nx, ny, tny);
    MI_HIP(hipGetLastError());
}
template <typename T>
void eng_move(hipStream_t st, T *dst, int Kd, int sd, const T *src, int Ks, int ss, int64_t n) {
    if (n <= 0) return;
    k_move<T><<<grid_of(n), kBlock, 0, st>>>(dst, Kd, sd, src, Ks, ss, n);
    MI_HIP(hipGetLastError());
}

void eng_copy(hipStream_t st, void *dst, const void *src, int64_t bytes) {
    MI_REQUIRE(bytes % 16 == 0, MI_E_ARG, "copy size must be a multiple of 16 bytes");
    const int64_t n = bytes / 16;
    if (n == 0) return;
    k_copy16<<<8192, kBlock, 0, st>>>((const u32x4 *)src, (u32x4 *)dst, n);
    MI_HIP(hipGetLastError());
}

#define MI_ENG_INST(T)                                                                                     \
    template void eng_fp_resid<T>(hipStream_t, const EngArgs<T> &, const BlockMap &, int, int, bool);       \
    template void eng_bp_grad<T>(hipStream_t, const EngArgs<T> &, const BlockMap &, int, int, size_t, int); \
    template void eng_fp_sq<T>(hipStream_t, const EngArgs<T> &, const BlockMap &, int, int, bool);         \
    template void eng_spread<T>(hipStream_t, const T *, const T *, float *, float *, void *, void *, int, int, int, int); \
    template void eng_nv<T>(hipStream_t, const EngArgs<T> &, const BlockMap &, int);                        \
    template void eng_axpy<T>(hipStream_t, const EngArgs<T> &, const BlockMap &, int);                      \
    template void eng_median<T>(hipStream_t, const EngArgs<T> &, const BlockMap &, int);                    \
    template void eng_edge_iter<T>(hipStream_t, const EngArgs<T> &, const BlockMap &, int, int, bool);      \
    template void eng_finalize<T>(hipStream_t, const EngArgs<T> &, int, int);                               \
    template void eng_put_rows<T>(hipStream_t, T *, int, int, int64_t, const int64_t *, const T *);         \
    template void eng_put_img<T>(hipStream_t, T *, int, int, int, int, int, const T *, T);                  \
    template void eng_get_img<T>(hipStream_t, T *, const T *, int, int, int, int, int);                     \
    template void eng_move<T>(hipStream_t, T *, int, int, const T *, int, int, int64_t);

MI_ENG_INST(float)
MI_ENG_INST(double)

}  // namespace mi
