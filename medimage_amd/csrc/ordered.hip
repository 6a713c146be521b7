// Reference-order FP64 operators and the GoldenC CG / SD drivers built on
// them (see ordered.hpp).  Every sum here is added in the order the
// reference program adds it, so results equal the reference's bit for bit:
//   * A: one lane per ray sums its products in the order proj.c emits them;
//   * AStar: one lane per pixel, likewise;
//   * energies, norms, inner products: one workgroup per sum, whose result
//     is the running double's after adding the terms one by one in
//     row-major order (k_chains).
#include "ordered.hpp"
#include "gc_stencil.hpp"

#include <algorithm>
#include <cstring>
#include <limits>

namespace mi {

void goldenc_lists(bool pixel_major, std::vector<int64_t> &ptr, std::vector<uint32_t> &other,
                   std::vector<double> &len);

namespace {

struct SeqView {
    int64_t items;
    const int64_t *base;
    const int32_t *steps, *cnt;
    const uint32_t *other;
    const double *len;
};
SeqView view_of(const SeqLists &L) {
    return SeqView{L.items, L.base.p, L.steps.p, L.cnt.p, L.other.p, L.len.p};
}

// One lane per item: s = sum over the item's entries, in list order, of
// x[other] * len in T (product rounded, then added: no contraction; the
// lengths are stored widened to double, exactly, and narrowed back).
template <typename T>
__device__ __forceinline__ T seq_item_sum(const SeqView &L, int64_t i, const T *__restrict__ x) {
    const int64_t gi = i >> 6;
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t b = L.base[gi];
    const int steps = L.steps[gi];
    const int c = i < L.items ? L.cnt[i] : 0;
    T s = T(0);
    for (int t = 0; t < steps; t += 4) {
        uint32_t k[4];
        T l[4], xv[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t at = b + (int64_t)(t + j) * kWave + lane;
            k[j] = L.other[at];
            l[j] = (T)L.len[at];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) xv[j] = x[k[j]];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (t + j < c) s = s + xv[j] * l[j];
    }
    return s;
}

template <typename T, bool RESID>
__global__ __launch_bounds__(kBlock) void k_seq_fp(SeqView L, const T *__restrict__ x, T *__restrict__ out,
                                                   const T *__restrict__ g, T *__restrict__ resid) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (((i >> 6) << 6) >= L.items) return;
    const T s = seq_item_sum<T>(L, i, x);
    if (i < L.items) {
        out[i] = s;
        if (RESID) resid[i] = g[i] - s;
    }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_seq_bp(SeqView L, int nx, int ny, const T *__restrict__ r,
                                                   const T *__restrict__ u, const T *__restrict__ v, double alpha,
                                                   double eps, T *__restrict__ d) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (((i >> 6) << 6) >= L.items) return;
    const T s = seq_item_sum<T>(L, i, r);
    if (i < L.items) {
        T dv = s;
        if (u) dv = (T)((double)dv + alpha * gc_reg(u, v, (int)(i / ny), (int)(i % ny), nx, ny, eps));
        d[i] = dv;
    }
}

// ---------------------------------------------------------------------------
// Sequential sums.  Terms (origin/GoldenC/src/main.c):
enum ChainTerm : int {
    CT_SQDIFF = 0,   // (a - b)^2, rows:  sqr(Af - g), :127-130
    CT_SQ = 1,       // a^2:              sqr(q), :162-164; sqr(d), :318-320
    CT_DOT = 2,      // a b:              p d, :159-161; Ad q, :241-243
    CT_REG_INT = 3,  // interior energy of f = a, v = b, :135-139
    CT_NV = 4,       // nV of p = a, v = b (p zero padded), :152-158
    CT_NABLA2 = 5,   // two terms per pixel of d = a (zero padded), :313-316
    CT_NDSQ = 6      // a b^2:            n d^2, :322-325
};
struct ChainSeg {
    int term;
    int64_t n;             // terms (pixels for CT_NABLA2)
    const double *a, *b;
};
struct ChainDesc {
    ChainSeg seg[2];       // the second segment continues the first's sum
    int nseg;
    double *out;
};
struct ChainArgs {
    ChainDesc c[4];
    int nchains;
    int nx, ny;
    double alpha, beta, eps;
    int edge_c;            // chains are nNablaD, nD, sum n d^2 of the edge step; then
    Scalars *sc;           //   sc->e_c (main.c:329); all skipped once edge_done
};

template <int TERM>
__device__ __forceinline__ void chain_term(const ChainSeg &s, const ChainArgs &a, int64_t e, double &t0, double &t1) {
    const double *A = s.a, *B = s.b;
    const int nx = a.nx, ny = a.ny;
    if constexpr (TERM == CT_SQDIFF) {
        const double x = A[e] - B[e];
        t0 = x * x;
    } else if constexpr (TERM == CT_SQ) {
        t0 = A[e] * A[e];
    } else if constexpr (TERM == CT_DOT) {
        t0 = A[e] * B[e];
    } else if constexpr (TERM == CT_REG_INT) {
        // pixel counts fit 32 bits (a 64-bit division is some 100 instructions)
        const unsigned w2 = (unsigned)(ny - 2), i = (unsigned)e / w2;
        const int64_t q = (int64_t)(1 + i) * ny + 1 + ((unsigned)e - i * w2);
        const double z = A[q], zu = A[q - ny], zl = A[q - 1], w = B[q];
        t0 = a.alpha * (w * w + 0.01 * (a.eps * a.eps)) * ((z - zu) * (z - zu) + (z - zl) * (z - zl));
    } else if constexpr (TERM == CT_NV) {
        const int i = (int)((unsigned)e / (unsigned)ny), j = (int)e - i * ny;
        const double z = A[e], zu = gc_ld(A, i - 1, j, nx, ny, 0.0), zl = gc_ld(A, i, j - 1, nx, ny, 0.0);
        const double w = B[e];
        t0 = (w * w + 0.01 * (a.eps * a.eps)) * ((z - zu) * (z - zu) + (z - zl) * (z - zl));
    } else if constexpr (TERM == CT_NABLA2) {
        const int i = (int)((unsigned)e / (unsigned)ny), j = (int)e - i * ny;
        const double x = 0.5 * (gc_ld(A, i + 1, j, nx, ny, 0.0) - gc_ld(A, i - 1, j, nx, ny, 0.0));
        const double y = 0.5 * (gc_ld(A, i, j + 1, nx, ny, 0.0) - gc_ld(A, i, j - 1, nx, ny, 0.0));
        t0 = x * x;
        t1 = y * y;
    } else {
        t0 = A[e] * (B[e] * B[e]);
    }
}

// One sequential sum per workgroup, 4096 terms a step.
//
// The terms are computed by all lanes, and folding them in index order
// (rounding after every add, as the reference's loop does) need not be a
// serial chain.  While the running sum acc stays inside one binade, adding a
// term t moves it by t rounded to acc's own unit in the last place, whatever
// acc's bits are, unless t lies exactly halfway between two multiples of it
// (then ties-to-even looks at acc).  So per 256 terms (one wave) the rounded
// terms are integers that may be added in any order, and the 16 waves' sums
// are applied in order as long as (a) no term is a tie, infinite, NaN or
// 2^50 units or more, and (b) acc plus the wave's positive terms stays below
// the binade's upper end and acc plus its negative ones (each up to half a
// unit more than its rounded value) above the lower end.
// A wave that fails this is folded term by term from LDS, after which the
// waves behind it are rounded again for acc's new binade.  acc's binade
// changes about log2(n) times, so a sum of 4e5 terms folds some 20 waves of
// 1600 serially.
//
// Measured over the sums of one GoldenC alternation (2.6e5 to 5.2e5 terms):
// 696 us a launch, against 5189 us (13 ns a term) with one wave per sum that
// took each term from its lane and added it.
constexpr int kChainThreads = 1024, kChainPer = 4, kChainStep = kChainThreads * kChainPer;
constexpr int kChainWaves = kChainThreads / kWave, kChainSub = kWave * kChainPer;

struct ChainLds {
    double term[kChainStep];
    long long sum[kChainWaves], pos[kChainWaves], low[kChainWaves];   // low: bound of the negative terms, 0 without any
    int bad[kChainWaves], zero[kChainWaves];
    double acc;
};

__device__ __forceinline__ long long wave_sum_i64(long long x) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) x += __shfl_xor(x, o, kWave);
    return x;
}

// The terms of lane slots first .. first + 3 of the segment (zeros past its
// end; adding +0 leaves every running sum but -0 as it is, and the sums start
// at +0).
template <int TERM>
__device__ __forceinline__ void chain_load(const ChainSeg &s, const ChainArgs &a, int64_t first, double (&t)[kChainPer]) {
    if constexpr (TERM == CT_NABLA2) {
#pragma unroll
        for (int k = 0; k < kChainPer; k += 2) {
            const int64_t e = (first + k) >> 1;
            t[k] = t[k + 1] = 0.0;
            if (e < s.n) chain_term<TERM>(s, a, e, t[k], t[k + 1]);
        }
    } else {
#pragma unroll
        for (int k = 0; k < kChainPer; ++k) {
            double none = 0.0;
            t[k] = 0.0;
            if (first + k < s.n) chain_term<TERM>(s, a, first + k, t[k], none);
        }
    }
}

template <int TERM>
__device__ double chain_segment(const ChainSeg &s, const ChainArgs &a, double acc, ChainLds &L) {
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
    const int64_t n = TERM == CT_NABLA2 ? 2 * s.n : s.n;
    double t[kChainPer], nx[kChainPer];
    chain_load<TERM>(s, a, (int64_t)tid * kChainPer, t);
    for (int64_t b0 = 0; b0 < n; b0 += kChainStep) {
        // the next step's terms load while this one is folded
        chain_load<TERM>(s, a, b0 + kChainStep + (int64_t)tid * kChainPer, nx);
#pragma unroll
        for (int k = 0; k < kChainPer; ++k) L.term[tid * kChainPer + k] = t[k];
        const int waves = (int)min((int64_t)kChainWaves, (n - b0 + kChainSub - 1) / kChainSub);
        for (int from = 0; from < waves;) {
            // acc = +-A 2^(e - 52), 2^52 <= A < 2^53, where e is its exponent
            const long long bits = __double_as_longlong(acc);
            const int be = (int)((bits >> 52) & 0x7ff);
            const bool normal = be >= 53 && be <= 2000;   // the scale 2^(52 - e) is a normal number too
            const double scale = __longlong_as_double(((long long)(2098 - be) << 52) | (bits & ((long long)1 << 63)));
            if (wv >= from && wv < waves) {
                long long p = 0, q = 0;
                bool bad = false, zero = true, below = false;
                constexpr double M = 6755399441055744.0;   // 1.5 2^52: adding it rounds to an integer
#pragma unroll
                for (int k = 0; k < kChainPer; ++k) {
                    const double x = t[k] * scale, r = x + M;
                    const long long i = __double_as_longlong(r) - __double_as_longlong(M);
                    bad |= !(fabs(x) < 1125899906842624.0) | (fabs(x - (r - M)) == 0.5);
                    zero &= t[k] == 0.0;
                    below |= x < 0.0;
                    p += i > 0 ? i : 0;
                    q += i < 0 ? i : 0;
                }
                bad |= !normal;
                bad = __any(bad);
                zero = __all(zero);
                below = __any(below);
                if (!bad) {
                    p = wave_sum_i64(p);
                    if (below) q = wave_sum_i64(q);
                }
                if (lane == 0) {
                    L.sum[wv] = p + q;
                    L.pos[wv] = p;
                    L.low[wv] = below ? q - kChainSub : 0;
                    L.bad[wv] = bad;
                    L.zero[wv] = zero;
                }
            }
            __syncthreads();
            // every thread applies the waves' sums in order
            constexpr long long kLo = (long long)1 << 52;
            long long A = (bits & (kLo - 1)) | kLo;
            int k = from;
            for (; k < waves; ++k) {
                if (L.zero[k]) continue;   // +-0 terms leave acc as it is
                if (L.bad[k] || A + L.pos[k] >= 2 * kLo || (L.low[k] < 0 && A + L.low[k] <= kLo)) break;
                A += L.sum[k];
            }
            if (normal) acc = __longlong_as_double((bits & ~(kLo - 1)) | (A & (kLo - 1)));
            if (k < waves) {
                // wave k term by term, by one wave (all lanes alike)
                if (wv == 0) {
                    const int m = (int)min((int64_t)kChainSub, n - b0 - (int64_t)k * kChainSub);
                    const double *q = L.term + k * kChainSub;
                    int i = 0;
                    for (; i + 16 <= m; i += 16) {
                        double x[16];
#pragma unroll
                        for (int j = 0; j < 16; ++j) x[j] = q[i + j];
#pragma unroll
                        for (int j = 0; j < 16; ++j) acc = acc + x[j];
                    }
                    for (; i < m; ++i) acc = acc + q[i];
                    if (lane == 0) L.acc = acc;
                }
                ++k;
                __syncthreads();
                acc = L.acc;
            }
            from = k;
            __syncthreads();   // the tables (and, at the end, the terms) are written again
        }
#pragma unroll
        for (int k = 0; k < kChainPer; ++k) t[k] = nx[k];
    }
    return acc;
}

// One workgroup per sum.
__global__ __launch_bounds__(kChainThreads) void k_chains(ChainArgs a) {
    __shared__ ChainLds L;
    if (a.edge_c && (a.sc->edge_done || a.sc->converged)) return;
    const ChainDesc &c = a.c[blockIdx.x];
    double acc = 0.0;
    for (int k = 0; k < c.nseg; ++k) {
        const ChainSeg &s = c.seg[k];
        switch (s.term) {
            case CT_SQDIFF: acc = chain_segment<CT_SQDIFF>(s, a, acc, L); break;
            case CT_SQ: acc = chain_segment<CT_SQ>(s, a, acc, L); break;
            case CT_DOT: acc = chain_segment<CT_DOT>(s, a, acc, L); break;
            case CT_REG_INT: acc = chain_segment<CT_REG_INT>(s, a, acc, L); break;
            case CT_NV: acc = chain_segment<CT_NV>(s, a, acc, L); break;
            case CT_NABLA2: acc = chain_segment<CT_NABLA2>(s, a, acc, L); break;
            default: acc = chain_segment<CT_NDSQ>(s, a, acc, L); break;
        }
    }
    if (threadIdx.x == 0) *c.out = acc;
}

// The edge step from its three sums (main.c:329).
__global__ void k_chain_edge(ChainArgs a) {
    Scalars *sc = a.sc;
    if (sc->edge_done || sc->converged) return;
    sc->e_c = sc->e_nd / (a.alpha * sc->e_nd2 + a.beta * a.eps * sc->e_nnd + (a.beta / (4 * a.eps)) * sc->e_nd);
}

void launch_chains(hipStream_t st, const ChainArgs &a) {
    MI_REQUIRE(a.nchains >= 1 && a.nchains <= 4, MI_E_ARG, "1 to 4 sums per launch");
    k_chains<<<a.nchains, kChainThreads, 0, st>>>(a);
    MI_HIP(hipGetLastError());
    if (a.edge_c) {
        k_chain_edge<<<1, 1, 0, st>>>(a);
        MI_HIP(hipGetLastError());
    }
}

ChainSeg seg(int term, int64_t n, const double *a, const double *b = nullptr) { return ChainSeg{term, n, a, b}; }
ChainDesc chain(double *out, ChainSeg s0) {
    ChainDesc c{};
    c.seg[0] = s0;
    c.nseg = 1;
    c.out = out;
    return c;
}
ChainDesc chain(double *out, ChainSeg s0, ChainSeg s1) {
    ChainDesc c = chain(out, s0);
    c.seg[1] = s1;
    c.nseg = 2;
    return c;
}

// ---------------------------------------------------------------------------
// Host construction of the lists.

template <typename T>
void upload_vec(DevBuf<T> &b, const std::vector<T> &h, hipStream_t st) {
    b.alloc(std::max<size_t>(h.size(), 1));
    if (!h.empty()) MI_HIP(hipMemcpyAsync(b.p, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice, st));
}

void build_lists(SeqLists &L, const std::vector<int64_t> &ptr, const std::vector<uint32_t> &oth,
                 const std::vector<double> &len, hipStream_t st) {
    const int64_t items = (int64_t)ptr.size() - 1;
    const int64_t groups = (items + kWave - 1) / kWave;
    std::vector<int64_t> base(groups);
    std::vector<int32_t> steps(groups), cnt(items);
    int64_t total = 0;
    for (int64_t gi = 0; gi < groups; ++gi) {
        int64_t most = 0;
        for (int64_t i = gi * kWave; i < std::min(items, (gi + 1) * kWave); ++i) {
            cnt[i] = (int32_t)(ptr[i + 1] - ptr[i]);
            most = std::max<int64_t>(most, cnt[i]);
        }
        MI_REQUIRE(most < (int64_t)1 << 30, MI_E_LIMIT, "entry list too long");
        steps[gi] = (int32_t)((most + 3) / 4 * 4);
        base[gi] = total;
        total += (int64_t)steps[gi] * kWave;
    }
    std::vector<uint32_t> ho((size_t)total, 0u);
    std::vector<double> hl((size_t)total, 0.0);
    for (int64_t i = 0; i < items; ++i) {
        const int64_t b = base[i / kWave] + i % kWave;
        for (int64_t t = 0; t < cnt[i]; ++t) {
            ho[b + t * kWave] = oth[ptr[i] + t];
            hl[b + t * kWave] = len[ptr[i] + t];
        }
    }
    L.items = items;
    upload_vec(L.base, base, st);
    upload_vec(L.steps, steps, st);
    upload_vec(L.cnt, cnt, st);
    upload_vec(L.other, ho, st);
    upload_vec(L.len, hl, st);
    MI_HIP(hipStreamSynchronize(st));
}

template <typename T>
std::vector<T> download(const T *p, int64_t n, hipStream_t st) {
    std::vector<T> h((size_t)n);
    if (n > 0) MI_HIP(hipMemcpyAsync(h.data(), p, n * sizeof(T), hipMemcpyDeviceToHost, st));
    MI_HIP(hipStreamSynchronize(st));
    return h;
}

}  // namespace

size_t seq_bytes(const SeqMatrix *q) { return q ? q->bytes() : 0; }

const SeqMatrix &get_seq(hipStream_t st, Matrix &m) {
    if (m.seq) return *m.seq;
    MI_REQUIRE(m.S == 1, MI_E_STATE, "reference-order lists need a one-subset matrix");
    auto q = std::make_shared<SeqMatrix>();
    std::vector<int64_t> ptr;
    std::vector<uint32_t> oth;
    std::vector<double> len;
    if (m.g.beam == MI_BEAM_GOLDENC) {
        goldenc_lists(false, ptr, oth, len);
        build_lists(q->rows, ptr, oth, len, st);
        goldenc_lists(true, ptr, oth, len);
        build_lists(q->pixels, ptr, oth, len, st);
    } else {
        // The tracer's lengths: double for the fan beams, float (stored
        // widened) for the parallel beam.
        MI_REQUIRE(m.has_csr && (m.has64 || m.g.beam == MI_BEAM_PARALLEL), MI_E_STATE,
                   "reference-order lists need the tracer's CSR / CSC");
        auto lengths = [&](const DevBuf<double> &l64, const DevBuf<float> &l32) {
            if (m.has64) return download(l64.p, m.nnz, st);
            const std::vector<float> f = download(l32.p, m.nnz, st);
            return std::vector<double>(f.begin(), f.end());
        };
        ptr = download(m.rowptr.p, m.nrows + 1, st);
        oth = download(m.idx.p, m.nnz, st);
        len = lengths(m.len64, m.len32);
        build_lists(q->rows, ptr, oth, len, st);
        ptr = download(m.colptr.p, (int64_t)m.npix + 1, st);
        oth = download(m.crow.p, m.nnz, st);
        len = lengths(m.clen64, m.clen32);
        build_lists(q->pixels, ptr, oth, len, st);
    }
    m.seq = q;
    return *m.seq;
}

template <typename T>
void seq_forward(hipStream_t st, const SeqMatrix &q, const T *x, T *out, const T *g, T *resid) {
    const SeqView L = view_of(q.rows);
    const unsigned grid = (unsigned)((L.items + kBlock - 1) / kBlock);
    if (g) k_seq_fp<T, true><<<grid, kBlock, 0, st>>>(L, x, out, g, resid);
    else k_seq_fp<T, false><<<grid, kBlock, 0, st>>>(L, x, out, nullptr, nullptr);
    MI_HIP(hipGetLastError());
}

template <typename T>
void seq_backproject(hipStream_t st, const SeqMatrix &q, int nx, int ny, const T *r, const T *u, const T *v,
                     double alpha, double eps, T *d) {
    const SeqView L = view_of(q.pixels);
    MI_REQUIRE(L.items == (int64_t)nx * ny, MI_E_STATE, "pixel lists do not match the image");
    const unsigned grid = (unsigned)((L.items + kBlock - 1) / kBlock);
    k_seq_bp<T><<<grid, kBlock, 0, st>>>(L, nx, ny, r, u, v, alpha, eps, d);
    MI_HIP(hipGetLastError());
}

template void seq_forward<float>(hipStream_t, const SeqMatrix &, const float *, float *, const float *, float *);
template void seq_forward<double>(hipStream_t, const SeqMatrix &, const double *, double *, const double *,
                                  double *);
template void seq_backproject<float>(hipStream_t, const SeqMatrix &, int, int, const float *, const float *,
                                     const float *, double, double, float *);
template void seq_backproject<double>(hipStream_t, const SeqMatrix &, int, int, const double *, const double *,
                                      const double *, double, double, double *);

// origin/GoldenC/src/main.c:81-257.  gen[] slots: 0 AT_f, 2 normAp, 3 nV,
// 4 pSkalard, 5 max |c1 p|, 6 AdSkalarAp.  Returns the CG iterations run;
// *why: 0 iteration cap, 1 IM_Tol, 2 unstable (reverted).
int gc_image_step_ordered(mi_context *ctx, Matrix &m, JobState<double> &js, double alpha, double eps,
                          int iter_image, int *why) {
    const hipStream_t st = ctx->stream;
    const SeqMatrix &q = get_seq(st, m);
    const int nx = js.nx, ny = js.ny;
    const int64_t npix = js.npix, nrows = js.nrows;
    const int64_t nint = (nx > 2 && ny > 2) ? (int64_t)(nx - 2) * (ny - 2) : 0;
    Scalars *sc = js.sc.p;
    const RedBuf rb = js.rb();
    const double inf = std::numeric_limits<double>::infinity();
    const int cadence = (int)(iter_image / 2 + 0.0001);
    const size_t ib = npix * sizeof(double);
    ChainArgs ca{};
    ca.nx = nx;
    ca.ny = ny;
    ca.alpha = alpha;
    ca.eps = eps;
    // AT_f = sum (Af - g)^2 over [view][bin], then + the interior energy.
    auto energy = [&] {
        ca.nchains = 1;
        ca.c[0] = chain(&sc->gen[0], seg(CT_SQDIFF, nrows, js.af.p, js.g.p), seg(CT_REG_INT, nint, js.u.p, js.v.p));
        launch_chains(st, ca);
    };
    int reason = 0, ran = 0;

    seq_forward(st, q, js.u.p, js.af.p, js.g.p, js.r.p);
    seq_backproject(st, q, nx, ny, js.r.p, js.u.p, js.v.p, alpha, eps, js.d.p);
    energy();
    MI_HIP(hipMemcpyAsync(js.p.p, js.d.p, ib, hipMemcpyDeviceToDevice, st));
    Scalars h = js.read_scalars(st);
    double at_old = h.gen[0];
    for (int k = 1; k <= iter_image; ++k) {
        ran = k;
        seq_forward(st, q, js.p.p, js.q.p);
        ca.nchains = 3;
        ca.c[0] = chain(&sc->gen[3], seg(CT_NV, npix, js.p.p, js.v.p));
        ca.c[1] = chain(&sc->gen[4], seg(CT_DOT, npix, js.p.p, js.d.p));
        ca.c[2] = chain(&sc->gen[2], seg(CT_SQ, nrows, js.q.p));
        launch_chains(st, ca);
        h = js.read_scalars(st);
        const double nap = h.gen[2];
        const double c1 = h.gen[4] / (nap + alpha * h.gen[3]);
        const unsigned grid = launch_axpy<double>(st, npix, js.u.p, js.p.p, nullptr, c1, -inf, inf, js.t.p,
                                                  rb.slot(5));
        FinArgs f{};
        f.op = FIN_STORE;
        f.nin = 1;
        f.in[0] = rb.slot(5);
        f.n[0] = (int)grid;
        f.is_max[0] = 1;
        f.dst = &sc->gen[5];
        launch_finalize(st, f);
        // The reference takes k % 0 when iter_image < 2 (undefined); no
        // median is applied then.
        if (cadence > 0 && k % cadence == 0) {
            launch_median<double>(st, nx, ny, js.u.p, js.w.p);
            MI_HIP(hipMemcpyAsync(js.u.p, js.w.p, ib, hipMemcpyDeviceToDevice, st));
        }
        h = js.read_scalars(st);
        if (k == iter_image) { reason = 0; break; }
        if (h.gen[5] < 1e-5) { reason = 1; break; }
        seq_forward(st, q, js.u.p, js.af.p);
        energy();
        h = js.read_scalars(st);
        const double at_new = h.gen[0];
        if (1.1 * at_old < at_new && 1 < k) {
            MI_HIP(hipMemcpyAsync(js.u.p, js.t.p, ib, hipMemcpyDeviceToDevice, st));
            reason = 2;
            break;
        }
        at_old = at_new;
        // r -= c1 q  (r + (-c1) q rounds the same way)
        launch_axpy<double>(st, nrows, js.r.p, js.q.p, nullptr, -c1, -inf, inf, nullptr, nullptr);
        seq_backproject(st, q, nx, ny, js.r.p, js.u.p, js.v.p, alpha, eps, js.d.p);
        seq_forward(st, q, js.d.p, js.af.p);
        ca.nchains = 1;
        ca.c[0] = chain(&sc->gen[6], seg(CT_DOT, nrows, js.af.p, js.q.p));
        launch_chains(st, ca);
        h = js.read_scalars(st);
        const double c2 = -h.gen[6] / nap;
        launch_xpby<double>(st, npix, js.p.p, js.d.p, c2);
    }
    MI_HIP(hipStreamSynchronize(st));
    if (why) *why = reason;
    return ran;
}

// origin/GoldenC/src/main.c:259-360 on js.v given js.u; n in js.w, the
// direction in js.d.  No host round trip: the step size and the early stop
// live in the job's Scalars.
void gc_edge_step_ordered(mi_context *ctx, JobState<double> &js, double alpha, double beta, double eps,
                          int iter_edge) {
    const hipStream_t st = ctx->stream;
    const int nx = js.nx, ny = js.ny;
    const int64_t npix = js.npix;
    ChainArgs ca{};
    ca.nx = nx;
    ca.ny = ny;
    ca.alpha = alpha;
    ca.beta = beta;
    ca.eps = eps;
    ca.edge_c = 1;
    ca.sc = js.sc.p;
    ca.nchains = 3;
    ca.c[0] = chain(&ca.sc->e_nnd, seg(CT_NABLA2, npix, js.d.p));
    ca.c[1] = chain(&ca.sc->e_nd, seg(CT_SQ, npix, js.d.p));
    ca.c[2] = chain(&ca.sc->e_nd2, seg(CT_NDSQ, npix, js.w.p, js.d.p));
    launch_pass_begin(st, js.sc.p);
    for (int k = 0; k < iter_edge; ++k) {
        launch_edge_grad_n<double>(st, nx, ny, js.u.p, js.v.p, js.d.p, js.w.p, alpha, beta, eps, js.sc.p);
        launch_chains(st, ca);
        launch_edge_update<double>(st, js.rb(), nx, ny, js.v.p, js.d.p, js.sc.p);
    }
    MI_HIP(hipStreamSynchronize(st));
}

}  // namespace mi
