// Reference-order FP64 operators and the GoldenC CG / SD drivers built on
// them (see ordered.hpp).  Every sum here is added in the order the
// reference program adds it, so results equal the reference's bit for bit:
//   * A: one lane per ray sums its products in the order proj.c emits them;
//   * AStar: one lane per pixel, likewise;
//   * energies, norms, inner products: the running double's value after
//     adding the terms one by one in row-major order (k_chain_scan).
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
//
// What bounds it: the gathers, whose 64 lanes touch about as many lines (a
// list's order follows the reference's tiles, not its neighbours'), and with two
// to four waves a SIMD (512 x 512 pixels, 180 views of 767 bins: 2160 waves for
// A, 4096 for AStar) their latency.  A lane so has kSeqAhead gathers in flight
// and the entries of the rows behind them: A 279 -> 262 us, AStar 174 -> 160,
// against four of each and none ahead.
constexpr int kSeqAhead = 16;
template <typename T>
__device__ __forceinline__ T seq_item_sum(const SeqView &L, int64_t i, const T *__restrict__ x) {
    const int64_t gi = i >> 6;
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t b = L.base[gi];
    const int steps = L.steps[gi];
    const int c = i < L.items ? L.cnt[i] : 0;
    T s = T(0);
    uint32_t k[kSeqAhead];
    T l[kSeqAhead];
    auto fetch = [&](int t) {   // past the list: its last row again
#pragma unroll
        for (int j = 0; j < kSeqAhead; ++j) {
            const int64_t at = b + (int64_t)min(t + j, steps - 1) * kWave + lane;
            k[j] = L.other[at];
            l[j] = (T)L.len[at];
        }
    };
    if (steps > 0) fetch(0);
    for (int t = 0; t < steps; t += kSeqAhead) {
        T xv[kSeqAhead], lv[kSeqAhead];
#pragma unroll
        for (int j = 0; j < kSeqAhead; ++j) {
            xv[j] = x[k[j]];
            lv[j] = l[j];
        }
        if (t + kSeqAhead < steps) fetch(t + kSeqAhead);
#pragma unroll
        for (int j = 0; j < kSeqAhead; ++j)
            if (t + j < c) s = s + xv[j] * lv[j];
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

// Folding the terms in index order, rounding after every add as the
// reference's loop does, need not be a serial chain.  While the running sum
// acc stays inside one binade, adding a term t moves it by t rounded to acc's
// own unit in the last place, whatever acc's bits are, unless t lies exactly
// halfway between two multiples of it (then ties-to-even looks at acc).  So
// per chunk of 64 terms the rounded terms are integers that may be added in
// any order, and the chunks' sums are applied in order as long as (a) no term
// is a tie, infinite, NaN or 2^50 units or more, and (b) acc plus the chunk's
// positive terms stays below the binade's upper end and acc plus its negative
// ones (each up to half a unit more than its rounded value) above the lower
// end.
//
// Three launches.  k_chain_terms computes all terms and their plain sums,
// k_chain_records rounds each chunk for the binade that the plain sums put
// acc in, and k_chain_scan, one wave per sum, applies the records, 64 x 1024
// terms at a time where all of them hold.  A record whose binade is not acc's
// (the plain sum may be off near a binade's end), or that fails (a) or (b), is
// folded term by term; acc's binade changes about log2(n) times, so a sum of
// 4e5 terms folds some 25 chunks of 6500.  The result does not depend on the
// plain sums: they only choose which chunks are folded.
//
// Bounded by the scan's folds and their latency.  Measured over the sums of
// one GoldenC alternation (2.6e5 to 5.2e5 terms): 63 us for the three
// launches, against 696 us with one workgroup per sum (4096 terms a step)
// and 5189 us (13 ns a term) with one wave that added each term from its lane.
constexpr int kChunk = kWave, kSupChunks = 16, kSup = kChunk * kSupChunks;
constexpr long long kUnit = (long long)1 << 52, kNoLow = (long long)1 << 61;

struct ChainRec {
    long long sum, pos, low;   // sum; bounds of the partial sums above and below (kNoLow: no negative term)
    int key;                   // sign and exponent of the running sum that it is rounded for
    int flags;                 // REC_BAD: fold term by term; REC_ZERO: all terms are zero
};
enum { REC_BAD = 1, REC_ZERO = 2 };
// Scratch of one sum (sups groups of kSup terms).
struct ChainBuf {
    double *terms, *chunk, *sup;   // the terms; plain sums per chunk and per group
    ChainRec *rec, *srec;
    int64_t sups;
};
struct ChainScratch {
    ChainBuf c[4];
};

__device__ __forceinline__ int64_t chain_terms(const ChainSeg &s) { return s.term == CT_NABLA2 ? 2 * s.n : s.n; }

__device__ __forceinline__ double chain_value(const ChainSeg &s, const ChainArgs &a, int64_t e) {
    double t = 0.0, t1 = 0.0;
    switch (s.term) {
        case CT_SQDIFF: chain_term<CT_SQDIFF>(s, a, e, t, t1); return t;
        case CT_SQ: chain_term<CT_SQ>(s, a, e, t, t1); return t;
        case CT_DOT: chain_term<CT_DOT>(s, a, e, t, t1); return t;
        case CT_REG_INT: chain_term<CT_REG_INT>(s, a, e, t, t1); return t;
        case CT_NV: chain_term<CT_NV>(s, a, e, t, t1); return t;
        case CT_NABLA2: chain_term<CT_NABLA2>(s, a, e >> 1, t, t1); return e & 1 ? t1 : t;
        default: chain_term<CT_NDSQ>(s, a, e, t, t1); return t;
    }
}

__device__ __forceinline__ bool chain_skip(const ChainArgs &a) {
    return a.edge_c && (a.sc->edge_done || a.sc->converged);
}

// Workgroup (x, y): group x of sum y; wave w its chunks 4 w .. 4 w + 3, one
// term per lane (zeros past the end: adding +0 leaves every running sum but
// -0 as it is, and the sums start at +0).
__global__ __launch_bounds__(kBlock) void k_chain_terms(ChainArgs a, ChainScratch q) {
    __shared__ double lds[kBlock / kWave];
    if (chain_skip(a)) return;
    const ChainDesc &c = a.c[blockIdx.y];
    const ChainBuf &b = q.c[blockIdx.y];
    const int64_t g = blockIdx.x;
    if (g >= b.sups) return;
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    const int64_t n0 = chain_terms(c.seg[0]), n = n0 + (c.nseg > 1 ? chain_terms(c.seg[1]) : 0);
    constexpr int PER = kSupChunks / (kBlock / kWave);
    double t[PER], all = 0.0;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int64_t e = g * kSup + (wv * PER + k) * kChunk + lane;
        t[k] = e >= n ? 0.0 : (e < n0 ? chain_value(c.seg[0], a, e) : chain_value(c.seg[1], a, e - n0));
    }
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int64_t ch = g * kSupChunks + wv * PER + k;
        b.terms[ch * kChunk + lane] = t[k];
        const double s = group_sum<kWave>(t[k]);
        if (lane == 0) b.chunk[ch] = s;
        all += s;
    }
    if (lane == 0) lds[wv] = all;
    __syncthreads();
    if (threadIdx.x == 0) b.sup[g] = (lds[0] + lds[1]) + (lds[2] + lds[3]);
}

__device__ __forceinline__ long long wave_sum_i64(long long x) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) x += __shfl_xor(x, o, kWave);
    return x;
}

__device__ __forceinline__ int chain_key(double acc) { return (int)(__double_as_longlong(acc) >> 52) & 0xfff; }
// The scale 2^(52 - e) of a running sum of exponent e is a normal number too.
__device__ __forceinline__ bool chain_normal(int key) { return (key & 0x7ff) >= 53 && (key & 0x7ff) <= 2000; }

__global__ __launch_bounds__(kBlock) void k_chain_records(ChainArgs a, ChainScratch q) {
    __shared__ double lds[kBlock / kWave];
    __shared__ ChainRec recs[kSupChunks];
    if (chain_skip(a)) return;
    const ChainBuf &b = q.c[blockIdx.y];
    const int64_t g = blockIdx.x;
    if (g >= b.sups) return;
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    constexpr int PER = kSupChunks / (kBlock / kWave);
    double t[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) t[k] = b.terms[(g * kSupChunks + wv * PER + k) * kChunk + lane];
    double mine = 0.0;
    for (int64_t i = threadIdx.x; i < g; i += kBlock) mine += b.sup[i];
    mine = group_sum<kWave>(mine);
    if (lane == 0) lds[wv] = mine;
    __syncthreads();
    double before = (lds[0] + lds[1]) + (lds[2] + lds[3]);
    for (int k = 0; k < wv * PER; ++k) before += b.chunk[g * kSupChunks + k];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int key = chain_key(before);
        const double scale = __longlong_as_double(((long long)(2098 - (key & 0x7ff)) << 52) | ((long long)(key >> 11) << 63));
        constexpr double M = 6755399441055744.0;   // 1.5 2^52: adding it rounds to an integer
        const double x = t[k] * scale, r = x + M;
        const long long i = __double_as_longlong(r) - __double_as_longlong(M);
        bool bad = !(fabs(x) < 1125899906842624.0) | (fabs(x - (r - M)) == 0.5) | !chain_normal(key);
        const bool zero = __all(t[k] == 0.0);
        bad = __any(bad);
        ChainRec o{0, 0, kNoLow, key, zero ? REC_ZERO : (bad ? REC_BAD : 0)};
        if (!zero && !bad) {
            const long long p = wave_sum_i64(i > 0 ? i : 0), m = __any(x < 0.0) ? wave_sum_i64(i < 0 ? i : 0) : 0;
            o.sum = p + m;
            o.pos = p;
            if (__any(x < 0.0)) o.low = m - kChunk;
            if (p >= 2 * kUnit || m <= -2 * kUnit) {   // cannot stay in the binade
                o = ChainRec{0, 0, kNoLow, key, REC_BAD};
            }
        }
        if (lane == 0) {
            b.rec[g * kSupChunks + wv * PER + k] = o;
            recs[wv * PER + k] = o;
        }
        before += b.chunk[g * kSupChunks + wv * PER + k];
    }
    __syncthreads();
    if (threadIdx.x == 0) {   // the group as one record, if its chunks are of one binade
        ChainRec o{0, 0, kNoLow, 0, REC_ZERO};
        for (int k = 0; k < kSupChunks; ++k) {
            const ChainRec c = recs[k];
            if (c.flags & REC_ZERO) continue;
            if (o.flags & REC_ZERO) {
                o.flags = 0;
                o.key = c.key;
            }
            if ((c.flags & REC_BAD) || c.key != o.key) o.flags = REC_BAD;
            o.pos = max(o.pos, o.sum + c.pos);
            if (c.low != kNoLow) o.low = min(o.low, o.sum + c.low);
            o.sum += c.sum;
        }
        if (o.pos >= 2 * kUnit || o.low <= -2 * kUnit) o.flags = REC_BAD;
        if (o.flags & REC_BAD) o = ChainRec{0, 0, kNoLow, o.key, REC_BAD};
        b.srec[g] = o;
    }
}

// Applies the records of lanes from .. 63 to acc as far as they hold; returns
// the first lane whose record does not (64: none).
__device__ __forceinline__ int chain_apply(const ChainRec &r, int from, int lane, double &acc) {
    const int key = chain_key(acc);
    const long long bits = __double_as_longlong(acc), A = (bits & (kUnit - 1)) | kUnit;
    const bool zero = lane < from || (r.flags & REC_ZERO);
    long long run = zero ? 0 : r.sum;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const long long up = __shfl_up(run, o, kWave);
        if (lane >= o) run += up;
    }
    const long long at = A + run - (zero ? 0 : r.sum);
    const bool holds = zero || (!(r.flags & REC_BAD) && r.key == key && chain_normal(key) && at + r.pos < 2 * kUnit &&
                                (r.low == kNoLow || at + r.low > kUnit));
    const unsigned long long fail = __ballot(!holds);
    const int f = fail ? __ffsll((long long)fail) - 1 : kWave;
    const long long to = f < kWave ? __shfl(at, f, kWave) : __shfl(A + run, kWave - 1, kWave);
    if (chain_normal(key)) acc = __longlong_as_double((bits & ~(kUnit - 1)) | (to & (kUnit - 1)));
    return f;
}

// One wave per sum.
__global__ __launch_bounds__(kWave) void k_chain_scan(ChainArgs a, ChainScratch q) {
    __shared__ double lt[kSup];
    if (chain_skip(a)) return;
    const ChainBuf &b = q.c[blockIdx.x];
    const int lane = threadIdx.x;
    const ChainRec none{0, 0, kNoLow, 0, REC_ZERO};
    double acc = 0.0;
    ChainRec next = lane < b.sups ? b.srec[lane] : none;
    for (int64_t g0 = 0; g0 < b.sups; g0 += kWave) {
        const ChainRec r = next;
        next = g0 + kWave + lane < b.sups ? b.srec[g0 + kWave + lane] : none;
        for (int from = 0;;) {
            const int f = chain_apply(r, from, lane, acc);
            if (f >= kWave) break;
            // group f chunk by chunk
            const int64_t g = g0 + f;
            const ChainRec c = lane < kSupChunks ? b.rec[g * kSupChunks + lane] : none;
            double t[kSupChunks];
#pragma unroll
            for (int k = 0; k < kSupChunks; ++k) t[k] = b.terms[g * kSup + k * kChunk + lane];
            __syncthreads();
#pragma unroll
            for (int k = 0; k < kSupChunks; ++k) lt[k * kChunk + lane] = t[k];
            __syncthreads();
            for (int at = 0;;) {
                const int k = chain_apply(c, at, lane, acc);
                if (k >= kWave) break;
                const double *x = lt + k * kChunk;   // term by term (all lanes alike)
#pragma unroll 1
                for (int i = 0; i < kChunk; i += 16) {
                    double y[16];
#pragma unroll
                    for (int j = 0; j < 16; ++j) y[j] = x[i + j];
#pragma unroll
                    for (int j = 0; j < 16; ++j) acc = acc + y[j];
                }
                at = k + 1;
            }
            from = f + 1;
        }
    }
    if (lane == 0) *a.c[blockIdx.x].out = acc;
}

// The edge step from its three sums (main.c:329).
__global__ void k_chain_edge(ChainArgs a) {
    Scalars *sc = a.sc;
    if (sc->edge_done || sc->converged) return;
    sc->e_c = sc->e_nd / (a.alpha * sc->e_nd2 + a.beta * a.eps * sc->e_nnd + (a.beta / (4 * a.eps)) * sc->e_nd);
}

// buf: scratch of the sums, grown as needed (the job's, on its stream).
void launch_chains(hipStream_t st, const ChainArgs &a, DevBuf<unsigned char> &buf) {
    MI_REQUIRE(a.nchains >= 1 && a.nchains <= 4, MI_E_ARG, "1 to 4 sums per launch");
    ChainScratch q{};
    int64_t sups[4] = {}, all = 0, most = 1;
    for (int i = 0; i < a.nchains; ++i) {
        int64_t n = 0;
        for (int k = 0; k < a.c[i].nseg; ++k) n += (a.c[i].seg[k].term == CT_NABLA2 ? 2 : 1) * a.c[i].seg[k].n;
        sups[i] = std::max<int64_t>(1, (n + kSup - 1) / kSup);
        all += sups[i];
        most = std::max(most, sups[i]);
    }
    constexpr size_t kPer = sizeof(double) * (kSup + kSupChunks + 1) + sizeof(ChainRec) * (kSupChunks + 1);
    if (buf.n < all * kPer) buf.alloc(all * kPer);
    unsigned char *p = buf.p;
    auto take = [&](size_t bytes) {
        unsigned char *r = p;
        p += bytes;
        return r;
    };
    for (int i = 0; i < a.nchains; ++i) {
        q.c[i].sups = sups[i];
        q.c[i].terms = (double *)take(sups[i] * kSup * sizeof(double));
        q.c[i].chunk = (double *)take(sups[i] * kSupChunks * sizeof(double));
        q.c[i].sup = (double *)take(sups[i] * sizeof(double));
        q.c[i].rec = (ChainRec *)take(sups[i] * kSupChunks * sizeof(ChainRec));
        q.c[i].srec = (ChainRec *)take(sups[i] * sizeof(ChainRec));
    }
    const dim3 grid((unsigned)most, a.nchains);
    k_chain_terms<<<grid, kBlock, 0, st>>>(a, q);
    MI_HIP(hipGetLastError());
    k_chain_records<<<grid, kBlock, 0, st>>>(a, q);
    MI_HIP(hipGetLastError());
    k_chain_scan<<<a.nchains, kWave, 0, st>>>(a, q);
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
        launch_chains(st, ca, js.chain);
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
        launch_chains(st, ca, js.chain);
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
        launch_chains(st, ca, js.chain);
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
        launch_chains(st, ca, js.chain);
        launch_edge_update<double>(st, js.rb(), nx, ny, js.v.p, js.d.p, js.sc.p);
    }
    MI_HIP(hipStreamSynchronize(st));
}

}  // namespace mi
