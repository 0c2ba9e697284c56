// Device helpers shared by the register-resident build kernels
// (build_tiled_kernel.hpp, build_refine_kernel.hpp, build_vjp_tiled.hip,
// fused_build_eval.hip).
#pragma once

#include <algorithm>

#include "internal.hpp"

namespace ddcx {
namespace tiled {

constexpr int kNbMax = 8;   // border (Schur) size limit
constexpr int kLamMax = 64; // lambda couplings limit

// Keeps the scheduler from hoisting the table loads of a whole segment at
// once (which would not fit in registers next to the segment's rows): a
// scheduling barrier after every M rows of an unrolled row loop.
template <int M = 8>
__device__ __forceinline__ void chunk_fence(int i)
{
    if (i % M == M - 1) __builtin_amdgcn_sched_barrier(0);
}

// The border data that a workgroup reads after its sweeps, copied to LDS in
// its prologue so that the border step waits on no global load: the border
// step's matrix, the inverse of the Schur complement, and (in dynamic LDS) the
// Q^-1 gamma blocks.  16-byte aligned like the dynamic LDS behind it: the row table
// is copied there two doubles at a time.
struct alignas(16) BorderLds {
    double m[kLamMax];
    double sinv[kNbMax * kNbMax];
};

template <int NT, bool GAMMA>
__device__ __forceinline__ void stage_border(TiledView const& tv, BorderLds& bl, double* gpad, int tid)
{
    for (int k = tid; k < tv.nb * tv.ncols; k += NT) bl.m[k] = tv.bm[k];
    for (int k = tid; k < tv.nb * tv.nb; k += NT) bl.sinv[k] = tv.sinv[k];
    if constexpr (GAMMA) {
        int const n = tv.ngb * tv.L * tv.nb;
        for (int k = tid; k < n; k += NT) gpad[k] = tv.Gblk[k];
    }
}

// The rows of a segment that lambda couples to the border, to their slots in
// LDS.  A static row loop with a bit test per row, entered only by the one or
// two segments that hold such rows: no register indexing, no scan of the
// couplings.
template <int LB, int L>
__device__ __forceinline__ void gather_coupled(double const (&y)[L], SegBorder const& sb, double (*lamx)[LB], int ln)
{
    static_assert(L <= 32, "one mask bit per row");
    if (sb.mask != 0) {
#pragma unroll
        for (int i = 0; i < L; ++i)
            if ((sb.mask >> i) & 1u) lamx[sb.slot0 + __popc(sb.mask & ((1u << i) - 1u))][ln] = y[i];
    }
}

// Row k of x2 = S^-1 b2 - (S^-1 lambda) y for one line: two short products of
// independent reads, so the rows need no exchange.  (As S^-1 (b2 - lambda y) with
// the couplings in a list, every thread summed the whole right-hand side through
// two dependent LDS reads per coupling, and with a border of 4 to 6 rows the
// others waited: quartic Hermite 203 cells x 65536 139 -> 166 us.)
template <int LB>
__device__ __forceinline__ double border_row(TiledView const& tv, BorderLds const& bl, double const (*b2)[LB],
                                             double const (*lamx)[LB], int k, int ln)
{
    double x = 0.0;
#pragma unroll 4
    for (int j = 0; j < tv.nb; ++j) x = fma(bl.sinv[k * tv.nb + j], b2[j][ln], x);
#pragma unroll 4
    for (int s = 0; s < tv.ncols; ++s) x = fma(-bl.m[k * tv.ncols + s], lamx[s][ln], x);
    return x;
}

// y -= G x2 for one segment's block G, stored column by column (nb columns of
// L rows).  A run-time loop over the columns around a static one over the
// rows: with the kNbMax columns unrolled a uniform cubic spline (nb = 1) spent
// eight times the multiply-adds, in the segments that the whole workgroup
// waits for; variants by column count made the compiler keep several copies
// of y (164 to 179 registers instead of 109 to 125, and spills at 128).
// Short segments have the registers to read four columns ahead.
template <int LB, int L>
__device__ __forceinline__ void apply_gamma(double (&y)[L], const double* G, int nb, double const (*x2s)[LB], int ln)
{
    auto column = [&](int k) {
        double const x = x2s[k][ln];
        const double* g = G + k * L;
#pragma unroll
        for (int i = 0; i < L; ++i) {
            y[i] = fma(-g[i], x, y[i]);
            if constexpr (L >= 16) chunk_fence(i);
        }
    };
    if constexpr (L < 16) {
#pragma unroll 4
        for (int k = 0; k < nb; ++k) column(k);
    } else {
        for (int k = 0; k < nb; ++k) column(k);
    }
}

// doubles of LDS that stage_border's Q^-1 gamma blocks take
inline size_t gamma_lds_doubles(TiledView const& tv) { return size_t(tv.ngb) * tv.L * tv.nb; }

__device__ __forceinline__ int64_t lay(Layout const& L, int64_t r, int64_t l)
{
    if (l < L.inner) return r * L.rs + l * L.is; // one batch dimension: no 64-bit division
    return r * L.rs + (l % L.inner) * L.is + (l / L.inner) * L.os;
}

// physical right-hand-side row i of one line (spline_builder.hpp:949-1033)
__device__ __forceinline__ double rhs_src(BuildView const& bv, const double* vals, Layout const& vl, int64_t vb,
                                          const double* dl, const double* dr, Layout const& dlay, int64_t db, int i)
{
    if (bv.periodic) return vals[vb + int64_t(i) * vl.rs];
    if (i < bv.nbe_l) return bv.bcl == DDCX_HERMITE ? dl[db + int64_t(i) * dlay.rs] * bv.dxpow[i + bv.odd] : 0.0;
    int const nv_end = bv.nbasis - bv.nbe_r;
    if (i < nv_end) return vals[vb + int64_t(i - bv.nbe_l) * vl.rs];
    return bv.bcu == DDCX_HERMITE ? dr[db + int64_t(i - nv_end) * dlay.rs] * bv.dxpow[i - nv_end + bv.odd] : 0.0;
}

// dgetrs on an nb x nb LU (nb <= kNbMax) held in registers
__device__ __forceinline__ void getrs_small(int nb, const double* a, const int* ipiv, double* b)
{
#pragma unroll
    for (int j = 0; j < kNbMax; ++j) {
        if (j < nb) {
            int const p = ipiv[j];
            double bp = 0.0;
#pragma unroll
            for (int k = 0; k < kNbMax; ++k)
                if (k == p) bp = b[k];
            double const bj = b[j];
#pragma unroll
            for (int k = 0; k < kNbMax; ++k)
                if (k == p) b[k] = bj;
            b[j] = bp;
        }
    }
#pragma unroll
    for (int j = 0; j < kNbMax; ++j)
#pragma unroll
        for (int i = j + 1; i < kNbMax; ++i)
            if (i < nb) b[i] = b[i] - b[j] * a[i * nb + j];
#pragma unroll
    for (int j = kNbMax - 1; j >= 0; --j) {
        if (j < nb) {
            b[j] = b[j] / a[j * nb + j];
#pragma unroll
            for (int i = 0; i < j; ++i) b[i] = b[i] - b[j] * a[i * nb + j];
        }
    }
}

// Interpolation-contiguous layouts (IC) stage the tile through LDS in chunks
// of kStageRows rows of all LB lines: each line's rows are read and written
// as contiguous runs, and every thread takes its L rows from LDS.
constexpr int kStageRows = 256;
// the chunk of a K x L tiling: the whole padded line when it is shorter
// (K * L rows; the short tilings have K * L = 128 or 144, so the pitch stays odd)
// and on the small-batch tiles of a few lines, where one chunk has one barrier
// pair and all its loads in flight at once; an odd pitch spreads the LDS banks
constexpr int stage_rows(int kl, int lb) { return kl < kStageRows || lb <= 8 ? kl : kStageRows; }
constexpr int stage_pitch(int kl, int lb) { return stage_rows(kl, lb) | 1; }

// Tile of workgroup b.  A tile of fewer than 16 lines shares its 128-byte
// cache lines with its neighbours in the batch-contiguous layout, and
// consecutive workgroups go to different XCDs, each with its own L2: there the
// eight XCDs take contiguous ranges of tiles instead, equally long but for one.
// The grid is then 8 * ceil(ntiles / 8), and the workgroups without a tile (a
// first line at or past nbatch) leave at once.  (With the last XCD's range cut
// short, a last tile of one line alone in its shader engine took 1.6 times as
// long as a full one: degree 6, 1802 cells x 513 lines, 84 us instead of 50.)
template <int LB>
__device__ __forceinline__ int64_t tile_of(unsigned b, int64_t nbatch)
{
    if constexpr (LB >= 16) return b;
    unsigned const n = unsigned((nbatch + LB - 1) / LB), x = b % 8, i = b / 8;
    if (i >= n / 8 + (x < n % 8)) return n;
    return x * (n / 8) + min(x, n % 8) + i;
}

// Small batches: at most one tile of 8 lines per CU (64 x 16 tiling) or two
// (32 x 8 tiling).  Up to there the 8-line tiles are faster than the 16- and
// 32-line ones, past it their shorter runs cost more than the idle CUs
// (figures in build_tiled_small.hip and build_tiled_short.hip).
inline bool small_batch(int64_t nbatch, int tiles_per_cu) { return nbatch <= 8 * int64_t(tiles_per_cu) * cu_count(); }

template <int LB>
inline unsigned tile_grid(int64_t nbatch)
{
    int64_t const n = (nbatch + LB - 1) / LB;
    return unsigned(LB >= 16 ? n : (n + 7) / 8 * 8);
}

// The tiled kernels address a tile as a workgroup-uniform base plus 32-bit
// per-lane offsets; true when every offset of the batch fits.
inline bool offsets_fit(Layout const& l, int64_t rows, int64_t nbatch)
{
    if (l.rs < 0 || l.is < 0 || l.os < 0 || l.inner < 1) return false;
    if (nbatch > l.inner && l.os < (l.inner - 1) * l.is + 1) return false;
    int64_t const span = rows * l.rs + std::min<int64_t>(nbatch, l.inner) * l.is + l.os;
    return span < (int64_t(1) << 31);
}


// The two sweeps of the main-block solve on a K x L tiling (one thread per
// segment and line, L rows in registers): local pass with a zero incoming
// state, exchange of the outgoing states through LDS, exact incoming state
// from the transfer products, correction by the homogeneous recurrence.
// Row records: the forward sweep reads Lf(KF) at OLF and 1/d at ORDF (FDIV),
// the backward sweep Ub(KB) at OUB and 1/d at ORDB; the records of the full
// row table are [Lf(KF) | Ub(KB) | rDb | rDf (FDIV)].  The forward sweep ends
// with a barrier; the backward sweep does not.
template <int LB, int K, int L, int KF, bool FDIV, int OLF, int ORDF>
__device__ __forceinline__ void tiled_forward(double (&y)[L], const double* T, int RS, const double* Mf, int wf,
                                              double (*ex)[K][LB], int seg, int ln)
{
    double s[KF];
#pragma unroll
    for (int k = 0; k < KF; ++k) s[k] = 0.0;
#pragma unroll
    for (int i = 0; i < L; ++i) {
        const double* R = T + i * RS;
        double t = y[i];
#pragma unroll
        for (int k = KF; k >= 1; --k) t = fma(-s[k - 1], R[OLF + k - 1], t);
        if constexpr (FDIV) t = t * R[ORDF];
        y[i] = t;
#pragma unroll
        for (int k = KF - 1; k > 0; --k) s[k] = s[k - 1];
        s[0] = t;
        chunk_fence(i);
    }
#pragma unroll
    for (int k = 0; k < KF; ++k) ex[k][seg][ln] = s[k];
    __syncthreads();
    double in[KF];
#pragma unroll
    for (int k = 0; k < KF; ++k) in[k] = 0.0;
    for (int w = 1; w <= wf; ++w) {
        int const src = seg - w;
        if (src >= 0) {
            const double* m = Mf + (seg * wf + (w - 1)) * (KF * KF);
#pragma unroll
            for (int a = 0; a < KF; ++a)
#pragma unroll
                for (int b = 0; b < KF; ++b) in[a] = fma(m[a * KF + b], ex[b][src][ln], in[a]);
        }
    }
    if (seg > 0) {
        // rows += homogeneous forward recurrence started from the incoming state
#pragma unroll
        for (int i = 0; i < L; ++i) {
            const double* R = T + i * RS;
            double t = 0.0;
#pragma unroll
            for (int k = KF; k >= 1; --k) t = fma(-in[k - 1], R[OLF + k - 1], t);
            if constexpr (FDIV) t = t * R[ORDF];
            y[i] += t;
#pragma unroll
            for (int k = KF - 1; k > 0; --k) in[k] = in[k - 1];
            in[0] = t;
            chunk_fence(i);
        }
    }
    __syncthreads();
}

template <int LB, int K, int L, int KB, bool BDIVF, int OUB, int ORDB>
__device__ __forceinline__ void tiled_backward(double (&y)[L], const double* T, int RS, const double* Mb, int wb,
                                               double (*ex)[K][LB], int seg, int ln)
{
    double s[KB];
#pragma unroll
    for (int k = 0; k < KB; ++k) s[k] = 0.0;
#pragma unroll
    for (int i = L - 1; i >= 0; --i) {
        const double* R = T + i * RS;
        double t;
        if constexpr (BDIVF) {
            t = fma(-s[0], R[OUB], y[i] * R[ORDB]);
        } else {
            t = y[i];
#pragma unroll
            for (int k = KB; k >= 1; --k) t = fma(-s[k - 1], R[OUB + k - 1], t);
            t = t * R[ORDB];
        }
        y[i] = t;
#pragma unroll
        for (int k = KB - 1; k > 0; --k) s[k] = s[k - 1];
        s[0] = t;
        chunk_fence(i);
    }
#pragma unroll
    for (int k = 0; k < KB; ++k) ex[k][seg][ln] = s[k];
    __syncthreads();
    double in[KB];
#pragma unroll
    for (int k = 0; k < KB; ++k) in[k] = 0.0;
    for (int w = 1; w <= wb; ++w) {
        int const src = seg + w;
        if (src < K) {
            const double* m = Mb + (seg * wb + (w - 1)) * (KB * KB);
#pragma unroll
            for (int a = 0; a < KB; ++a)
#pragma unroll
                for (int b = 0; b < KB; ++b) in[a] = fma(m[a * KB + b], ex[b][src][ln], in[a]);
        }
    }
    if (seg + 1 < K) {
        // rows += homogeneous backward recurrence started from the incoming state
#pragma unroll
        for (int i = L - 1; i >= 0; --i) {
            const double* R = T + i * RS;
            double t;
            if constexpr (BDIVF) {
                t = -in[0] * R[OUB];
            } else {
                t = 0.0;
#pragma unroll
                for (int k = KB; k >= 1; --k) t = fma(-in[k - 1], R[OUB + k - 1], t);
                t = t * R[ORDB];
            }
            y[i] += t;
#pragma unroll
            for (int k = KB - 1; k > 0; --k) in[k] = in[k - 1];
            in[0] = t;
            chunk_fence(i);
        }
    }
}

template <int LB, int K, int L, int KF, int KB, bool FDIV, bool BDIVF, int KE>
__device__ __forceinline__ void tiled_sweeps(double (&y)[L], const double* T, int RS, const double* Mf, int wf,
                                             const double* Mb, int wb, double (*ex)[K][LB], int seg, int ln)
{
    tiled_forward<LB, K, L, KF, FDIV, 0, KF + KB + 1>(y, T, RS, Mf, wf, ex, seg, ln);
    tiled_backward<LB, K, L, KB, BDIVF, KF, KF + KB>(y, T, RS, Mb, wb, ex, seg, ln);
}

// The small-batch tiles (4 and 8 lines) also keep the
// segment transfer products in LDS: the two carry steps then wait on no
// global load.  The larger tiles have no LDS to spare for them.
constexpr bool transfer_in_lds(int lb) { return lb <= 8; }
inline size_t transfer_doubles(TiledView const& tv)
{
    return size_t(tv.K) * (tv.wf * tv.kf * tv.kf + tv.wb * tv.kb * tv.kb);
}

template <int NT>
__device__ __forceinline__ void stage_transfer(TiledView const& tv, double* dst, int tid)
{
    int const nf = tv.K * tv.wf * tv.kf * tv.kf, nb = tv.K * tv.wb * tv.kb * tv.kb;
    for (int k = tid; k < nf; k += NT) dst[k] = tv.Mf[k];
    for (int k = tid; k < nb; k += NT) dst[nf + k] = tv.Mb[k];
}

// The row table to LDS: every load of a thread in flight before its first
// LDS write (RS <= 10 doubles per row)
template <int NT, int ROWS, int RS>
__device__ __forceinline__ void stage_table(const double* rt, double* dst, int tid)
{
    static_assert(ROWS * RS % 2 == 0);
    constexpr int N2 = ROWS * RS / 2, PER = (N2 + NT - 1) / NT;
    const double2* src = reinterpret_cast<const double2*>(rt);
    double2* d2 = reinterpret_cast<double2*>(dst);
    constexpr int CH = PER < 16 ? PER : 16;
    for (int k0 = 0; k0 < PER; k0 += CH) {
        double2 v[CH];
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            int const idx = tid + (k0 + k) * NT;
            v[k] = src[idx < N2 ? idx : N2 - 1];
        }
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            int const idx = tid + (k0 + k) * NT;
            if (idx < N2) d2[idx] = v[k];
        }
    }
}

// Split staging of the row table, for tables that do not fit LDS whole:
// the fields one sweep reads, copied from the full records (stride RS) into
// compact records in LDS ([Lf(KF) | rDf] for the forward sweep, [Ub(KB) |
// rDb] for the backward one).  The caller synchronises.
template <int NT, int KF, int KB, bool FDIV, bool FORWARD>
__device__ __forceinline__ void stage_half(const double* __restrict__ rt, int RS, int rows, double* dst, int tid)
{
    constexpr int W = FORWARD ? KF + (FDIV ? 1 : 0) : KB + 1;
    for (int e = tid; e < rows * W; e += NT) {
        int const r = e / W, f = e % W;
        int src;
        if constexpr (FORWARD) src = f < KF ? f : KF + KB + 1;
        else src = f < KB ? KF + f : KF + KB;
        dst[e] = rt[size_t(r) * RS + src];
    }
}
} // namespace tiled
} // namespace ddcx
