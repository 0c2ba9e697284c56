// Fused batched build + evaluation: SplineBuilder::operator()
// (spline_builder.hpp:905) followed by SplineEvaluator::operator()
// (spline_evaluator.hpp:263) on the same lines, in one kernel.  A workgroup
// solves LB lines with the register-resident tiled sweeps (build_tiled_kernel.hpp,
// 16-row segments), writes the coefficients into an LDS tile that reuses the
// row table's space, and evaluates every point of those lines from it
// (eval_tiled.hip's batch-contiguous mapping).  The coefficients go to HBM only
// when the caller asks for them, so a step reads vals and coords and writes
// the values: 24 bytes per point-and-row instead of the 40 of the two calls.
#include "tiled_common.hpp"

namespace ddcx {

namespace {

using namespace tiled;

template <int LB, int K, int L, int KF, int KB, bool FDIV, bool BDIVF, int D, bool MLDS>
__global__ void __launch_bounds__(LB* K, 4) fused_build_eval_kernel(TiledView tv, BuildView bv, BSplinesView b,
                                                                Rules1D rules, const double* __restrict__ vals,
                                                                Layout vl, const double* __restrict__ dl,
                                                                const double* __restrict__ dr, Layout dlay,
                                                                double* __restrict__ coef, Layout cl,
                                                                double* __restrict__ out,
                                                                const double* __restrict__ coords, Layout pl,
                                                                int64_t npts, int64_t nbatch,
                                                                const double* __restrict__ fpts,
                                                                const double* __restrict__ fshift)
{
    constexpr int KE = KF > KB ? KF : KB;
    constexpr int NT = LB * K;
    constexpr int ROWS = NT / LB; // point rows per pass (= K)
    constexpr int U = 8;
    __shared__ double ex[KE][K][LB];
    __shared__ double lamx[kLamMax][LB];
    __shared__ double b2s[kNbMax][LB];
    // the border's solution, in the space of the sweeps' exchange (over when it is
    // written); K >= kNbMax
    double(*const x2s)[LB] = ex[0];
    // row table, Q^-1 gamma blocks, segment transfer products (MLDS) and border
    // data during the build, coefficient tile (size x LB) after
    alignas(16) extern __shared__ double dyn[];

    int const tid = threadIdx.x;
    int const ln = tid % LB;
    int const seg = tid / LB;
    int64_t const line0 = tile_of<LB>(blockIdx.x, nbatch) * LB;
    if (LB < 16 && line0 >= nbatch) return; // whole workgroup
    int64_t const line = line0 + ln;
    bool const active = line < nbatch;
    int64_t const lc = active ? line : line0;
    int64_t const vb = lay(vl, 0, lc);
    int64_t const cb = lay(cl, 0, lc);
    int const r0 = seg * L;
    int const nq = tv.nq;
    constexpr int RS = KF + KB + 1 + (FDIV ? 1 : 0); // row record length, fixed by the band shape
    const double* __restrict__ vwg = vals + lay(vl, 0, line0);
    uint32_t const vlo = uint32_t(vb - lay(vl, 0, line0)) + uint32_t(tv.q0 + r0) * uint32_t(vl.rs);
    uint32_t const vrs = uint32_t(vl.rs);
    bool const store = coef != nullptr;

    // ---------------- build ----------------
    double y[L];
    if (r0 + L <= nq) {
#pragma unroll
        for (int i = 0; i < L; ++i) y[i] = __builtin_nontemporal_load(&vwg[vlo + uint32_t(i) * vrs]);
    } else {
        uint32_t const vl0 = vlo - uint32_t(r0) * vrs; // row q0 of this line
#pragma unroll
        for (int i = 0; i < L; ++i) {
            double const v = __builtin_nontemporal_load(&vwg[vl0 + uint32_t(min(r0 + i, nq - 1)) * vrs]);
            y[i] = r0 + i < nq ? v : 0.0;
        }
    }
    // the border rows' right-hand side and the segment's part of the border
    // step, read with the tile
    double b2 = 0.0;
    if (seg < tv.nb && active)
        b2 = rhs_src(bv, vals, vl, vb, dl, dr, dlay, lay(dlay, 0, lc), seg < tv.top ? seg : tv.nq + seg);
    SegBorder const sb = tv.seg[seg];
    double* const gpad = dyn + K * L * RS;
    double* const mtr = gpad + tv.ngb * L * tv.nb;
    BorderLds& bl = *reinterpret_cast<BorderLds*>(mtr + (MLDS ? K * (tv.wf * KF * KF + tv.wb * KB * KB) : 0));
    {
        stage_table<NT, K * L, RS>(tv.rt, dyn, tid);
        if constexpr (MLDS) stage_transfer<NT>(tv, mtr, tid);
        stage_border<NT, true>(tv, bl, gpad, tid);
        if (seg < tv.nb) b2s[seg][ln] = b2;
        __syncthreads();
    }
    tiled_sweeps<LB, K, L, KF, KB, FDIV, BDIVF, KE>(y, dyn + r0 * RS, RS, MLDS ? mtr : tv.Mf, tv.wf,
                                                    MLDS ? mtr + K * tv.wf * KF * KF : tv.Mb, tv.wb, ex, seg, ln);

    int const nb = tv.nb;
    int const off = bv.offset;
    int const nbas = bv.nbasis;
    if (nb > 0) {
        gather_coupled<LB, L>(y, sb, lamx, ln);
        __syncthreads();
        if (seg < nb) x2s[seg][ln] = border_row<LB>(tv, bl, b2s, lamx, seg, ln);
        __syncthreads();
        if (sb.gblk >= 0) apply_gamma<LB>(y, gpad + sb.gblk * L * nb, nb, x2s, ln);
    }
    __syncthreads(); // the row table is dead from here on

    // ---------------- coefficients: LDS tile (and HBM when asked) ----------------
    double* tile = dyn;
    auto put = [&](int row, double v) {
        tile[row * LB + ln] = v;
        if (store && active) __builtin_nontemporal_store(v, &coef[cb + int64_t(row) * cl.rs]);
    };
#pragma unroll
    for (int i = 0; i < L; ++i) {
        int const prow = tv.top + r0 + i;
        if (r0 + i < nq) {
            put(prow + off, y[i]);
            if (bv.periodic) {
                if (prow + off - nbas >= 0) put(prow + off - nbas, y[i]);
                if (prow + off + nbas < nbas + bv.degree) put(prow + off + nbas, y[i]);
            }
        }
    }
    if (seg < nb) {
        double const v = x2s[seg][ln];
        int const j = (seg < tv.top ? seg : nq + seg) + off;
        put(j, v);
        if (bv.periodic) {
            if (j - nbas >= 0) put(j - nbas, v);
            if (j + nbas < nbas + bv.degree) put(j + nbas, v);
        }
    }
    __syncthreads();

    // ---------------- evaluation of every point of the LB lines ----------------
    if (!active) return;
    int64_t const pb = lay(pl, 0, lc);
    const double* tl = tile + ln;
    int const prow0 = seg; // point row of this thread within a pass
    // the point: read from coords, or the foot fpts[i] - fshift[line] of an
    // advection step (npts interpolation points)
    double const sh = fshift ? fshift[lc] : 0.0;
    auto point = [&](int64_t ii) {
        return fshift ? fpts[ii] - sh : __builtin_nontemporal_load(&coords[pb + ii * pl.rs]);
    };
    double xa[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        int64_t const ii = prow0 + int64_t(u) * ROWS;
        xa[u] = ii < npts ? point(ii) : 0.0;
    }
    for (int64_t i = prow0; i < npts; i += U * ROWS) {
        double xb[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int64_t const ii = i + int64_t(U + u) * ROWS;
            xb[u] = ii < npts ? point(ii) : 0.0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int64_t const ii = i + int64_t(u) * ROWS;
            if (ii < npts) {
                double x = xa[u];
                bool outside;
                double yv = 0.0;
                if (apply_bc(b, rules, x, outside)) {
                    double v[D + 1];
                    int const jmin = eval_basis<D, true>(b, b.knots, x, v);
#pragma unroll
                    for (int k = 0; k < D + 1; ++k) yv += tl[(jmin + k) * LB] * v[k];
                }
                __builtin_nontemporal_store(yv, &out[pb + ii * pl.rs]);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) xa[u] = xb[u];
    }
}

template <int K, int NT, bool MLDS, int KF, int KB, bool FDIV, bool BDIVF, int D>
void launch_one(BuilderPlan const& p, BSplinesView const& b, Rules1D rules, double* coef, Layout cl,
                const double* vals, Layout vl, const double* dl, const double* dr, Layout dlay, double* out,
                const double* coords, Layout pl, int64_t npts, int64_t nbatch, hipStream_t stream, size_t lds,
                const double* fpts, const double* fshift)
{
    if (p.tiled_f.rs != KF + KB + 1 + (FDIV ? 1 : 0))
        throw Error(DDCX_ERR_INVALID, "row table record length does not match the band shape");
    constexpr int LB = NT / K, L = 16;
    auto kern = fused_build_eval_kernel<LB, K, L, KF, KB, FDIV, BDIVF, D, MLDS>;
    hip_check(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  int(lds)),
              "hipFuncSetAttribute");
    hipLaunchKernelGGL(kern, dim3(tile_grid<LB>(nbatch)), dim3(NT), lds, stream, p.tview_f, p.view, b, rules, vals,
                       vl, dl, dr, dlay, coef, cl, out, coords, pl, npts, nbatch, fpts, fshift);
    hip_check(hipGetLastError(), "fused_build_eval_kernel launch");
}

template <int K, int NT, bool MLDS>
bool launch_K(BuilderPlan const& p, BSplinesView const& b, Rules1D rules, double* coef, Layout cl,
              const double* vals, Layout vl, const double* dl, const double* dr, Layout dlay, double* out,
              const double* coords, Layout pl, int64_t npts, int64_t nbatch, hipStream_t stream, size_t lds,
              const double* fpts, const double* fshift)
{
    TiledHost const& t = p.tiled_f;
    int const deg = b.degree;
    bool done = false;
    auto go = [&]<int KF, int KB, bool FD, bool BD, int D>() {
        if (!done && deg == D) {
            launch_one<K, NT, MLDS, KF, KB, FD, BD, D>(p, b, rules, coef, cl, vals, vl, dl, dr, dlay, out, coords, pl,
                                            npts, nbatch, stream, lds, fpts, fshift);
            done = true;
        }
    };
    if (t.bwd_divfirst) { // PDS tridiagonal: uniform periodic of degree 2, 3
        go.template operator()<1, 1, false, true, 2>();
        go.template operator()<1, 1, false, true, 3>();
    } else if (t.fwd_div) { // PDS band: uniform periodic of degree 4, 5
        if (t.kf == 2) {
            go.template operator()<2, 2, true, false, 4>();
            go.template operator()<2, 2, true, false, 5>();
        }
    } else if (t.kf == 1) { // band, kl = degree / 2 (uniform) or degree - 1 (non-uniform)
        go.template operator()<1, 1, false, false, 2>();
        go.template operator()<1, 1, false, false, 3>();
    } else if (t.kf == 2) {
        go.template operator()<2, 2, false, false, 3>();
        go.template operator()<2, 2, false, false, 4>();
        go.template operator()<2, 2, false, false, 5>();
    } else if (t.kf == 3) {
        go.template operator()<3, 3, false, false, 4>();
    } else if (t.kf == 4) {
        go.template operator()<4, 4, false, false, 5>();
    }
    return done;
}

} // namespace

bool launch_build_eval_fused(BuilderPlan const& p, BSplinesPlan const& bs, Rules1D rules, double* coef,
                             Layout cl, const double* vals, Layout vl, const double* dl, const double* dr,
                             Layout dlay, double* out, const double* coords, Layout pl, int64_t npts, int64_t nbatch,
                             hipStream_t stream, const double* feet_shift)
{
    TiledHost const& t = p.tiled_f;
    if (!t.ok || p.bs.get() != &bs) return false;
    if (feet_shift && npts != int64_t(p.points.size())) return false;
    const double* const fpts = feet_shift ? p.d_points : nullptr;
    if (vl.rs == 1 || pl.rs == 1 || (coef && cl.rs == 1)) return false; // batch-contiguous layouts only
    int const K = t.K, L = t.L;
    if (L != 16 || (K != 64 && K != 128)) return false;
    if (!offsets_fit(vl, int64_t(K) * L + p.tview_f.q0, nbatch)) return false;
    BSplinesView const b = bs.device_view();
    int const KE = std::max(t.kf, t.kb);
    // LDS of a workgroup of LB lines: the tables of the build, then the
    // coefficient tile; 0 when it does not fit
    auto lds_of = [&](int LB, bool transfer) {
        size_t const table = (size_t(K) * L * t.rs + gamma_lds_doubles(p.tview_f) +
                              (transfer ? transfer_doubles(p.tview_f) : 0)) *
                                 sizeof(double) +
                             sizeof(BorderLds);
        size_t const lds = std::max(table, size_t(bs.size()) * LB * sizeof(double));
        size_t const stat = size_t(KE * K * LB + kLamMax * LB + kNbMax * LB) * sizeof(double);
        return lds + stat > size_t(160 * 1024) ? size_t(0) : lds;
    };
    auto go = [&]<int KK, int NT, bool MLDS>() {
        size_t const lds = lds_of(NT / KK, MLDS);
        return lds > 0 && launch_K<KK, NT, MLDS>(p, b, rules, coef, cl, vals, vl, dl, dr, dlay, out, coords, pl, npts,
                                                 nbatch, stream, lds, fpts, feet_shift);
    };
    // Bases whose widest tile does not fit (non-uniform quintic from 944 cells)
    // take the two kernels where a build and an evaluation can follow each other:
    // few lines of many points are evaluated faster there (1000 cells, 3000 points x
    // 3 lines 30 us, 4-line tiles here 76).  Otherwise the narrower tiles do.
    bool const widest = lds_of(1024 / K, false) > 0;
    if (!widest && coef && !feet_shift) return false;
    // small batches (build_tiled_small.hip), 4 or 8 lines per workgroup: an
    // advection step of uniform cubic 512 cells x 1000 lines takes 15.5 us on 4
    // lines, 15.9 on 8 and 19.0 on 16; x 2000 lines 20.1, 16.3 and 18.9;
    // 1000 cells x 256 lines 18.2, 19.6 and 25.0
    if (K == 64) {
        bool const four = 2 * nbatch <= 8 * int64_t(cu_count()), eight = small_batch(nbatch, 1);
        return (four && go.template operator()<64, 256, true>()) ||
               ((eight || !widest) && go.template operator()<64, 512, true>()) ||
               go.template operator()<64, 1024, false>() || (!widest && go.template operator()<64, 256, true>());
    }
    // the transfer products in LDS where they fit; without them (non-uniform quartic
    // splines) the two kernels are faster for large batches of many points, where
    // they can follow each other: 2000 cells and points, us here / two kernels, x
    // 2048 lines 75 / 79, x 8000 271 / 225; 100 points x 2048 34 / 61
    if (go.template operator()<128, 1024, true>()) return true;
    if (coef && !feet_shift && nbatch > 8 * int64_t(cu_count()) && 2 * npts >= bs.size()) return false;
    return go.template operator()<128, 1024, false>();
}

} // namespace ddcx
