// Register-resident tiled adjoint of the batched build: the transposed solve
// of SplinesLinearProblem2x2Blocks::solve(b, true)
// (splines_linear_problem_2x2_blocks.cpp:275-298: the direct order reversed)
// after the fold of the periodic duplicate rows (the transpose of
// spline_builder.hpp:1074-1100), on the tiling of build_tiled_kernel.hpp:
//   1. y = folded gradient of the main-block rows (L per thread), b2 = the
//      folded gradient of the border rows;
//   2. b2 -= (Q^-1 gamma)^T y: partial sums of the segments that hold Q^-1
//      gamma blocks, combined in segment order by one thread per line;
//   3. x2 = S^-T b2 (the inverse of the Schur complement, transposed);
//   4. y -= lambda^T x2;
//   5. y = Q^-T y with the tiled sweeps (transposed tables);
//   6. the rows back to the value and Hermite-derivative gradients.
#include "tiled_common.hpp"

namespace ddcx {

namespace {

using namespace tiled;

// One segment's part of (Q^-1 gamma)^T y, a column of the block G per row of
// part (the loops as in apply_gamma).
template <int LB, int L>
__device__ __forceinline__ void gamma_trans(double const (&y)[L], const double* G, int nb, double (*part)[LB], int ln)
{
    for (int k = 0; k < nb; ++k) {
        const double* g = G + k * L;
        double acc = 0.0;
#pragma unroll
        for (int i = 0; i < L; ++i) acc = fma(g[i], y[i], acc);
        part[k][ln] = acc;
    }
}

template <int LB, int K, int L, int KF, int KB, bool FDIV, bool BDIVF, bool TLDS, bool IC>
__global__ void __launch_bounds__(LB* K, 4) build_vjp_tiled_kernel(TiledView tv, BuildView bv,
                                                               const double* __restrict__ gcoef, Layout cl,
                                                               double* __restrict__ gvals, Layout vl,
                                                               double* __restrict__ gdl, double* __restrict__ gdr,
                                                               Layout dlay, int64_t nbatch)
{
    constexpr int KE = KF > KB ? KF : KB;
    constexpr int NT = LB * K;
    constexpr int SR = stage_rows(K * L, LB), SP = stage_pitch(K * L, LB); // staging chunk rows, pitch (IC)
    __shared__ double ex[KE][K][LB];
    __shared__ double b2s[kNbMax][LB];
    __shared__ double x2s[kNbMax][LB];
    __shared__ BorderLds bl;
    alignas(16) extern __shared__ double rt_lds[];

    int const tid = threadIdx.x;
    int const ln = tid % LB;
    int const seg = tid / LB;
    int64_t const line0 = tile_of<LB>(blockIdx.x, nbatch) * LB;
    if (LB < 16 && line0 >= nbatch) return; // whole workgroup
    int64_t const line = line0 + ln;
    bool const active = line < nbatch;
    int64_t const lc = active ? line : line0;
    int64_t const cb = lay(cl, 0, lc);
    int64_t const vb = lay(vl, 0, lc);
    int const r0 = seg * L;
    int const nq = tv.nq, nb = tv.nb, top = tv.top;
    int const off = bv.offset, nbas = bv.nbasis, nsz = bv.size;
    constexpr int RS = KF + KB + 1 + (FDIV ? 1 : 0); // row record length, fixed by the band shape
    const double* __restrict__ cwg = gcoef + lay(cl, 0, line0);
    double* __restrict__ vwg = gvals + lay(vl, 0, line0);
    uint32_t const clo = uint32_t(cb - lay(cl, 0, line0));
    uint32_t const vlo = uint32_t(vb - lay(vl, 0, line0)) + uint32_t(tv.q0 + r0) * uint32_t(vl.rs);
    uint32_t const crs = uint32_t(cl.rs), vrs = uint32_t(vl.rs);

    // dynamic LDS: the row table (TLDS) in the space of the staging area (IC,
    // as in the build), the Q^-1 gamma blocks (TLDS), the segment transfer
    // products (MLDS), the partial sums of the border step (ngb * nb rows of LB)
    // and the per-line offsets of gcoef and gvals (IC)
    constexpr bool MLDS = TLDS && transfer_in_lds(LB);
    int const tab = TLDS ? K * L * RS : 0;
    double* stg = rt_lds;
    double* gpad = rt_lds + (IC ? max(tab, LB * SP) : tab);
    double* mtr = gpad + (TLDS ? tv.ngb * L * nb : 0);
    double* partp = mtr + (MLDS ? K * (tv.wf * KF * KF + tv.wb * KB * KB) : 0);
    double(*part)[LB] = reinterpret_cast<double(*)[LB]>(partp);
    uint32_t* loff = reinterpret_cast<uint32_t*>(partp + tv.ngb * nb * LB);
    int const nl = int(min<int64_t>(LB, nbatch - line0));
    if constexpr (IC) {
        if (tid < LB) {
            int64_t const l = line0 + min(tid, nl - 1);
            loff[tid] = uint32_t(lay(cl, 0, l) - lay(cl, 0, line0));
            loff[LB + tid] = uint32_t(lay(vl, 0, l) - lay(vl, 0, line0));
        }
        __syncthreads();
    }

    // 1. folded gradient: unknown i collects the coefficient rows j with
    //    (j - offset) mod nbasis == i (a single row except at the periodic ends)
    double y[L];
    {
        uint32_t const c0 = clo + uint32_t(top + r0 + off) * crs;
        if constexpr (IC) {
            // each line's main-block rows as contiguous runs through LDS
            constexpr int PER = LB * SR / NT;
            for (int rbase = 0; rbase < K * L; rbase += SR) {
                double tmp[PER];
#pragma unroll
                for (int k = 0; k < PER; ++k) {
                    int const e = tid + k * NT;
                    int const l = e / SR, u = rbase + e % SR;
                    tmp[k] = (l < nl && u < nq) ? __builtin_nontemporal_load(&cwg[loff[l] + uint32_t(top + u + off)])
                                                : 0.0;
                }
#pragma unroll
                for (int k = 0; k < PER; ++k) {
                    int const e = tid + k * NT;
                    stg[(e / SR) * SP + e % SR] = tmp[k];
                }
                __syncthreads();
                if (r0 >= rbase && r0 < rbase + SR) {
#pragma unroll
                    for (int i = 0; i < L; ++i) y[i] = stg[ln * SP + (r0 - rbase) + i];
                }
                __syncthreads();
            }
        } else if (r0 + L <= nq) {
#pragma unroll
            for (int i = 0; i < L; ++i) y[i] = __builtin_nontemporal_load(&cwg[c0 + uint32_t(i) * crs]);
        } else {
            uint32_t const cl0 = clo + uint32_t(top + off) * crs;
#pragma unroll
            for (int i = 0; i < L; ++i) {
                double const v = __builtin_nontemporal_load(&cwg[cl0 + uint32_t(min(r0 + i, nq - 1)) * crs]);
                y[i] = r0 + i < nq ? v : 0.0;
            }
        }
        if (bv.periodic && (r0 < bv.degree || r0 + L > nbas - off)) {
#pragma unroll
            for (int i = 0; i < L; ++i) {
                int const j1 = top + r0 + i + off;
                if (r0 + i < nq) {
                    if (j1 - nbas >= 0) y[i] += cwg[clo + uint32_t(j1 - nbas) * crs];
                    if (j1 + nbas < nsz) y[i] += cwg[clo + uint32_t(j1 + nbas) * crs];
                }
            }
        }
    }

    // the border rows' incoming gradient, folded like the main rows
    double b2 = 0.0;
    if (seg < nb && active) {
        int const j1 = (seg < top ? seg : nq + seg) + off;
        b2 = gcoef[cb + int64_t(j1) * cl.rs];
        if (bv.periodic) {
            if (j1 - nbas >= 0) b2 += gcoef[cb + int64_t(j1 - nbas) * cl.rs];
            if (j1 + nbas < nsz) b2 += gcoef[cb + int64_t(j1 + nbas) * cl.rs];
        }
    }
    SegBorder const sb = tv.seg[seg];

    // per-row table and border data in LDS when they fit
    const double* T;
    if constexpr (TLDS) {
        stage_table<NT, K * L, RS>(tv.rt, rt_lds, tid);
        if constexpr (MLDS) stage_transfer<NT>(tv, mtr, tid);
        stage_border<NT, true>(tv, bl, gpad, tid);
        __syncthreads();
        T = rt_lds + r0 * RS;
    } else {
        stage_border<NT, false>(tv, bl, gpad, tid); // without the Q^-1 gamma blocks
        T = tv.rt + size_t(r0) * RS;
    }

    // 2. partial sums of (Q^-1 gamma)^T y over this segment's rows
    if (sb.gblk >= 0) {
        if constexpr (TLDS) gamma_trans<LB>(y, gpad + sb.gblk * L * nb, nb, part + sb.gblk * nb, ln);
        else gamma_trans<LB>(y, tv.Gblk + size_t(sb.gblk) * L * nb, nb, part + sb.gblk * nb, ln);
    }
    if (seg < nb) b2s[seg][ln] = b2;
    __syncthreads();

    // 3. the border: b2 -= sum of the partials (segment order), x2 = S^-T b2;
    // every border row's thread sums the whole right-hand side for its own
    // row of the product
    if (seg < nb) {
        double x2 = 0.0;
        for (int j = 0; j < nb; ++j) {
            double v = b2s[j][ln];
            for (int g = 0; g < tv.ngb; ++g) v -= part[g * nb + j][ln];
            x2 = fma(bl.sinv[seg * nb + j], v, x2);
        }
        x2s[seg][ln] = x2;
        // 6 (border part). rows back to the gradients they came from
        if (active) {
            int64_t const db = lay(dlay, 0, lc);
            int const nv_end = nbas - bv.nbe_r;
            int const i = seg < top ? seg : nq + seg;
            if (bv.periodic) {
                gvals[vb + int64_t(i) * vl.rs] = x2;
            } else if (i < bv.nbe_l) {
                if (bv.bcl == DDCX_HERMITE) gdl[db + int64_t(i) * dlay.rs] = x2 * bv.dxpow[i + bv.odd];
            } else if (i < nv_end) {
                gvals[vb + int64_t(i - bv.nbe_l) * vl.rs] = x2;
            } else if (bv.bcu == DDCX_HERMITE) {
                gdr[db + int64_t(i - nv_end) * dlay.rs] = x2 * bv.dxpow[i - nv_end + bv.odd];
            }
        }
    }
    __syncthreads();

    // 4. y -= lambda^T x2, in the segments that hold coupled rows
    if (sb.mask != 0) {
#pragma unroll
        for (int i = 0; i < L; ++i)
            if ((sb.mask >> i) & 1u) {
                int const g = sb.slot0 + __popc(sb.mask & ((1u << i) - 1u));
                for (int j = 0; j < nb; ++j) y[i] = fma(-bl.m[g * nb + j], x2s[j][ln], y[i]);
            }
    }

    // 5. y = Q^-T y
    tiled_sweeps<LB, K, L, KF, KB, FDIV, BDIVF, KE>(y, T, RS, MLDS ? mtr : tv.Mf, tv.wf,
                                                    MLDS ? mtr + K * tv.wf * KF * KF : tv.Mb, tv.wb, ex, seg, ln);

    // 6. main-block rows to the value gradients
    if constexpr (IC) {
        __syncthreads(); // the staging area holds the row table until here
        constexpr int PER = LB * SR / NT;
        for (int rbase = 0; rbase < K * L; rbase += SR) {
            if (r0 >= rbase && r0 < rbase + SR) {
#pragma unroll
                for (int i = 0; i < L; ++i) stg[ln * SP + (r0 - rbase) + i] = y[i];
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < PER; ++k) {
                int const e = tid + k * NT;
                int const l = e / SR, u = rbase + e % SR;
                if (l < nl && u < nq)
                    __builtin_nontemporal_store(stg[l * SP + e % SR],
                                                &vwg[loff[LB + l] + uint32_t(tv.q0 + u)]);
            }
            __syncthreads();
        }
    } else if (active) {
        if (r0 + L <= nq) {
#pragma unroll
            for (int i = 0; i < L; ++i) __builtin_nontemporal_store(y[i], &vwg[vlo + uint32_t(i) * vrs]);
        } else {
#pragma unroll
            for (int i = 0; i < L; ++i)
                if (r0 + i < nq) __builtin_nontemporal_store(y[i], &vwg[vlo + uint32_t(i) * vrs]);
        }
    }
}

template <int K, int L, int KF, int KB, bool FDIV, bool BDIVF, int NT>
bool launch_cfg(BuilderPlan const& p, TiledView const& tv, const double* gcoef, Layout cl, double* gvals, Layout vl, double* gdl,
                double* gdr, Layout dlay, int64_t nbatch, hipStream_t stream)
{
    if (tv.rs != KF + KB + 1 + (FDIV ? 1 : 0))
        throw Error(DDCX_ERR_INVALID, "row table record length does not match the band shape");
    constexpr int LB = NT / K;
    constexpr int KE = KF > KB ? KF : KB;
    constexpr size_t static_lds =
        size_t(KE * K * LB + 2 * kNbMax * LB) * sizeof(double) + sizeof(BorderLds);
    bool const ic = vl.rs == 1 && cl.rs == 1;
    size_t const stage = ic ? size_t(LB) * stage_pitch(K * L, LB) * sizeof(double) : 0;
    size_t const rest = size_t(tv.ngb) * tv.nb * LB * sizeof(double) + (ic ? 2 * LB * sizeof(uint32_t) : 0);
    size_t const table = std::max(size_t(K) * L * tv.rs * sizeof(double), stage) + rest +
                         (gamma_lds_doubles(tv) + (transfer_in_lds(LB) ? transfer_doubles(tv) : 0)) * sizeof(double);
    bool const tlds = static_lds + table <= size_t(160 * 1024) && tv.rs <= 10;
    size_t const lds = tlds ? table : stage + rest;
    auto go = [&]<bool TL, bool I>() {
        auto kern = build_vjp_tiled_kernel<LB, K, L, KF, KB, FDIV, BDIVF, TL, I>;
        if (lds > 0)
            hip_check(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)),
                      "hipFuncSetAttribute");
        hipLaunchKernelGGL(kern, dim3(tile_grid<LB>(nbatch)), dim3(NT), lds, stream, tv, p.view, gcoef, cl, gvals,
                           vl, gdl, gdr, dlay, nbatch);
    };
    if constexpr (transfer_in_lds(LB)) {
        // the small-batch tiles exist with the table in LDS only
        if (!tlds) return false;
        if (ic) go.template operator()<true, true>();
        else go.template operator()<true, false>();
    } else if (ic) {
        if (tlds) go.template operator()<true, true>();
        else go.template operator()<false, true>();
    } else {
        if (tlds) go.template operator()<true, false>();
        else go.template operator()<false, false>();
    }
    hip_check(hipGetLastError(), "build_vjp_tiled_kernel launch");
    return true;
}

// NT threads per workgroup: NT / K lines of K segments of L rows
template <int K, int L, int NT = 1024>
bool launch_K(BuilderPlan const& p, TiledHost const& t, TiledView const& tv, const double* gcoef, Layout cl, double* gvals, Layout vl, double* gdl,
              double* gdr, Layout dlay, int64_t nbatch, hipStream_t stream)
{
    auto go = [&]<int KF, int KB, bool FD, bool BD>() {
        return launch_cfg<K, L, KF, KB, FD, BD, NT>(p, tv, gcoef, cl, gvals, vl, gdl, gdr, dlay, nbatch, stream);
    };
    if (t.bwd_divfirst) {
        if (t.kf == 1 && t.kb == 1 && !t.fwd_div) return go.template operator()<1, 1, false, true>();
        return false;
    }
    if (!t.fwd_div) return false;
    // PDS band, and the transposed unpivoted band
    if (t.kf == 1 && t.kb == 1) return go.template operator()<1, 1, true, false>();
    if (t.kf == 2 && t.kb == 2) return go.template operator()<2, 2, true, false>();
    if (t.kf == 3 && t.kb == 3) return go.template operator()<3, 3, true, false>();
    if (t.kf == 4 && t.kb == 4) return go.template operator()<4, 4, true, false>();
    return false;
}

} // namespace

bool launch_build_vjp_tiled(BuilderPlan const& p, const double* gcoef, Layout cl, double* gvals, Layout vl,
                            double* gdl, double* gdr, Layout dlay, int64_t nbatch, hipStream_t stream)
{
    if (!p.tiled_t.ok) return false;
    if (!offsets_fit(vl, p.tiled_t.K * p.tiled_t.L + p.tview_t.q0, nbatch) || !offsets_fit(cl, p.view.size, nbatch))
        return false;
    int const K = p.tiled_t.K, L = p.tiled_t.L;
    auto go = [&]<int KK, int LL, int NT>(TiledHost const& t, TiledView const& tv) {
        return launch_K<KK, LL, NT>(p, t, tv, gcoef, cl, gvals, vl, gdl, gdr, dlay, nbatch, stream);
    };
    auto one = [&]<int KK, int LL, int NT>() { return go.template operator()<KK, LL, NT>(p.tiled_t, p.tview_t); };
    // the small-batch tiles of the build (build_tiled_small.hip: 1000 cells x
    // 1000 lines 21.8 -> 12.8 us, rows contiguous 28.1 -> 13.8;
    // build_tiled_short.hip: 200 cells x 1000 lines 9.4 -> 7.9, 11.5 -> 8.8)
    if (small_batch(nbatch, 1) && p.tiled_ts.ok && go.template operator()<64, 16, 512>(p.tiled_ts, p.tview_ts))
        return true;
    if (L == 32) return K == 32 ? one.template operator()<32, 32, 1024>() : one.template operator()<64, 32, 1024>();
    if (K == 8) return L == 4 ? one.template operator()<8, 4, 256>() : one.template operator()<8, 8, 256>();
    if (K == 16) return L == 8 ? one.template operator()<16, 8, 512>() : one.template operator()<16, 9, 512>();
    if (small_batch(nbatch, 2) && one.template operator()<32, 8, 256>()) return true;
    return one.template operator()<32, 8, 1024>();
}

} // namespace ddcx
