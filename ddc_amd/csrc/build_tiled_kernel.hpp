// Register-resident tiled batched spline build (the hot path of
// SplineBuilder::operator(), spline_builder.hpp:896-1101).
//
// A workgroup of LB*K threads owns LB batch lines; thread (segment s, line l)
// holds rows [s*L, s*L + L) of line l's main-block right-hand side in
// registers.  Each line is therefore read from HBM once and written once:
//   1. load the L rows (lanes of a wave cover LB consecutive lines, so each
//      load instruction reads 64/LB contiguous runs of LB*8 bytes in the
//      batch-contiguous layout);
//   2. forward sweep, local pass with a zero incoming state -> outgoing
//      state, exchanged through LDS; the exact incoming state of every
//      segment is a short sum of precomputed transfer products, and the
//      segment's rows are corrected by the homogeneous recurrence of the
//      sweep started from that state;
//   3. the same for the backward sweep;
//   4. 2x2-block border (splines_linear_problem_2x2_blocks.cpp:275-298):
//      lambda couplings gathered through LDS, the small Schur system solved
//      by its inverse, one thread per border row and line, the Q^-1 gamma
//      correction applied in registers;
//   5. store, including the periodic duplicate rows (spline_builder.hpp:
//      1074-1100).
#pragma once

#include <algorithm>

#include "tiled_common.hpp"

namespace ddcx {
namespace tiled_build {

using namespace tiled;

// Long lines in batch-contiguous arrays (the whole table in LDS): one workgroup
// per resident place walks the tiles, so that the table and border data are
// staged once, and each row of the next tile is requested as the current one's
// row is stored.  us, a workgroup per tile -> this: cubic 300 x 100000 218 -> 207,
// non-uniform quintic 1024 x 65536 335 -> 329, 513 x 65536 275 -> 261, 1024 x 20000
// 135 -> 129, non-uniform cubic 1024 x 20000 86 -> 75.  With the table staged in
// halves (quintic Hermite 2048 x 32768) the staging waits behind the tile's loads:
// 383 -> 418, so those keep a workgroup per tile.
constexpr bool loops(int L, bool ic, int tmode) { return L == 32 && !ic && tmode == 1; }

// The exception, by grid size alone.  With rows a multiple of 8 KiB apart all
// rows of a tile share few memory channels, and workgroups that walk in step
// meet there; up to two multipliers that costs long lines more than the staging
// saves, until there are more than about nq / 128 tiles for each place.  us,
// walking -> a workgroup per tile: cubic 1024 x 16384 72 -> 61, x 65536 230 -> 220,
// 2048 x 8192 72 -> 59, non-uniform 1024 x 16384 80 -> 65, quintic 1024 x 16384
// 83 -> 70, cubic 512 x 16384 42 -> 37; but 1024 x 16400 56 -> 59, 300 x 16384
// 36 -> 38, 513 x 65536 158 -> 161.
inline bool walks(int kf, int nq, int64_t vrs, int64_t crs, int64_t tiles, int64_t places)
{
    return !(kf <= 2 && nq > 400 && vrs % 1024 == 0 && crs % 1024 == 0 && tiles * 128 <= places * nq);
}

// Wavefronts per SIMD to allocate registers for.  The batch-contiguous kernel
// of 129-256 rows in 1024 threads needs 64 to 66 registers up to three
// multipliers: held to 64 (the degree-6 forms move 4-9 of them around the
// border step), two workgroups share a CU.  At 66, one did: 224 x 28542 of
// degree 6 took 86 us against 67, 203 x 65536 quartic 151 against 115.  All
// others have 128 registers.
constexpr int waves_per_simd(int lb, int k, int l, int kf, bool ic)
{
    return lb == 32 && k == 32 && l == 8 && kf <= 3 && !ic ? 8 : 4;
}

// TMODE: 0 row table read from global memory (L2), 1 staged in LDS whole,
// 2 staged in LDS one sweep's fields at a time (tables too large for 1)
template <int LB, int K, int L, int KF, int KB, bool FDIV, bool BDIVF, int TMODE, bool IC>
__global__ void __launch_bounds__(LB* K, waves_per_simd(LB, K, L, KF, IC))
                build_tiled_kernel(TiledView tv, BuildView bv,
                                                           const double* __restrict__ vals, Layout vl,
                                                           const double* __restrict__ dl,
                                                           const double* __restrict__ dr, Layout dlay,
                                                           double* __restrict__ coef, Layout cl, int64_t nbatch)
{
    constexpr int KE = KF > KB ? KF : KB;
    constexpr int NT = LB * K;
    constexpr int SR = stage_rows(K * L, LB), SP = stage_pitch(K * L, LB); // staging chunk rows, pitch (IC)
    constexpr bool TLDS = TMODE != 0;
    constexpr bool MLDS = TMODE == 1 && transfer_in_lds(LB);
    constexpr int RSF = KF + (FDIV ? 1 : 0), RSB = KB + 1; // split records
    constexpr bool LOOP = loops(L, IC, TMODE);
    __shared__ double ex[KE][K][LB];
    __shared__ double lamx[kLamMax][LB];
    __shared__ double b2s[kNbMax][LB];
    // the border's solution, in the space of the sweeps' exchange (over when it is
    // written, and begun again behind a barrier); K >= kNbMax
    double(*const x2s)[LB] = ex[0];
    __shared__ BorderLds bl;
    alignas(16) extern __shared__ double rt_lds[];

    int const tid = threadIdx.x;
    int ln = tid % LB;
    int seg = tid / LB;
    int64_t line0 = tile_of<LB>(blockIdx.x, nbatch) * LB;
    if (LB < 16 && line0 >= nbatch) return; // whole workgroup
    int r0 = seg * L;
    int const nq = tv.nq;
    constexpr int RS = KF + KB + 1 + (FDIV ? 1 : 0); // row record length, fixed by the band shape
    // Workgroup-uniform bases plus 32-bit per-lane offsets (the host checks
    // that every offset of a tile fits), so that each load/store needs one
    // address register instead of two.
    const double* __restrict__ vwg;
    double* __restrict__ cwg;
    uint32_t vlo, clo; // of the line's first main-block row of this segment, and of its coefficient row 0
    bool active;
    // this thread's line of the tile that starts at l0 (lines past the batch: the first)
    auto line_of = [&](int64_t l0) { return l0 + ln < nbatch ? l0 + ln : l0; };
    auto at_vals = [&](int64_t l0) {
        vwg = vals + lay(vl, 0, l0);
        vlo = uint32_t(lay(vl, 0, line_of(l0)) - lay(vl, 0, l0)) + uint32_t(tv.q0 + r0) * uint32_t(vl.rs);
    };
    auto at_coef = [&](int64_t l0) {
        active = l0 + ln < nbatch;
        cwg = coef + lay(cl, 0, l0);
        clo = uint32_t(lay(cl, 0, line_of(l0)) - lay(cl, 0, l0));
    };
    at_vals(line0);
    at_coef(line0);

    // dynamic LDS: the row table (TLDS) in the space of the staging area (IC,
    // LB x stage_pitch doubles, in use before the table is loaded and after its
    // last read), the Q^-1 gamma blocks (TLDS), the segment transfer products
    // (MLDS) and the per-line offsets of vals and coef (IC)
    int const tab = TMODE == 2 ? K * L * (RSF > RSB ? RSF : RSB) : K * L * RS; // doubles of the table region
    int const area = IC ? max(TLDS ? tab : 0, LB * SP) : TLDS ? tab : 0;
    double* gpad = rt_lds + area;
    double* mtr = gpad + tv.ngb * L * tv.nb;
    double* stg = rt_lds;
    uint32_t* loff = reinterpret_cast<uint32_t*>(
        (TLDS ? mtr : gpad) + (MLDS ? K * (tv.wf * KF * KF + tv.wb * KB * KB) : 0));
    int const nl = int(min<int64_t>(LB, nbatch - line0));
    int off = bv.offset;
    int nbas = bv.nbasis;
    int const nb = tv.nb;

    double y[L];
    // Row i of the segment.  Past the main block (last segments): row nq - 1, in
    // bounds; the table's padding rows couple it to nothing and it is not
    // stored.  Values and coefficients are touched once: non-temporal loads and
    // stores keep them from displacing what the next kernel reads.
    int last = nq - 1 - r0;
    uint32_t vrs = uint32_t(vl.rs), crs = uint32_t(cl.rs);
    auto load_row = [&](int i) { return __builtin_nontemporal_load(&vwg[vlo + uint32_t(min(i, last)) * vrs]); };
    // the border rows' right-hand side and the segment's part of the border
    // step do not depend on the sweeps: read first, ahead of the tile
    auto load_border = [&](int64_t l0) {
        if (seg >= nb || l0 + ln >= nbatch) return 0.0;
        return rhs_src(bv, vals, vl, lay(vl, 0, l0 + ln), dl, dr, dlay, lay(dlay, 0, l0 + ln),
                       seg < tv.top ? seg : nq + seg);
    };
    double b2 = load_border(line0);
    SegBorder sb = tv.seg[seg];
    if constexpr (IC) {
        constexpr int PER = LB * SR / NT; // staged elements per thread and chunk
        if (tid < LB) {
            int64_t const l = line0 + min(tid, nl - 1);
            loff[tid] = uint32_t(lay(vl, 0, l) - lay(vl, 0, line0));
            loff[LB + tid] = uint32_t(lay(cl, 0, l) - lay(cl, 0, line0));
        }
        __syncthreads();
        for (int rbase = 0; rbase < K * L; rbase += SR) {
            double tmp[PER];
#pragma unroll
            for (int k = 0; k < PER; ++k) {
                int const e = tid + k * NT;
                int const l = e / SR, u = rbase + e % SR;
                tmp[k] = (l < nl && u < nq) ? __builtin_nontemporal_load(&vwg[loff[l] + uint32_t(tv.q0 + u)]) : 0.0;
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
    } else if (last >= L - 1) {
#pragma unroll
        for (int i = 0; i < L; ++i) y[i] = __builtin_nontemporal_load(&vwg[vlo + uint32_t(i) * vrs]);
    } else {
#pragma unroll
        for (int i = 0; i < L; ++i) y[i] = load_row(i);
    }

    if constexpr (TMODE == 1) {
        stage_table<NT, K * L, RS>(tv.rt, rt_lds, tid);
        if constexpr (MLDS) stage_transfer<NT>(tv, mtr, tid);
    }
    stage_border<NT, TLDS>(tv, bl, gpad, tid);

    // LOOP: the workgroup walks the tiles blockIdx.x, blockIdx.x + gridDim.x, ...
    for (;;) {
    // the compiler is not to keep every row's offsets in registers across the loop
    if constexpr (LOOP) {
        asm volatile("" : "+v"(last), "+s"(vrs), "+s"(crs), "+v"(r0), "+v"(seg), "+v"(ln));
        asm volatile("" : "+v"(sb.mask), "+v"(sb.slot0), "+v"(sb.gblk), "+s"(off), "+s"(nbas));
    }
    if (seg < nb) b2s[seg][ln] = b2;
    if constexpr (TMODE == 2) {
        // the forward sweep's fields, then (after its closing barrier) the
        // backward sweep's, in the same LDS region
        stage_half<NT, KF, KB, FDIV, true>(tv.rt, RS, K * L, rt_lds, tid);
        __syncthreads();
        tiled_forward<LB, K, L, KF, FDIV, 0, KF>(y, rt_lds + r0 * RSF, RSF, tv.Mf, tv.wf, ex, seg, ln);
        stage_half<NT, KF, KB, FDIV, false>(tv.rt, RS, K * L, rt_lds, tid);
        __syncthreads();
        tiled_backward<LB, K, L, KB, BDIVF, 0, KB>(y, rt_lds + r0 * RSB, RSB, tv.Mb, tv.wb, ex, seg, ln);
    } else {
        __syncthreads();
        const double* const T = TLDS ? rt_lds + r0 * RS : tv.rt + size_t(r0) * RS;
        const double* const Mf = MLDS ? mtr : tv.Mf;
        const double* const Mb = MLDS ? mtr + K * tv.wf * KF * KF : tv.Mb;
        tiled_sweeps<LB, K, L, KF, KB, FDIV, BDIVF, KE>(y, T, RS, Mf, tv.wf, Mb, tv.wb, ex, seg, ln);
    }

    // ---------------- border (2x2 blocks) ----------------
    if (nb > 0) {
        gather_coupled<LB, L>(y, sb, lamx, ln);
        __syncthreads();
        if (seg < nb) {
            double const x2 = border_row<LB>(tv, bl, b2s, lamx, seg, ln);
            x2s[seg][ln] = x2;
            if (active) {
                int const j = (seg < tv.top ? seg : nq + seg) + off;
                cwg[clo + uint32_t(j) * crs] = x2;
                if (bv.periodic) {
                    if (j - nbas >= 0) cwg[clo + uint32_t(j - nbas) * crs] = x2;
                    if (j + nbas < nbas + bv.degree) cwg[clo + uint32_t(j + nbas) * crs] = x2;
                }
            }
        }
        __syncthreads();
        // Q^-1 gamma is nonzero only in the segments near the block ends
        if (sb.gblk >= 0) {
            if constexpr (TLDS) apply_gamma<LB>(y, gpad + sb.gblk * L * nb, nb, x2s, ln);
            else apply_gamma<LB>(y, tv.Gblk + size_t(sb.gblk) * L * nb, nb, x2s, ln);
        }
    }

    // ---------------- store ----------------
    if constexpr (IC) {
        constexpr int PER = LB * SR / NT;
        __syncthreads(); // the staging area holds the row table until here
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
                                                &cwg[loff[LB + l] + uint32_t(tv.top + u + off)]);
            }
            __syncthreads();
        }
    }
    if (active && bv.periodic && (r0 < bv.degree || r0 + L > nbas - off)) {
#pragma unroll
        for (int i = 0; i < L; ++i) {
            int const prow = tv.top + r0 + i;
            if (prow < nq) {
                int const j0 = prow + off - nbas;
                if (j0 >= 0) cwg[clo + uint32_t(j0) * crs] = y[i];
                int const j2 = prow + off + nbas;
                if (j2 < nbas + bv.degree) cwg[clo + uint32_t(j2) * crs] = y[i];
            }
        }
    }
    if constexpr (IC) return; // rows stored above
    uint32_t const c0 = clo + uint32_t(tv.top + r0 + off) * crs;
    int64_t const next = line0 + int64_t(gridDim.x) * LB;
    if (!LOOP || next >= nbatch) {
        if (!active) return;
        if (last >= L - 1) {
#pragma unroll
            for (int i = 0; i < L; ++i) __builtin_nontemporal_store(y[i], &cwg[c0 + uint32_t(i) * crs]);
        } else {
#pragma unroll
            for (int i = 0; i < L; ++i)
                if (i <= last) __builtin_nontemporal_store(y[i], &cwg[c0 + uint32_t(i) * crs]);
        }
        return;
    }
    // a row leaves and the next tile's row takes its register (every line of
    // this tile is in the batch: a later tile exists)
    at_vals(next);
#pragma unroll
    for (int i = 0; i < L; ++i) {
        if (i <= last) __builtin_nontemporal_store(y[i], &cwg[c0 + uint32_t(i) * crs]);
        y[i] = load_row(i);
        chunk_fence(i);
    }
    b2 = load_border(next);
    at_coef(next);
    line0 = next;
    }
}

template <int K, int L, int KF, int KB, bool FDIV, bool BDIVF, int TMODE, bool IC, int NT>
void launch_one(BuilderPlan const& p, TiledView const& tv, size_t static_lds, size_t lds, double* coef, Layout cl, const double* vals, Layout vl,
                const double* dl, const double* dr, Layout dlay, int64_t nbatch, hipStream_t stream)
{
    constexpr int LB = NT / K;
    auto kern = build_tiled_kernel<LB, K, L, KF, KB, FDIV, BDIVF, TMODE, IC>;
    if (lds > 0)
        hip_check(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                      int(lds)),
                  "hipFuncSetAttribute");
    unsigned grid = tile_grid<LB>(nbatch);
    if (loops(L, IC, TMODE)) {
        // resident places: 128 registers allow 1024 threads per CU, and the LDS must hold them
        constexpr size_t cu_lds = 160 * 1024;
        unsigned const per_cu = std::max<size_t>(1, std::min<size_t>(1024 / NT, cu_lds / (static_lds + lds)));
        unsigned const places = unsigned(cu_count()) * per_cu;
        if (walks(KF, tv.nq, vl.rs, cl.rs, grid, places)) grid = std::min(grid, places);
    }
    hipLaunchKernelGGL(kern, dim3(grid), dim3(NT), lds, stream, tv, p.view, vals, vl, dl, dr, dlay,
                       coef, cl, nbatch);
    hip_check(hipGetLastError(), "build_tiled_kernel launch");
}

template <int K, int L, int KF, int KB, bool FDIV, bool BDIVF, int NT>
bool launch_cfg(BuilderPlan const& p, TiledView const& tv, double* coef, Layout cl, const double* vals, Layout vl, const double* dl,
                const double* dr, Layout dlay, int64_t nbatch, hipStream_t stream)
{
    if (tv.rs != KF + KB + 1 + (FDIV ? 1 : 0))
        throw Error(DDCX_ERR_INVALID, "row table record length does not match the band shape");
    constexpr int LB = NT / K;
    constexpr int KE = KF > KB ? KF : KB;
    constexpr size_t static_lds =
        size_t(KE * K * LB + kLamMax * LB + kNbMax * LB) * sizeof(double) + sizeof(BorderLds);
    bool const ic = vl.rs == 1 && cl.rs == 1;
    size_t const stage = ic ? size_t(LB) * stage_pitch(K * L, LB) * sizeof(double) : 0;
    size_t const off = ic ? 2 * LB * sizeof(uint32_t) : 0;
    constexpr int RSH = (KF + (FDIV ? 1 : 0)) > (KB + 1) ? (KF + (FDIV ? 1 : 0)) : (KB + 1);
    size_t const gam = gamma_lds_doubles(tv) * sizeof(double) +
                       (transfer_in_lds(LB) ? transfer_doubles(tv) * sizeof(double) : 0);
    size_t const table = std::max(size_t(K) * L * tv.rs * sizeof(double), stage) + gam + off;
    size_t const half = std::max(size_t(K) * L * RSH * sizeof(double), stage) + gam + off;
    size_t constexpr budget = 160 * 1024;
    int const mode = (static_lds + table <= budget && tv.rs <= 10) ? 1 : static_lds + half <= budget ? 2 : 0;
    size_t const lds = mode == 1 ? table : mode == 2 ? half : stage + off;
    auto go = [&]<int TM, bool I>() {
        launch_one<K, L, KF, KB, FDIV, BDIVF, TM, I, NT>(p, tv, static_lds, lds, coef, cl, vals, vl, dl, dr, dlay, nbatch, stream);
    };
    // the small-batch tiles exist with the whole table in LDS only
    if constexpr (transfer_in_lds(LB)) {
        if (mode != 1) return false;
        if (ic) go.template operator()<1, true>();
        else go.template operator()<1, false>();
        return true;
    }
    auto pick = [&]<bool I>() {
        if (mode == 1) go.template operator()<1, I>();
        else if (mode == 2) go.template operator()<2, I>();
        else go.template operator()<0, I>();
    };
    if (ic) pick.template operator()<true>();
    else pick.template operator()<false>();
    return true;
}

// NT threads per workgroup: NT / K lines of K segments of L rows, the tables
// t and their device view tv on that tiling
template <int K, int L, int NT = 1024>
bool launch_K(BuilderPlan const& p, TiledHost const& t, TiledView const& tv, double* coef, Layout cl, const double* vals, Layout vl, const double* dl,
              const double* dr, Layout dlay, int64_t nbatch, hipStream_t stream)
{
    auto go = [&]<int KF, int KB, bool FD, bool BD>() {
        return launch_cfg<K, L, KF, KB, FD, BD, NT>(p, tv, coef, cl, vals, vl, dl, dr, dlay, nbatch, stream);
    };
    if (t.bwd_divfirst) {
        if (t.kf == 1 && t.kb == 1 && !t.fwd_div) return go.template operator()<1, 1, false, true>();
        return false;
    }
    if (t.fwd_div) { // PDSBand
        if (t.kf == 2 && t.kb == 2) return go.template operator()<2, 2, true, false>();
        if (t.kf == 3 && t.kb == 3) return go.template operator()<3, 3, true, false>();
        return false;
    }
    // unpivoted band
    if (t.kf == 1 && t.kb == 1) return go.template operator()<1, 1, false, false>();
    if (t.kf == 2 && t.kb == 2) return go.template operator()<2, 2, false, false>();
    if (t.kf == 3 && t.kb == 3) return go.template operator()<3, 3, false, false>();
    if (t.kf == 4 && t.kb == 4) return go.template operator()<4, 4, false, false>();
    return false;
}

} // namespace tiled_build
} // namespace ddcx
