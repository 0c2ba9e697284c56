// The LDS-staged batched evaluation kernel (described in eval_tiled.hip) and
// its launcher, shared by eval_tiled.hip and eval_narrow.hip.
#pragma once

#include "tiled_common.hpp"

namespace ddcx {
namespace tiled {

constexpr size_t kMaxLds = 160 * 1024;

// The value (ORDER 0) or derivative of a point; icell: its cell (non-uniform
// bases).
template <int D, int ORDER, int KIND>
__device__ __forceinline__ double tile_value(BSplinesView const& b, const double* kn, double x, int icell,
                                             const double* tile, int pitch)
{
    double v[D + 1];
    int jmin;
    if constexpr (ORDER == 0 && KIND != kUniformBasis) {
        nonuniform_basis<D, true, KIND == kSafeNonUniform>(kn, icell, x, v);
        jmin = icell - D;
    } else if constexpr (ORDER == 0) {
        jmin = eval_basis<D, true, KIND>(b, kn, x, v);
    } else if constexpr (ORDER == 1 && KIND != kUniformBasis) {
        double values[D + 1];
        nonuniform_basis_deriv<D>(kn, icell, x, values, v);
        jmin = icell - D;
    } else {
        double der[(D + 1) * (ORDER + 1)];
        jmin = eval_basis_and_n_derivs<D, ORDER, true, KIND, KIND != kUniformBasis>(b, kn, x, der, icell);
#pragma unroll
        for (int i = 0; i < D + 1; ++i) v[i] = der[i * (ORDER + 1) + ORDER];
    }
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < D + 1; ++i) s += tile[(jmin + i) * pitch] * v[i];
    return s;
}

// Values v and first derivatives dv of the splines on x's cell; returns the
// first spline.  icell: x's cell (non-uniform bases).
template <int D, int KIND>
__device__ __forceinline__ int basis_and_deriv(BSplinesView const& b, const double* kn, double x, int icell, double* v,
                                               double* dv)
{
    if constexpr (KIND != kUniformBasis) {
        nonuniform_basis_deriv<D>(kn, icell, x, v, dv);
        return icell - D;
    } else {
        double der[(D + 1) * 2];
        int const jmin = eval_basis_and_n_derivs<D, 1, true, KIND>(b, kn, x, der);
#pragma unroll
        for (int k = 0; k < D + 1; ++k) {
            v[k] = der[k * 2];
            dv[k] = der[k * 2 + 1];
        }
        return jmin;
    }
}

// The values (ORDER 0, with the extrapolation rules) or derivatives of U points
// of one line from its tile.
template <int D, int ORDER, int KIND, int U>
__device__ __forceinline__ void point_values(BSplinesView const& b, const double* kn, Rules1D rules, double* x,
                                             const double* tile, int pitch, double* y)
{
    if constexpr (KIND != kUniformBasis) {
        int icell[U];
        uint32_t zero = 0; // bit u: the Null rule gives 0
        if constexpr (ORDER == 0) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                bool outside;
                if (!apply_bc(b, rules, x[u], outside)) zero |= 1u << u;
            }
        }
        nonuniform_cells<U>(b, kn, x, icell);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // keeps the knots and divisors of one point at a time in registers (with a
            // branch in the basis the scheduling barrier alone does not)
            if constexpr (ORDER == 0 && KIND == kNonUniformBasis)
                if (u > 0) asm volatile("" : "+v"(x[u]), "+v"(y[u - 1]));
            double const s = tile_value<D, ORDER, KIND>(b, kn, x[u], icell[u], tile, pitch);
            y[u] = (zero >> u) & 1u ? 0.0 : s;
            if constexpr (ORDER == 0) __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_sched_barrier(0);
    } else {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            bool outside;
            if (ORDER == 0 && !apply_bc(b, rules, x[u], outside)) y[u] = 0.0;
            else y[u] = tile_value<D, ORDER, KIND>(b, kn, x[u], 0, tile, pitch);
        }
    }
}

// point_values in groups of G points, of which `live` (the same number in all
// lanes of a wave) are points of the line: groups past them are left out, and
// their y as it was.  Of a first derivative's last group, the points one by one.
template <int D, int ORDER, int KIND, int U, int G>
__device__ __forceinline__ void live_values(BSplinesView const& b, const double* kn, Rules1D rules, double (&x)[U],
                                            int live, const double* tile, int pitch, double (&y)[U])
{
    static_assert(U % G == 0);
#pragma unroll
    for (int u = 0; u < U; u += G) {
        if constexpr (ORDER == 1 && KIND != kUniformBasis && G > 1) {
            if (u + G > live) {
#pragma unroll
                for (int k = u; k < u + G; ++k)
                    if (k == 0 || k < live) point_values<D, ORDER, KIND, 1>(b, kn, rules, x + k, tile, pitch, y + k);
                continue;
            }
        }
        if (u == 0 || u < live) point_values<D, ORDER, KIND, G>(b, kn, rules, x + u, tile, pitch, y + u);
    }
}

// The coefficient tile of a workgroup's lines to LDS: thread (line ln, row
// prow) takes the rows prow, prow + NT / LB, ... of its line, in chunks of TC
// whose loads are all in flight before the first LDS write.  Batch-contiguous:
// the lanes of a row read LB consecutive lines; interpolation-contiguous: the
// threads of a line read consecutive rows of it.  Tiles of up to 4 rows per
// thread take chunks of 4: the 16 or 20 steps of a chunk are issued whether they
// have a row or not (16 cells x 120000 lines, rows contiguous, deriv(2): 191 us
// instead of 163).
template <int LB, int NT, int TC>
__device__ __forceinline__ void load_tile(double* tile, int pitch, const double* __restrict__ c, int64_t rs, int ncoef,
                                          int ln, int prow)
{
    constexpr int ROWS = NT / LB;
    if (TC > 4 && ncoef <= 4 * ROWS) return load_tile<LB, NT, TC < 4 ? TC : 4>(tile, pitch, c, rs, ncoef, ln, prow);
    for (int c0 = prow; c0 < ncoef; c0 += TC * ROWS) {
        double tv[TC];
#pragma unroll
        for (int k = 0; k < TC; ++k) {
            int const r = c0 + k * ROWS;
            tv[k] = r < ncoef ? c[int64_t(r) * rs] : 0.0;
        }
#pragma unroll
        for (int k = 0; k < TC; ++k) {
            int const r = c0 + k * ROWS;
            if (r < ncoef) tile[r * pitch + ln] = tv[k];
        }
    }
}

// UP: points per thread and stage (0: chosen here).
template <int D, int ORDER, int LB, int NT, int KIND, int UP = 0>
__global__ void __launch_bounds__(NT) eval_tiled_kernel(BSplinesView b, Rules1D rules, double* __restrict__ out,
                                                        const double* __restrict__ coords, Layout xl, Layout pl,
                                                        int64_t npts,
                                                        const double* __restrict__ coef, Layout cl, int64_t nbatch,
                                                        int ncoef, int pitch, int nknots, int line_major)
{
    extern __shared__ double smem[];
    double* tile = smem;
    double* kn = smem + size_t(ncoef) * pitch;
    uint32_t* cells = reinterpret_cast<uint32_t*>(kn + nknots);
    constexpr int ROWS = NT / LB;
    // points per pipeline stage per thread: as many as the registers hold
    // without spilling (derivative tables of non-uniform bases are the largest)
    constexpr int U = UP > 0 ? UP
                      : LB < 16 && NT < 1024 ? 4
                      : ORDER == 0 ? 8
                      : KIND == kUniformBasis ? (D <= 4 ? 8 : 4)
                                              : (D <= 1 ? 8 : (D <= 3 ? 4 : 2));
    // points worked through together
    constexpr int G = KIND == kUniformBasis ? U : ORDER == 0 && KIND == kSafeNonUniform ? 4 : ORDER == 1 ? U : 2;
    constexpr int TC = 20;         // tile rows per thread per load chunk (one chunk up to 20 * ROWS rows)
    int const tid = threadIdx.x;
    int const ln = line_major ? tid / ROWS : tid % LB;
    int const prow = line_major ? tid % ROWS : tid / LB;
    int64_t const line0 = tile_of<LB>(blockIdx.x, nbatch) * LB;
    if (LB < 16 && line0 >= nbatch) return; // whole workgroup
    int64_t const line = line0 + ln;
    bool const active = line < nbatch;
    int64_t const lc = active ? line : 0;
    int64_t const cb = lay(cl, 0, lc);
    int64_t const pb = lay(pl, 0, lc);
    // Point i of the line is at cp[i * prs].  Indices past the end are clamped
    // to the last point: such a slot loads the last coordinate and stores the
    // last point's own value again, so every load and store of the loop below
    // is unconditional and the loads of the next stage stay in flight while
    // the current stage is evaluated.
    int const last = int(npts) - 1;
    uint32_t const prs = uint32_t(pl.rs), xrs = uint32_t(xl.rs);
    const double* __restrict__ cp = coords + lay(xl, 0, lc);
    double* __restrict__ op = out + pb;
    auto at = [&](int ii) { return uint64_t(uint32_t(min(ii, last))) * prs; };
    auto atx = [&](int ii) { return uint64_t(uint32_t(min(ii, last))) * xrs; };
    // first batch of coordinates, then the whole coefficient tile: every load
    // of the tile is in flight before the first LDS write
    double xa[U];
#pragma unroll
    for (int u = 0; u < U; ++u) xa[u] = __builtin_nontemporal_load(&cp[atx(prow + u * ROWS)]);
    // the tile is loaded in chunks of TC elements per thread, every load of a
    // chunk in flight before its LDS writes
    load_tile<LB, NT, TC>(tile, pitch, coef + cb, cl.rs, ncoef, ln, prow);
    if (!is_uniform_kind(KIND, b.uniform)) {
        for (int k = tid; k < nknots; k += NT) kn[k] = b.knots[k];
        for (int k = tid; k < b.nbucket; k += NT) cells[k] = b.cells[k];
    }
    __syncthreads();
    if (!active) return;
    const double* knots = is_uniform_kind(KIND, b.uniform) ? nullptr : kn;
    BSplinesView bl = b;
    bl.cells = b.nbucket > 0 ? cells : nullptr;
    const double* tl = tile + ln;
    // software pipeline: the next batch of coordinates is in flight while the
    // current one is evaluated and stored
    for (int i = prow; i <= last; i += U * ROWS) {
        double xb[U];
#pragma unroll
        for (int u = 0; u < U; ++u) xb[u] = __builtin_nontemporal_load(&cp[atx(i + (U + u) * ROWS)]);
        double y[U];
        // The uniform basis is cheap, and its U points overlap; of the others only
        // the points of the line are worked through (64 points of 16 lines are one
        // of the U that a thread takes).  A wave's first lane holds its first point.
        int const live = (last - __builtin_amdgcn_readfirstlane(i)) / ROWS + 1;
        live_values<D, ORDER, KIND, U, G>(bl, knots, rules, xa, live, tl, pitch, y);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (KIND == kUniformBasis || (G == U && ORDER != 1) || (ORDER == 1 ? u == 0 || u < live : u / G * G < live)) __builtin_nontemporal_store(y[u], &op[at(i + u * ROWS)]);
#pragma unroll
        for (int u = 0; u < U; ++u) xa[u] = xb[u];
    }
}

// eval_tiled_kernel on tiles of LB lines with the given LDS pitch
template <int D, int ORDER, int LB, int NT>
void launch_eval_tile(BSplinesPlan const& bs, Rules1D rules, double* out, const double* coords, Layout xl, Layout pl,
                      int64_t npts, const double* coef, Layout cl, int64_t nbatch, int pitch, hipStream_t stream)
{
    int const ncoef = bs.size();
    int const nknots = bs.view.uniform ? 0 : int(bs.knots_host.size());
    BSplinesView const b = bs.device_view();
    size_t const lds = (size_t(ncoef) * pitch + nknots) * sizeof(double) + size_t(b.nbucket) * sizeof(uint32_t);
    // First derivatives of non-uniform bases: one point per thread and stage where
    // threads have only one or two points (64 points of 8192 quintic lines, us for 1
    // / 2 / 4 points: 12.5 / 17.4 / 23.4), and in batch-contiguous arrays whose rows
    // do not start at 128-byte lines: the fewer rows of points are in flight there,
    // the fewer DRAM pages compete (cubic 173 cells, 800 points x 65541: 431 / 574 /
    // 555), unless the lines are long, the workgroups on a CU few, and each waits
    // for its own chain (1024 to 1448 rows 1.24, 1.08 of the best).  Otherwise four
    // (rows contiguous 1024 x 65536 cubic 497 -> 419; 136 lines of 6144 points 54 ->
    // 38), or two with 1024 threads, four of which would spill.
    constexpr bool dnu = ORDER == 1;
    constexpr int many = NT < 1024 ? 4 : 2;
    bool const ahead = npts > 2 * (NT / LB) &&
                       (pl.rs % 16 == 0 || pl.rs == 1 || (many == 4 && (ncoef > 700 || nbatch <= 8 * int64_t(cu_count()))));
    auto kern = b.uniform ? eval_tiled_kernel<D, ORDER, LB, NT, kUniformBasis>
                : ORDER == 0 && bs.safe_products
                    ? eval_tiled_kernel<D, ORDER, LB, NT, ORDER == 0 ? kSafeNonUniform : kNonUniformBasis>
                : dnu && ahead ? eval_tiled_kernel<D, ORDER, LB, NT, kNonUniformBasis, dnu ? many : 0>
                               : eval_tiled_kernel<D, ORDER, LB, NT, kNonUniformBasis, dnu ? 1 : 0>;
    hip_check(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  int(lds)),
              "hipFuncSetAttribute");
    hipLaunchKernelGGL(kern, dim3(tile_grid<LB>(nbatch)), dim3(NT), lds, stream, b, rules, out, coords, xl, pl, npts,
                       coef, cl, nbatch, ncoef, pitch, nknots, pl.rs == 1 ? 1 : 0);
    hip_check(hipGetLastError(), "eval_tiled_kernel launch");
}

} // namespace tiled
} // namespace ddcx
