// LDS-staged batched evaluation (SplineEvaluator::operator() / deriv(),
// spline_evaluator.hpp:263-478).
//
// Random evaluation points gather the coefficients of their line at random,
// so a workgroup takes LB consecutive lines, stages their coefficient tile
// (size() x LB) and, for non-uniform bases, the knot vector and the cell-search
// brackets in LDS, and then evaluates all the points of those lines with
// coalesced coordinate loads and output stores.  HBM sees every coefficient,
// coordinate and output once.  Two thread mappings:
//  - batch-contiguous (line_major = 0): lanes take consecutive lines, so
//    tile rows and point rows are read as LB*8-byte runs;
//  - interpolation-contiguous (line_major = 1): the tile is read line by
//    line (size() contiguous doubles each) and the NT/LB threads of a line
//    take consecutive points of it.
// Values and first derivatives on plain batch-contiguous arrays take
// eval_stream_kernel, a persistent form that loads the next tile while the
// current one is evaluated; small batches, short lines and interpolation-
// contiguous arrays take narrower tiles (eval_narrow.hip).
#include "eval_tiled_kernel.hpp"

namespace ddcx {

namespace {

using tiled::basis_and_deriv;
using tiled::kMaxLds;
using tiled::lay;
using tiled::load_tile;
using tiled::point_values;

// Buffer resources (raw buffers, stride 0) for the streaming kernel: a load
// at a byte offset at or past num_records returns 0 and a store there is
// dropped, which is how the kernel handles the points past the end of a line.
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
constexpr int kBufferWord3 = 0x00020000; // 32-bit data format, gfx9 family

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const double* p, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(p), 0, int(bytes), kBufferWord3);
}

// Cache-policy bit NT (non-temporal) of the buffer instructions: every
// coordinate, coefficient and output of the streaming kernel is touched once,
// so its lines need not displace what the next kernel reads.
constexpr int kNonTemporal = 2;

template <int AUX = 0>
__device__ __forceinline__ double buffer_load(__amdgpu_buffer_rsrc_t r, uint32_t off)
{
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, int(off), 0, AUX));
}

template <int AUX = 0>
__device__ __forceinline__ void buffer_store(double v, __amdgpu_buffer_rsrc_t r, uint32_t off)
{
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, int(off), 0, AUX);
}

// Persistent form of eval_tiled_kernel for values and first derivatives with
// plain batch-contiguous arrays (element (row, line) at row * rs + line, 16-line
// tiles, NT threads: 512 for uniform bases, 768 for non-uniform ones).  Each
// workgroup walks the tiles blockIdx.x, blockIdx.x + gridDim.x, ...: while the
// points of one tile are evaluated, the coefficients
// of its next tile are loaded into registers (PR rows per thread, one slice per
// stage of U points), and they go to LDS once the current tile has been read.
// Coefficient loads, point loads and stores therefore overlap inside every CU
// instead of alternating in lockstep across the chip.  Every load and store of
// a tile is unconditional, so the compiler keeps each stage's loads in flight
// with exact vmcnt waits: points past the end of a line fall outside the
// buffers (loads give 0, stores are dropped), rows past the end of the tile
// repeat the last row, and lines past the batch repeat the last line.
// Addresses are 32-bit byte offsets into buffers of at most 4 GiB.
template <int D, int ORDER, int KIND, int NT, int U, int NST, int PR>
__global__ void __launch_bounds__(NT) eval_stream_kernel(BSplinesView b, Rules1D rules,
                                                           double* __restrict__ out,
                                                           const double* __restrict__ coords, uint32_t prs,
                                                           uint32_t pbytes, const double* __restrict__ coef,
                                                           uint32_t crs, uint32_t cbytes, int64_t nbatch, int ncoef,
                                                           int pitch, int nknots, int64_t ntiles, int npts)
{
    constexpr int LB = 16, ROWS = NT / LB;
    constexpr int PS = (PR + NST - 1) / NST; // prefetch rows per stage
    extern __shared__ double smem[];
    double* tile = smem;
    double* kn = smem + size_t(ncoef) * pitch;
    uint32_t* cells = reinterpret_cast<uint32_t*>(kn + nknots);
    int const tid = threadIdx.x;
    int const ln = tid % LB;
    int const prow = tid / LB;
    uint32_t const lastr = uint32_t(ncoef - 1);
    __amdgpu_buffer_rsrc_t const rc = buffer_of(coords, pbytes);
    __amdgpu_buffer_rsrc_t const ro = buffer_of(out, pbytes);
    __amdgpu_buffer_rsrc_t const rk = buffer_of(coef, cbytes);
    // byte offsets of point slot p and coefficient row j of line l.  Slot p
    // of tile t is point (p + rot(t)) mod npts, slots past npts stay outside
    // the buffer; the rotation of 64 points per tile spreads the rows that the
    // workgroups read at the same time over more DRAM banks.
    int rot = 0;
    auto pt = [&](int p, uint32_t l) {
        int q = p + rot;
        q = q >= npts ? q - npts : q;
        q = p < npts ? q : p;
        return (uint32_t(q) * prs + l) * 8u;
    };
    auto cr = [&](int j, uint32_t l) { return (min(uint32_t(prow + j * ROWS), lastr) * crs + l) * 8u; };
    auto line_of = [&](int64_t t) { return uint32_t(min(t * LB + ln, nbatch - 1)); };

    if (!is_uniform_kind(KIND, b.uniform)) {
        for (int k = tid; k < nknots; k += NT) kn[k] = b.knots[k];
        for (int k = tid; k < b.nbucket; k += NT) cells[k] = b.cells[k];
    }
    const double* knots = is_uniform_kind(KIND, b.uniform) ? nullptr : kn;
    BSplinesView bl = b;
    bl.cells = b.nbucket > 0 ? cells : nullptr;

    int64_t const G = gridDim.x;
    int64_t t = blockIdx.x;
    uint32_t lt = line_of(t);
    auto rot_of = [&](int64_t tt) { return int((tt * 64) % npts); };
    rot = rot_of(t);
    double xa[U];
#pragma unroll
    for (int u = 0; u < U; ++u) xa[u] = buffer_load<kNonTemporal>(rc, pt(prow + u * ROWS, lt));
    {
        double tv[PR];
#pragma unroll
        for (int j = 0; j < PR; ++j) tv[j] = buffer_load<kNonTemporal>(rk, cr(j, lt));
        int const col = int(int64_t(lt) - t * LB);
#pragma unroll
        for (int j = 0; j < PR; ++j) {
            int const r = prow + j * ROWS;
            if (r < ncoef) tile[r * pitch + col] = tv[j];
        }
    }
    while (true) {
        int64_t const tn = t + G;
        bool const more = tn < ntiles;
        uint32_t const ltn = line_of(more ? tn : t);
        // after the last tile the prefetch reads empty buffers: every access
        // is out of range, so it costs no memory traffic
        __amdgpu_buffer_rsrc_t const rcn = buffer_of(coords, more ? pbytes : 0u);
        __amdgpu_buffer_rsrc_t const rkn = buffer_of(coef, more ? cbytes : 0u);
        const double* tl = tile + (int64_t(lt) - t * LB);
        __syncthreads(); // tile t is in LDS
        double pf[PR];
#pragma unroll
        for (int s = 0; s < NST; ++s) {
            double xb[U];
            if (s + 1 < NST) {
#pragma unroll
                for (int u = 0; u < U; ++u) xb[u] = buffer_load<kNonTemporal>(rc, pt((s + 1) * U * ROWS + prow + u * ROWS, lt));
            } else {
                int const r0 = rot;
                rot = rot_of(more ? tn : t);
#pragma unroll
                for (int u = 0; u < U; ++u) xb[u] = buffer_load<kNonTemporal>(rcn, pt(prow + u * ROWS, ltn));
                rot = r0;
            }
#pragma unroll
            for (int j = s * PS; j < (s + 1) * PS && j < PR; ++j) pf[j] = buffer_load<kNonTemporal>(rkn, cr(j, ltn));
            double y[U] = {};
            // non-uniform bases: not for the slots past the end of the line (those of
            // the wave's first lane come first)
            if (KIND == kUniformBasis || s * U * ROWS + __builtin_amdgcn_readfirstlane(prow) < npts)
                point_values<D, ORDER, KIND, U>(bl, knots, rules, xa, tl, pitch, y);
#pragma unroll
            for (int u = 0; u < U; ++u) buffer_store<kNonTemporal>(y[u], ro, pt(s * U * ROWS + prow + u * ROWS, lt));
#pragma unroll
            for (int u = 0; u < U; ++u) xa[u] = xb[u];
        }
        __syncthreads(); // every read of tile t is done
        if (!more) break;
        int const col = int(int64_t(ltn) - tn * LB);
#pragma unroll
        for (int j = 0; j < PR; ++j) {
            int const r = prow + j * ROWS;
            if (r < ncoef) tile[r * pitch + col] = pf[j];
        }
        t = tn;
        lt = ltn;
        rot = rot_of(t);
    }
}

// Adjoint of the value form on 8-line tiles: gx = w * f'(x) where the spline
// itself is evaluated (0 where an extrapolation rule applies), and the
// coefficient gradient of the LB lines accumulated in an LDS tile with LDS
// atomics, then written once (every row, so no separate zeroing).
//
// Two tiles in LDS leave room for 8 lines, 64-byte runs in batch-contiguous
// arrays.  Neighbouring tiles on one XCD at the same time share their 128-byte
// lines in its L2 (so the loads and stores are not non-temporal: with them quartic
// 1024 x 20011 took 441 us instead of 309), one point per thread ahead keeps few
// rows in flight, and the basis of the kernel's kind alone needs 96 registers
// where the run-time choice spilled for quintic splines.  us, before -> after:
// uniform quintic 1024 x 65536 999 -> 842 (rows contiguous 777 -> 621), cubic 60000
// lines 676 -> 621 (623 -> 492), non-uniform cubic 1024 x 65536 1086 -> 877 (932 ->
// 697), quintic 1266 -> 1081 (1207 -> 884).
//
// Threads by the number of tiles that a CU's LDS holds, in batches of more than a
// tile per CU: 1024 where one fits, 512 for two and three, 256 for four and more
// in batches of four tiles per CU.  us on 256, 512 and 1024 threads, uniform cubic:
// 60 cells, 64 points x 65536 31, 43, 70; 150 cells, 384 x 20000 44, 48, 58; 300
// cells, 384 x 16384 44, 43, 51; 500 cells, 600 x 60000 398, 329, 357; 1024 cells,
// 100 x 65536 453, 370, 373 and 1024 x 65536 1101, 818, 814; one tile per CU, 300
// cells, 600 x 1000 16, 12, 11.
template <int D, int LB, int NT, int KIND>
__global__ void __launch_bounds__(NT) eval_vjp_tiled_kernel(BSplinesView b, Rules1D rules,
                                                            const double* __restrict__ coords,
                                                            const double* __restrict__ w, double* __restrict__ gx,
                                                            Layout pl, int64_t npts, const double* __restrict__ coef,
                                                            double* __restrict__ gcoef, Layout cl, int64_t nbatch,
                                                            int ncoef, int pitch, int nknots, int line_major)
{
    extern __shared__ double smem[];
    double* tile = smem;
    double* gt = smem + size_t(ncoef) * pitch;
    double* kn = gt + size_t(ncoef) * pitch;
    uint32_t* cells = reinterpret_cast<uint32_t*>(kn + nknots);
    constexpr int ROWS = NT / LB;
    constexpr int U = 1;
    constexpr int TC = 16;
    int const tid = threadIdx.x;
    int const ln = line_major ? tid / ROWS : tid % LB;
    int const prow = line_major ? tid % ROWS : tid / LB;
    // two tiles of 64-byte runs share their 128-byte lines: workgroups b and b +
    // 8, which run on one XCD, take neighbouring tiles
    static_assert(LB == 8);
    unsigned const bx = blockIdx.x;
    int64_t const line0 = int64_t(bx / 16 * 16 + bx % 8 * 2 + bx / 8 % 2) * LB;
    if (line0 >= nbatch) return; // whole workgroup
    int64_t const line = line0 + ln;
    bool const active = line < nbatch;
    int64_t const lc = active ? line : 0;
    int64_t const cb = lay(cl, 0, lc);
    int64_t const pb = lay(pl, 0, lc);
    // coefficient tile (as in eval_tiled_kernel) and a zeroed gradient tile
    load_tile<LB, NT, TC>(tile, pitch, coef + cb, cl.rs, ncoef, ln, prow);
    for (int k = tid; k < ncoef * pitch; k += NT) gt[k] = 0.0;
    if constexpr (KIND != kUniformBasis) {
        for (int k = tid; k < nknots; k += NT) kn[k] = b.knots[k];
        for (int k = tid; k < b.nbucket; k += NT) cells[k] = b.cells[k];
    }
    __syncthreads();
    const double* knots = KIND == kUniformBasis ? nullptr : kn;
    BSplinesView bl = b;
    bl.cells = b.nbucket > 0 ? cells : nullptr;
    if (active) {
        const double* tl = tile + ln;
        double* gl = gt + ln;
        // software pipeline: the next U points are read while the current ones
        // are worked through; indices past the end read the last point
        int const last = int(npts) - 1; // npts >= 64
        uint32_t const prs = uint32_t(pl.rs);
        const double* __restrict__ cp = coords + pb;
        const double* __restrict__ wp = w + pb;
        double* __restrict__ gp = gx + pb;
        auto at = [&](int ii) { return uint64_t(uint32_t(min(ii, last))) * prs; };
        double xn[U], wn[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            xn[u] = cp[at(prow + u * ROWS)];
            wn[u] = wp[at(prow + u * ROWS)];
        }
        for (int i = prow; i <= last; i += U * ROWS) {
            double xa[U], wa[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                xa[u] = xn[u];
                wa[u] = wn[u];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                xn[u] = cp[at(i + (U + u) * ROWS)];
                wn[u] = wp[at(i + (U + u) * ROWS)];
            }
            // bits: the spline is evaluated (not a Null rule's 0), a rule applies
            uint32_t in = 0, rule = 0;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                bool outside;
                if (apply_bc(bl, rules, xa[u], outside)) in |= 1u << u;
                if (outside) rule |= 1u << u;
            }
            int icell[U] = {};
            if constexpr (KIND == kNonUniformBasis) nonuniform_cells<U>(bl, knots, xa, icell);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                int const ii = i + u * ROWS;
                if (ii > last) continue;
                if (!((in >> u) & 1u)) {
                    gp[at(ii)] = 0.0;
                    continue;
                }
                double v[D + 1], dv[D + 1];
                int const jmin = basis_and_deriv<D, KIND>(bl, knots, xa[u], icell[u], v, dv);
                double dy = 0.0;
#pragma unroll
                for (int k = 0; k < D + 1; ++k) {
                    dy += tl[(jmin + k) * pitch] * dv[k];
                    atomicAdd(&gl[(jmin + k) * pitch], wa[u] * v[k]);
                }
                gp[at(ii)] = (rule >> u) & 1u ? 0.0 : wa[u] * dy;
            }
        }
    }
    __syncthreads();
    if (active) {
        for (int r = prow; r < ncoef; r += ROWS) gcoef[cb + int64_t(r) * cl.rs] = gt[r * pitch + ln];
    }
}

// The adjoint on 16-line tiles of batch-contiguous arrays, with one LDS tile used
// twice: first the coefficients, for gx = w f'(x) over all the tile's points; then
// the coefficient gradient, accumulated over the same points read again and
// written once.  Same arithmetic per point as eval_vjp_tiled_kernel.
//
// Against the 8-line tiles it halves the number of runs and works out the basis
// twice, so it pays for uniform bases up to degree 3 where a CU holds only one of
// those tiles and the coefficients outweigh the points, or the rows lie a large
// power of two apart, which makes the runs dearer.  us, 8-line tiles and here,
// cubic: 1024 cells x 65536, 100 points 373 and 294, 1024 points 814 and 791; 700
// cells x 16384, 384 points 109 and 95; x 60000 (no power of two), 200 points of
// 1024 cells 342 and 310, 1024 points 621 and 664.
template <int D, int LB, int NT>
__global__ void __launch_bounds__(NT) eval_vjp_2pass_kernel(BSplinesView b, Rules1D rules,
                                                            const double* __restrict__ coords,
                                                            const double* __restrict__ w, double* __restrict__ gx,
                                                            Layout pl, int64_t npts, const double* __restrict__ coef,
                                                            double* __restrict__ gcoef, Layout cl, int64_t nbatch,
                                                            int ncoef, int pitch)
{
    extern __shared__ double smem[];
    double* tile = smem;
    constexpr int ROWS = NT / LB;
    constexpr int U = 4;
    int const tid = threadIdx.x;
    int const ln = tid % LB;
    int const prow = tid / LB;
    int64_t const line0 = int64_t(blockIdx.x) * LB;
    int64_t const line = line0 + ln;
    bool const active = line < nbatch;
    int64_t const lc = active ? line : 0;
    int64_t const cb = lay(cl, 0, lc);
    int64_t const pb = lay(pl, 0, lc);
    load_tile<LB, NT, 16>(tile, pitch, coef + cb, cl.rs, ncoef, ln, prow);
    __syncthreads();
    double* tl = tile + ln;
    // every point of the line, U at a time: put(point, x, w, evaluated, rule applied)
    auto points = [&](auto put) {
        if (!active) return;
        for (int64_t i = prow; i < npts; i += U * ROWS) {
            double xa[U], wa[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                int64_t const ii = i + int64_t(u) * ROWS;
                xa[u] = ii < npts ? coords[pb + ii * pl.rs] : 0.0;
                wa[u] = ii < npts ? w[pb + ii * pl.rs] : 0.0;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                int64_t const ii = i + int64_t(u) * ROWS;
                if (ii >= npts) continue;
                double x = xa[u];
                bool outside;
                bool const in = apply_bc(b, rules, x, outside);
                put(ii, x, wa[u], in, outside);
            }
        }
    };
    points([&](int64_t ii, double x, double wv, bool in, bool outside) {
        if (!in) {
            gx[pb + ii * pl.rs] = 0.0;
            return;
        }
        double v[D + 1], dv[D + 1];
        int const jmin = basis_and_deriv<D, kUniformBasis>(b, nullptr, x, 0, v, dv);
        double dy = 0.0;
#pragma unroll
        for (int k = 0; k < D + 1; ++k) dy += tl[(jmin + k) * pitch] * dv[k];
        gx[pb + ii * pl.rs] = outside ? 0.0 : wv * dy;
    });
    __syncthreads();
    for (int k = tid; k < ncoef * pitch; k += NT) tile[k] = 0.0;
    __syncthreads();
    points([&](int64_t, double x, double wv, bool in, bool) {
        if (!in) return;
        double v[D + 1], dv[D + 1];
        int const jmin = basis_and_deriv<D, kUniformBasis>(b, nullptr, x, 0, v, dv);
#pragma unroll
        for (int k = 0; k < D + 1; ++k) atomicAdd(&tl[(jmin + k) * pitch], wv * v[k]);
    });
    __syncthreads();
    if (active)
        for (int r = prow; r < ncoef; r += ROWS) gcoef[cb + int64_t(r) * cl.rs] = tile[r * pitch + ln];
}

// eval_stream_kernel for the value form and the first derivative (up to degree
// 3) when its shape fits: plain batch-contiguous points and coefficients
// (element (row, line) at row * rs + line), npts <= NST * U * ROWS, size() <= PR *
// ROWS, buffers below 4 GiB including the offsets of the point slots past the end
// of a line.  Uniform bases: 512 threads, 33 prefetch rows; non-uniform bases
// (whose cell search wants more waves to hide its dependent LDS reads): 768
// threads, 22 prefetch rows, degrees up to 3.
//
// U = 2 points per thread and stage: 64 (or 96) rows of each array at a time.
// The workgroups walk the rows nearly together, and the fewer rows are in flight
// the fewer DRAM pages compete: a plain copy in 16-line tiles at this stride
// runs at 4.0 TB/s with 512 rows in flight per workgroup and at 4.7 with 128 to
// 256.  us at 1024 x 65536 for U = 8 / 4 / 2 / 1: cubic 369 / 356 / 351 / 376,
// quintic 400 / 382 / 378 / 387; 300 x 100000 284 / 243 / 232 / 247; first
// derivative of cubic 355 (U = 4) / 349 / 341; non-uniform cubic 457 (U = 4) /
// 439 / 434.
template <int D, int ORDER>
bool launch_stream(BSplinesPlan const& bs, Rules1D rules, double* out, const double* coords, Layout pl,
                   int64_t npts, const double* coef, Layout cl, int64_t nbatch, hipStream_t stream)
{
    int const ncoef = bs.size();
    int const nknots = bs.view.uniform ? 0 : int(bs.knots_host.size());
    BSplinesView const b = bs.device_view();
    constexpr int LB = 16, pitch = 17;
    auto plain = [&](Layout const& L) { return L.is == 1 && L.inner >= nbatch && L.rs >= nbatch; };
    if (!plain(pl) || !plain(cl)) return false;
    // batches of fewer than two tiles per CU keep eval_tiled_kernel: nothing
    // is left to prefetch
    int64_t const ntiles = (nbatch + LB - 1) / LB;
    if (ntiles < 2 * int64_t(cu_count())) return false;
    size_t const lds = size_t(ncoef) * pitch * sizeof(double) + nknots * sizeof(double) +
                       size_t(b.nbucket) * sizeof(uint32_t);
    if (lds > kMaxLds) return false;
    unsigned const grid = unsigned(std::min<int64_t>(ntiles, cu_count()));
    // the instantiations below hold their prefetch rows and point stages in
    // registers without spilling
    auto go = [&]<int KIND, int NT, int U, int NST, int PR>() {
        constexpr int ROWS = NT / LB;
        if (npts > int64_t(NST) * U * ROWS || ncoef > PR * ROWS) return false;
        uint64_t const lim = uint64_t(1) << 32;
        // byte offsets up to the last slot of the last stage must fit 32 bits
        if ((uint64_t(NST) * U * ROWS * uint64_t(pl.rs) + uint64_t(nbatch)) * 8 >= lim) return false;
        if ((uint64_t(ncoef) * uint64_t(cl.rs) + uint64_t(nbatch)) * 8 >= lim) return false;
        uint32_t const pbytes = uint32_t((uint64_t(npts - 1) * uint64_t(pl.rs) + uint64_t(nbatch)) * 8);
        uint32_t const cbytes = uint32_t((uint64_t(ncoef - 1) * uint64_t(cl.rs) + uint64_t(nbatch)) * 8);
        auto kern = eval_stream_kernel<D, ORDER, KIND, NT, U, NST, PR>;
        hip_check(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)),
                  "hipFuncSetAttribute");
        hipLaunchKernelGGL(kern, dim3(grid), dim3(NT), lds, stream, b, rules, out, coords, uint32_t(pl.rs),
                           pbytes, coef, uint32_t(cl.rs), cbytes, nbatch, ncoef, pitch, nknots, ntiles, int(npts));
        hip_check(hipGetLastError(), "eval_stream_kernel launch");
        return true;
    };
    // stages for at least npts points: 512, 768 or 1024 (uniform), 768 or 1152
    auto uniform = [&] {
        return npts <= 16 * 32   ? go.template operator()<kUniformBasis, 512, 2, 8, 33>()
               : npts <= 24 * 32 ? go.template operator()<kUniformBasis, 512, 2, 12, 33>()
                                 : go.template operator()<kUniformBasis, 512, 2, 16, 33>();
    };
    auto nonuniform = [&]<int KIND>() {
        return npts <= 16 * 48 ? go.template operator()<KIND, 768, 2, 8, 22>()
                               : go.template operator()<KIND, 768, 2, 12, 22>();
    };
    // higher degrees of the other forms spill and keep eval_tiled_kernel
    if constexpr (ORDER == 0 || D <= 3)
        if (b.uniform) return uniform();
    if constexpr (D <= 3) {
        if constexpr (ORDER == 1) return nonuniform.template operator()<kNonUniformBasis>();
        else if (bs.safe_products) return nonuniform.template operator()<kSafeNonUniform>();
        else return nonuniform.template operator()<kNonUniformBasis>();
    }
    return false;
}

template <int D, int ORDER>
bool launch_orders(BSplinesPlan const& bs, Rules1D rules, double* out, const double* coords, Layout xl, Layout pl,
                   int64_t npts, const double* coef, Layout cl, int64_t nbatch, hipStream_t stream)
{
    int const ncoef = bs.size();
    int const nknots = bs.view.uniform ? 0 : int(bs.knots_host.size());
    BSplinesView const b = bs.device_view();
    size_t const extra = nknots * sizeof(double) + size_t(b.nbucket) * sizeof(uint32_t);
    auto fits = [&](int lb, int pitch) { return size_t(ncoef) * pitch * sizeof(double) + extra <= kMaxLds; };
    auto go = [&]<int LB, int NT>(int pitch) {
        tiled::launch_eval_tile<D, ORDER, LB, NT>(bs, rules, out, coords, xl, pl, npts, coef, cl, nbatch, pitch, stream);
        return true;
    };
    if (ncoef > 2560) return false;
    auto same = [](Layout const& a, Layout const& c) {
        return a.rs == c.rs && a.inner == c.inner && a.is == c.is && a.os == c.os;
    };
    if constexpr (ORDER <= 1) {
        if (same(xl, pl) && launch_stream<D, ORDER>(bs, rules, out, coords, pl, npts, coef, cl, nbatch, stream))
            return true;
    }
    if (fits(16, 17)) return go.template operator()<16, 1024>(17);
    if (fits(16, 16)) return go.template operator()<16, 1024>(16);
    if (fits(8, 9)) return go.template operator()<8, 1024>(9);
    if (fits(8, 8)) return go.template operator()<8, 1024>(8);
    return false;
}

} // namespace

int cu_count()
{
    static int cached[64] = {};
    int dev = 0;
    hip_check(hipGetDevice(&dev), "hipGetDevice");
    if (dev < 0 || dev >= 64) dev = 0;
    if (cached[dev] == 0) {
        int n = 0;
        hip_check(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev), "hipDeviceGetAttribute");
        cached[dev] = n > 0 ? n : 1;
    }
    return cached[dev];
}

bool launch_eval_tiled(BSplinesPlan const& bs, Rules1D rules, int order, double* out, const double* coords,
                       Layout xl, Layout pl, int64_t npts, const double* coef, Layout cl, int64_t nbatch,
                       hipStream_t stream)
{
    // tiny batches, and mixed layouts (points and coefficients not both
    // batch-contiguous or both interpolation-contiguous), take the generic kernel
    if (npts < 64 || nbatch < 8) return false;
    if ((pl.rs == 1) != (cl.rs == 1)) return false;
    // 32-bit point indices and point strides in the kernel
    if (npts >= (int64_t(1) << 30) || pl.rs >= (int64_t(1) << 32) || xl.rs >= (int64_t(1) << 32)) return false;
    bool launched = launch_eval_narrow(bs, rules, order, out, coords, xl, pl, npts, coef, cl, nbatch, stream);
    if (launched) return true;
    dispatch_degree(bs.view.degree, [&]<int D>() {
        auto ord = [&]<int O>() {
            if constexpr (O <= D) {
                if (!launched && order == O)
                    launched = launch_orders<D, O>(bs, rules, out, coords, xl, pl, npts, coef, cl, nbatch, stream);
            }
        };
        ord.template operator()<0>();
        ord.template operator()<1>();
        ord.template operator()<2>();
        ord.template operator()<3>();
    });
    return launched;
}

bool launch_eval_vjp_tiled(BSplinesPlan const& bs, Rules1D rules, const double* coords, const double* w,
                           double* gx, Layout pl, int64_t npts, const double* coef, double* gcoef, Layout cl,
                           int64_t nbatch, hipStream_t stream)
{
    if (npts < 64 || nbatch < 8) return false;
    if ((pl.rs == 1) != (cl.rs == 1)) return false;
    // 32-bit point indices and point strides in the kernels
    if (npts >= (int64_t(1) << 30) || pl.rs >= (int64_t(1) << 32)) return false;
    int const ncoef = bs.size();
    if (ncoef > 2560) return false;
    int const nknots = bs.view.uniform ? 0 : int(bs.knots_host.size());
    BSplinesView const b = bs.device_view();
    size_t const extra = nknots * sizeof(double) + size_t(b.nbucket) * sizeof(uint32_t);
    auto lds_of = [&](int pitch) { return 2 * size_t(ncoef) * pitch * sizeof(double) + extra; };
    int pitch = 0;
    if (lds_of(9) <= kMaxLds) pitch = 9;
    else if (lds_of(8) <= kMaxLds) pitch = 8;
    else return false;
    bool const line_major = pl.rs == 1;
    bool launched = false;
    int64_t const cus = cu_count();
    int const resident = int(kMaxLds / lds_of(pitch)); // 8-line tiles that a CU's LDS holds
    // (the rules below: figures at the kernels)
    int const lds2 = ncoef * 17 * int(sizeof(double));
    if (!line_major && resident == 1 && nbatch >= 32 * cus && b.uniform && b.degree <= 3 && lds2 <= int(kMaxLds) &&
        (4 * npts <= ncoef || (pl.rs % 8192 == 0 && npts <= ncoef))) {
        dispatch_degree(b.degree, [&]<int D>() {
            if constexpr (D <= 3) {
                auto kern = eval_vjp_2pass_kernel<D, 16, 1024>;
                hip_check(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, lds2),
                          "hipFuncSetAttribute");
                hipLaunchKernelGGL(kern, dim3(unsigned((nbatch + 15) / 16)), dim3(1024), lds2, stream, b, rules,
                                   coords, w, gx, pl, npts, coef, gcoef, cl, nbatch, ncoef, 17);
                hip_check(hipGetLastError(), "eval_vjp_2pass_kernel launch");
                launched = true;
            }
        });
        if (launched) return true;
    }
    dispatch_degree(b.degree, [&]<int D>() {
        auto go = [&]<int NT>() {
            constexpr int LB = 8;
            auto kern = b.uniform ? eval_vjp_tiled_kernel<D, LB, NT, kUniformBasis>
                                  : eval_vjp_tiled_kernel<D, LB, NT, kNonUniformBasis>;
            size_t const lds = lds_of(pitch);
            hip_check(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)),
                      "hipFuncSetAttribute");
            int64_t const blocks = ((nbatch + LB - 1) / LB + 15) / 16 * 16;
            hipLaunchKernelGGL(kern, dim3(unsigned(blocks)), dim3(NT), lds, stream, b, rules, coords, w, gx, pl, npts,
                               coef, gcoef, cl, nbatch, ncoef, pitch, nknots, line_major ? 1 : 0);
            hip_check(hipGetLastError(), "eval_vjp_tiled_kernel launch");
            launched = true;
        };
        if (nbatch >= 32 * cus && resident >= 4) go.template operator()<256>();
        else if (nbatch > 8 * cus && resident >= 2) go.template operator()<512>();
        else go.template operator()<1024>();
    });
    return launched;
}

} // namespace ddcx
