// eval_tiled_kernel on tiles of 4 or 8 lines, 512 threads, for values and first
// derivatives of degrees 2 to 5.
//
// The 16-line tile fills most of a CU's LDS and has 1024 threads: small batches
// leave CUs idle, short lines leave threads idle (16 lines of 100 points are 1.6
// points per thread), and one resident workgroup alternates between loading its
// tile and its points.  Narrow tiles put two or more workgroups on a CU.  Their
// runs in batch-contiguous arrays are 32 or 64 bytes, which costs bandwidth where
// the arrays come from HBM and the lines are long; neighbouring tiles run on one
// XCD, whose L2 then holds the shared lines.  Times in us, the 16-line kernels ->
// here (value form; batch-contiguous, then rows contiguous):
//  - small batches, latency-bound: uniform cubic 512 points x 1000 lines 11.6 ->
//    7.2, 10.8 -> 5.9; 1000 x 1000 17.2 -> 9.6, 16.1 -> 7.5; non-uniform 32.3 ->
//    15.7, 31.0 -> 14.0; 2000 lines of 1000 points 16.8 -> 12.6 on 8 lines, 19.6
//    on 4;
//  - rows contiguous, any batch: uniform cubic 64 x 90001 184 -> 110, 300 x 90001
//    198 -> 167, 600 x 60000 241 -> 166, 1024 x 65536 322 -> 290; non-uniform 700
//    x 60001 369 -> 248; where two 8-line tiles do not fit a CU 4 lines: non-
//    uniform 1024 x 65536 443 -> 421 (517 on 8 lines), 2000 x 20000 200 -> 168;
//    where one 4-line tile fills a CU and there are a few points, 8 lines (uniform,
//    2125 rows, 100 points x 16384 94 -> 68);
//  - batch-contiguous, uniform, rows too long for two 8-line tiles: the wide kernel
//    has 8 or 16 lines on the whole CU there (1757 rows, 200 points x 16384 116 ->
//    68; 1579 rows, 100 points x 4010 25 -> 18);
//  - batch-contiguous, uniform, up to 512 points: 64 x 65536 122 -> 82, 256 x 65536
//    140 -> 105, 512 x 65536 200 -> 191.  Above, the streaming kernel is faster (1024
//    x 65536 357, here 500), and with more cells than points already there (1000
//    cells, 300 points x 65536 201, here 236; but 557 cells, 100 points x 32768 75 ->
//    50).  Up to 1024 where the batch has too few tiles to stream (33 -> 31 for 300
//    cells, 1000 points x 5008, but x 8000 37, here 47), 256 where it is one 16-line
//    tile per CU (500 x 4000 11.8, here 14.4);
//  - batch-contiguous, non-uniform: always above degree 3, which does not stream
//    (5 to 18% at 512 points and more); up to 256 points below (200 points of as
//    many cells 1.2 to 1.4 times; 300 points x 65536 160, here 191), and where the
//    batch is too small to stream (300 cells, 1000 points x 5008 50 -> 39);
//  - rows that do not start at 128-byte lines, where 16-line runs straddle two:
//    up to 1024 points (600 x 60001 451 -> 374, 1000 x 60001 736 -> 699, non-uniform
//    751 -> 657; 3000 points of 1000 cells x 32769 1030, here 1123) or 1.5 a row
//    (1026 x 16389 207 -> 141), above that non-uniform where the wide kernel does not
//    stream; not for a few points of long non-uniform lines in a large batch.
#include "eval_tiled_kernel.hpp"

namespace ddcx {

bool launch_eval_narrow(BSplinesPlan const& bs, Rules1D rules, int order, double* out, const double* coords, Layout xl,
                        Layout pl, int64_t npts, const double* coef, Layout cl, int64_t nbatch, hipStream_t stream)
{
    int const degree = bs.view.degree;
    if (order > 1 || degree < 2 || degree > 5) return false;
    size_t const extra = (bs.view.uniform ? 0 : bs.knots_host.size()) * sizeof(double) +
                         bs.cells_host.size() * sizeof(uint32_t);
    // LDS of a tile with the given (odd) pitch
    auto lds = [&](int pitch) { return size_t(bs.size()) * pitch * sizeof(double) + extra; };
    int64_t const cus = cu_count();
    bool const uniform = bs.view.uniform, rows = pl.rs == 1, aligned = pl.rs % 16 == 0;
    bool const two = lds(9) <= tiled::kMaxLds / 2;     // 8-line tiles, two per CU
    bool const one4 = lds(5) > tiled::kMaxLds / 2;     // 4-line tiles, one per CU
    bool const few = 4 * npts < bs.size();
    // where not even an 8-line tile holds the line and its knots, the per-point
    // kernel spreads a few lines over all CUs, and reads only what a few points need
    if (!uniform && lds(8) > tiled::kMaxLds && (nbatch < 2 * cus || 16 * npts < bs.size())) return false;
    auto narrow = [&] { // 8 lines, against the wider kernels
        if (uniform) {
            if (!two && lds(17) > tiled::kMaxLds) return true; // the wide kernel has no 16-line tile
            if (aligned && nbatch <= 16 * cus) return npts <= 256;
            if (!aligned) return npts <= 1024 || (2 * npts <= 3 * bs.size() && nbatch < 128 * cus);
            if (nbatch < 32 * cus) return npts <= 512 || (npts <= 1024 && nbatch < 24 * cus);
            return npts <= 512 && (bs.size() <= (few ? 800 : 520) || nbatch <= 128 * cus);
        }
        // the streaming kernel takes non-uniform bases up to degree 3
        if (lds(16) > tiled::kMaxLds) return few || !aligned;
        if (!aligned) return (npts <= 1024 || (degree > 3) == two) && (two || !few || nbatch < 128 * cus);
        return two && (nbatch < 32 * cus || degree > 3 || npts <= 256);
    };
    int lines = 0;
    if (nbatch <= 4 * cus) lines = 4;
    else if (rows || nbatch <= 8 * cus) lines = two || (nbatch <= 8 * cus && !rows) || (few && one4) ? 8 : 4;
    else if (narrow()) lines = 8;
    if (lines == 0 || lds(lines + 1) > tiled::kMaxLds) return false;
    auto go = [&]<int D, int ORDER>() {
        if (lines == 4)
            tiled::launch_eval_tile<D, ORDER, 4, 512>(bs, rules, out, coords, xl, pl, npts, coef, cl, nbatch, 5, stream);
        else
            tiled::launch_eval_tile<D, ORDER, 8, 512>(bs, rules, out, coords, xl, pl, npts, coef, cl, nbatch, 9, stream);
    };
    auto pick = [&]<int D>() { order == 0 ? go.template operator()<D, 0>() : go.template operator()<D, 1>(); };
    switch (degree) {
    case 2: pick.template operator()<2>(); break;
    case 3: pick.template operator()<3>(); break;
    case 4: pick.template operator()<4>(); break;
    default: pick.template operator()<5>(); break;
    }
    return true;
}

} // namespace ddcx
