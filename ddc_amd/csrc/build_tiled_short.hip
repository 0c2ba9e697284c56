// FP64 tiled build for short lines (main blocks of up to 255 rows, such as the
// passes of a 3D build on a 128^3 grid), 32 lines per workgroup as on the 32 x
// 32 tiling, so that the staging of interpolation-contiguous tiles fits in LDS
// as well:
//  - up to 64 rows on 8 segments of 4 or 8 rows (256 threads).  These lines ran
//    on the one-thread-per-line kernel, whose sweeps wait on a cache round trip
//    per row: 32 cells x 1000 lines 23 -> 6.2 us.  With 8 lines per workgroup
//    6.3 us, so there is no small-batch form;
//  - up to 144 rows on 16 segments of 8 or 9 rows (512 threads, so that every
//    thread holds rows of the line);
//  - longer lines on 32 segments of 8 rows: 1024 threads, or 8 lines per
//    workgroup of 256 threads for small batches (200 cells x 1000 lines 9.2 ->
//    7.3 us, rows contiguous 11.6 -> 9.1; x 4096 lines 9.5 -> 8.8, 12.1 -> 10.0;
//    x 8192 lines 10.3 -> 11.3).
#include "build_tiled_kernel.hpp"

namespace ddcx {

bool launch_build_tiled_short(BuilderPlan const& p, double* coef, Layout cl, const double* vals, Layout vl,
                              const double* dl, const double* dr, Layout dlay, int64_t nbatch, hipStream_t stream)
{
    int const K = p.tiled.K, L = p.tiled.L;
    auto go = [&]<int KK, int LL, int NT>() {
        return tiled_build::launch_K<KK, LL, NT>(p, p.tiled, p.tview, coef, cl, vals, vl, dl, dr, dlay, nbatch, stream);
    };
    if (K == 8) return L == 4 ? go.template operator()<8, 4, 256>() : go.template operator()<8, 8, 256>();
    if (K == 16) return L == 8 ? go.template operator()<16, 8, 512>() : go.template operator()<16, 9, 512>();
    if (tiled::small_batch(nbatch, 2) && go.template operator()<32, 8, 256>()) return true;
    return go.template operator()<32, 8, 1024>();
}

} // namespace ddcx
