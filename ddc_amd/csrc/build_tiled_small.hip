// FP64 tiled build for small batches (at most one 8-line tile per CU) of lines
// of 256 to 1024 rows: 64 segments of 16 rows (the tables of the fused kernel's
// tiling), 8 lines per workgroup of 512 threads.
//
// Bound by latency: the arrays sit in cache, and 1000 lines are 63 workgroups
// of the 16-line tile, each one chain of loads, sweeps over 32 rows, carries,
// border and stores.  Here the segments are half as long, the transfer products
// wait in LDS, an interpolation-contiguous tile is staged in one chunk, and
// there are twice as many workgroups, neighbours on one XCD.  1000 lines,
// kernel to kernel in a graph, the 16-line tile -> this one: uniform cubic 512
// cells 14.8 -> 11.2 us (rows contiguous 17.6 -> 12.6), 1000 cells 16.3 -> 12.3
// (20.0 -> 13.5), non-uniform cubic 1000 cells 17.8 -> 14.8 (21.5 -> 16.1).
// 2000 lines: 15.0 -> 14.1 (20.9 -> 14.5); 3000 lines, two tiles on some CUs:
// 18.0 -> 17.9 (21.6 -> 17.8), quintic 19.6 -> 30.3, so they keep the 16-line
// tile.  Four lines per workgroup: 11.1 us at 512 cells x 1000 lines, 14.4 at
// 1000 cells and 25.9 at 2000 lines (32-byte runs).
#include "build_tiled_kernel.hpp"

namespace ddcx {

bool launch_build_tiled_small(BuilderPlan const& p, double* coef, Layout cl, const double* vals, Layout vl,
                              const double* dl, const double* dr, Layout dlay, int64_t nbatch, hipStream_t stream)
{
    if (!p.tiled_f.ok || p.tiled_f.K != 64) return false;
    return tiled_build::launch_K<64, 16, 512>(p, p.tiled_f, p.tview_f, coef, cl, vals, vl, dl, dr, dlay, nbatch,
                                              stream);
}

} // namespace ddcx
