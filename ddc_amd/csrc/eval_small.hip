// eval_tiled_kernel for small batches (at most one 8-line tile per CU): values
// and first derivatives of degrees 2 to 5.
//
// Bound by latency: the arrays sit in cache, and 1000 lines are 63 tiles of 16
// lines, a quarter of the chip's CUs, each loading its tile and then working
// through 16 points per thread.  Four lines per workgroup of 512 threads, or
// eight when there are more than four lines per CU, neighbouring tiles on one
// XCD.  Kernel to kernel in a graph, 1024-thread 16-line tile -> here:
//   uniform cubic, 512 points x 1000 lines 11.6 -> 7.2 us (rows contiguous 10.8
//   -> 5.9), 1000 x 1000 17.2 -> 9.6 (16.1 -> 7.5), 100 x 1000 10.0 -> 5.7;
//   non-uniform cubic 1000 x 1000 32.3 -> 15.7 (31.0 -> 14.0);
//   2000 lines, 1000 points: 16.8 -> 12.6 on 8 lines, 19.6 on 4;
//   3000 lines: 24.0 on 16 lines, 22.9 on 8; 4096 lines: 22.9 and 30.4.
// 256 threads for four lines: 7.3 us at 512 points, 11.0 at 1000, 23.1 on the
// non-uniform basis.
#include "eval_tiled_kernel.hpp"

namespace ddcx {

bool launch_eval_small(BSplinesPlan const& bs, Rules1D rules, int order, double* out, const double* coords, Layout xl,
                       Layout pl, int64_t npts, const double* coef, Layout cl, int64_t nbatch, hipStream_t stream)
{
    int const degree = bs.view.degree;
    if (order > 1 || degree < 2 || degree > 5 || !tiled::small_batch(nbatch, 1)) return false;
    int const nknots = bs.view.uniform ? 0 : int(bs.knots_host.size());
    // an odd LDS pitch of at least LB doubles per row
    auto fits = [&](int pitch) {
        return (size_t(bs.size()) * pitch + nknots) * sizeof(double) + bs.cells_host.size() * sizeof(uint32_t) <=
               tiled::kMaxLds;
    };
    bool const four = nbatch <= 4 * int64_t(cu_count());
    auto go = [&]<int D, int ORDER>() {
        if (four && fits(5))
            tiled::launch_eval_tile<D, ORDER, 4, 512>(bs, rules, out, coords, xl, pl, npts, coef, cl, nbatch, 5, stream);
        else if (fits(9))
            tiled::launch_eval_tile<D, ORDER, 8, 512>(bs, rules, out, coords, xl, pl, npts, coef, cl, nbatch, 9, stream);
        else return false;
        return true;
    };
    auto pick = [&]<int D>() { return order == 0 ? go.template operator()<D, 0>() : go.template operator()<D, 1>(); };
    switch (degree) {
    case 2: return pick.template operator()<2>();
    case 3: return pick.template operator()<3>();
    case 4: return pick.template operator()<4>();
    default: return pick.template operator()<5>();
    }
}

} // namespace ddcx
