// Binning of scattered evaluation points by cell tile, shared by the binned
// 2D adjoint (eval2d_binned.hip) and the binned 3D evaluation
// (eval_nd.hip).  A caller's count pass gives each point a tile (16
// bits, kNoBin for a point an extrapolation rule settles by itself) and per
// batch entry and tile a count; then
//   bin_scan_kernel    turns the counts into tile offsets (starts) and the
//                      offsets of each tile's groups (cursor) for the scatter;
//   bin_scatter_kernel writes each point's record (its NX coordinates, then
//                      its weight when W) and index in tile order: a
//                      workgroup takes kScatT * PTS points, reads each once,
//                      orders the records by tile in LDS and writes the
//                      records of one tile as one run of consecutive lanes
//                      and addresses;
// after which one workgroup per (batch entry, tile) reads its points in order.
//
// The scatter is bound by memory, and by the lines its runs share more than by
// their bytes: 4096 points over 256 tiles are runs of 16 records (384 B), so
// most lines at the ends of a run are completed by the next workgroup that
// reserves a run of the tile.  On another XCD that is a second partial write
// of the line.  So a tile's range is divided into kGroups parts by the points'
// workgroup modulo the XCD count, and each part is filled from one XCD's L2:
// 930 -> 680 us for 16 x 4M points on 1024 x 1024 cells (runs half as long,
// 2048 points per workgroup and two workgroups per CU: 1080 us), 250 -> 184 us
// for 4 x 4M points on 128^3 (two XCDs per tile: 210 us).  The kernels
// that read a tile's points take as long as before at 4M points per batch
// entry; at 16M the 2D adjoint's takes 8% longer, against 27% less here.
#pragma once

#include "internal.hpp"

namespace ddcx {
namespace binning {
namespace {

constexpr int kMaxBins = 4096;          // tiles per batch entry
constexpr int kNoBin = 0xffff;          // stored tile of a point that no tile takes
constexpr int kScatT = 1024;            // threads of the scatter workgroups
constexpr int kScatPts = 4;             // points per thread there
constexpr int kChunk = kScatT * kScatPts; // points per workgroup, in the count and the scatter
constexpr int kGroups = 8;              // parts of a tile's range: one per XCD
constexpr size_t kLdsBytes = 160 * 1024;

// j / T for cells 0 <= j < 2^26 and tile sides 1 < T <= 64, as the high half of
// one product: inverse(T) exceeds 2^32 / T by less than 1, which moves the
// quotient by less than j / 2^32, below the 1 / T it may.
constexpr unsigned inverse(int T) { return unsigned(((uint64_t(1) << 32) + unsigned(T) - 1) / unsigned(T)); }
__device__ __forceinline__ int tile_index(int j, unsigned inv_T) { return int(__umulhi(unsigned(j), inv_T)); }

__global__ void __launch_bounds__(256) fill_int_kernel(int* __restrict__ p, int64_t n)
{
    int64_t const i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// exclusive scan over kScatT threads; every wave's total passes through LDS
__device__ __forceinline__ int scan_threads(int sum, int& total)
{
    constexpr int kWaves = kScatT / 64;
    __shared__ int part[kWaves];
    int const lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int incl = sum;
#pragma unroll
    for (int s = 1; s < 64; s *= 2) {
        int const v = __shfl_up(incl, s);
        incl += lane >= s ? v : 0;
    }
    if (lane == 63) part[wave] = incl;
    __syncthreads();
    int run = incl - sum;
    total = 0;
#pragma unroll
    for (int v = 0; v < kWaves; ++v) {
        int const pv = part[v];
        run += v < wave ? pv : 0;
        total += pv;
    }
    return run;
}

// exclusive scan of one batch entry's counts, [group][tile], in the order tile,
// group (nbins <= 4096, 1024 threads, 4 tiles each); starts gets the nbins + 1
// tile offsets, cursor every group's offset within its tile's range
__global__ void __launch_bounds__(kScatT) bin_scan_kernel(int nbins, int groups, const int* __restrict__ counts,
                                                          int* __restrict__ starts, int* __restrict__ cursor)
{
    int64_t const l = blockIdx.x;
    int const t = threadIdx.x;
    const int* const cl = counts + l * nbins * groups;
    int* const ol = cursor + l * nbins * groups;
    int c[4][kGroups];
    int sum = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int g = 0; g < kGroups; ++g) {
            c[u][g] = g < groups && 4 * t + u < nbins ? cl[g * nbins + 4 * t + u] : 0;
            sum += c[u][g];
        }
    int total;
    int run = scan_threads(sum, total);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        int const k = 4 * t + u;
        if (k < nbins) starts[l * (nbins + 1) + k] = run;
#pragma unroll
        for (int g = 0; g < kGroups; ++g) {
            if (g < groups && k < nbins) ol[g * nbins + k] = run;
            run += c[u][g];
        }
    }
    if (t == 0) starts[l * (nbins + 1) + nbins] = total;
}

// LDS of a scatter workgroup with records of rw doubles: the records in tile
// order, the tile histogram (then each tile's global minus local offset) and
// the local tile offsets, nbins ints each, and per slot its tile and local
// index
constexpr size_t scatter_lds(int nbins, int rw)
{
    return size_t(kChunk) * rw * sizeof(double) + size_t(2) * nbins * sizeof(int) + size_t(kChunk) * 2 * sizeof(uint16_t);
}
static_assert(scatter_lds(kMaxBins, 3) + 1024 <= kLdsBytes, "the scatter's records and tables fit in LDS");

template <int NX, bool W>
__global__ void __launch_bounds__(kScatT) bin_scatter_kernel(int nbins, int groups, const double* __restrict__ coords,
                                                             const double* __restrict__ w, int64_t npts, int64_t bpb,
                                                             int* __restrict__ cursor, int* __restrict__ perm,
                                                             double* __restrict__ recs,
                                                             const uint16_t* __restrict__ bins)
{
    constexpr int PTS = kScatPts, NP = kChunk;
    constexpr int RW = NX + (W ? 1 : 0);
    constexpr int kPer = kMaxBins / kScatT; // tiles per thread in the scan
    static_assert(NP <= 65536 && kMaxBins <= 65536, "slot tile and local index are 16-bit");
    extern __shared__ double srec[];
    int* const hist = reinterpret_cast<int*>(srec + RW * NP);
    int* const lofs = hist + nbins;
    uint16_t* const sbin = reinterpret_cast<uint16_t*>(lofs + nbins);
    uint16_t* const sloc = sbin + NP;
    int const tid = threadIdx.x;
    int64_t const l = blockIdx.x / bpb;
    int64_t const p0 = (blockIdx.x % bpb) * int64_t(NP);
    int* const cg = cursor + (l * groups + blockIdx.x % groups) * nbins;
    for (int k = tid; k < nbins; k += kScatT) hist[k] = 0;
    double rv[PTS][RW];
    int bin[PTS], rank[PTS];
#pragma unroll
    for (int u = 0; u < PTS; ++u) {
        int64_t const p = p0 + u * kScatT + tid;
        int const b = bins[l * npts + (p < npts ? p : npts - 1)];
        bin[u] = p < npts && b != kNoBin ? b : -1;
    }
#pragma unroll
    for (int u = 0; u < PTS; ++u) {
        int64_t const p = p0 + u * kScatT + tid;
        int64_t const t = l * npts + (p < npts ? p : npts - 1);
#pragma unroll
        for (int k = 0; k < NX; ++k) rv[u][k] = coords[NX * t + k];
        if constexpr (W) rv[u][NX] = w[t];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PTS; ++u) rank[u] = bin[u] >= 0 ? atomicAdd(&hist[bin[u]], 1) : 0;
    __syncthreads();
    // local exclusive offsets: thread t takes tiles [t*per, (t+1)*per); its
    // reservations in the tiles' global ranges are requested first and needed
    // only after the records are in LDS
    int const per = (nbins + kScatT - 1) / kScatT;
    int const kb = tid * per;
    int cnt[kPer], base[kPer];
    int sum = 0;
#pragma unroll
    for (int v = 0; v < kPer; ++v) {
        cnt[v] = v < per && kb + v < nbins ? hist[kb + v] : 0;
        base[v] = cnt[v] ? atomicAdd(&cg[kb + v], cnt[v]) : 0;
        sum += cnt[v];
    }
    int total;
    int run = scan_threads(sum, total);
    int first[kPer];
#pragma unroll
    for (int v = 0; v < kPer; ++v) {
        first[v] = run;
        if (v < per && kb + v < nbins) lofs[kb + v] = run;
        run += cnt[v];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PTS; ++u)
        if (bin[u] >= 0) {
            int const j = lofs[bin[u]] + rank[u];
#pragma unroll
            for (int k = 0; k < RW; ++k) srec[RW * j + k] = rv[u][k];
            sbin[j] = uint16_t(bin[u]);
            sloc[j] = uint16_t(u * kScatT + tid);
        }
    // every thread has read the counts it needs: they become the offsets
#pragma unroll
    for (int v = 0; v < kPer; ++v)
        if (cnt[v]) hist[kb + v] = base[v] - first[v];
    __syncthreads();
    int* const pl = perm + l * npts;
    double* const rl = recs + RW * (l * npts);
    for (int j = tid; j < total; j += kScatT) pl[j + hist[sbin[j]]] = int(p0 + sloc[j]);
    // one double per lane: the lanes of a wave write whole runs
    for (int i = tid; i < RW * total; i += kScatT) {
        int const j = int(unsigned(i) / RW);
        rl[i + int64_t(RW) * hist[sbin[j]]] = srec[i];
    }
}

// The workspace: counts, starts, cursor (per batch entry and tile; counts and
// cursor per group as well), then per point its index in tile order, its record
// (rw doubles) and its tile.
struct Work {
    int* counts;
    int* starts;
    int* cursor;
    int* perm;
    double* recs;
    uint16_t* bins;
    int groups;
    int64_t bytes;
};

// One group where an entry has fewer than 64 chunks: few workgroups per XCD
// then append to one tile, and the counts would outgrow the points.
int groups_for(int64_t npts)
{
    return npts >= int64_t(64) * kChunk ? kGroups : 1;
}

Work carve(int nbins, int rw, int64_t npts, int64_t nbatch, void* base, int groups)
{
    auto up = [](int64_t n, int64_t size) { return (n * size + 255) / 256 * 256; };
    int64_t const a = up(nbatch * nbins * groups, 4), b = up(nbatch * (nbins + 1), 4), c = a,
                  d = up(nbatch * npts, 4), e = up(rw * nbatch * npts, 8), f = up(nbatch * npts, 2);
    char* p = static_cast<char*>(base);
    return Work{reinterpret_cast<int*>(p),
                reinterpret_cast<int*>(p + a),
                reinterpret_cast<int*>(p + a + b),
                reinterpret_cast<int*>(p + a + b + c),
                reinterpret_cast<double*>(p + a + b + c + d),
                reinterpret_cast<uint16_t*>(p + a + b + c + d + e),
                groups,
                a + b + c + d + e + f};
}

// the most groups whose workspace fits in work_bytes (one group fits in the
// least size a caller may bring)
Work carve_within(int nbins, int rw, int64_t npts, int64_t nbatch, void* base, int64_t work_bytes)
{
    Work const w = carve(nbins, rw, npts, nbatch, base, groups_for(npts));
    return w.bytes <= work_bytes ? w : carve(nbins, rw, npts, nbatch, base, 1);
}

unsigned grid_blocks(int64_t n, int threads)
{
    int64_t const b = (n + threads - 1) / threads;
    if (b > int64_t(0x7fffffff)) throw Error(DDCX_ERR_INVALID, "batch too large for one launch");
    return unsigned(b);
}

// scan the counts and scatter the records
template <int NX, bool W>
void scan_and_scatter(int nbins, const double* coords, const double* w, int64_t npts, int64_t nbatch,
                      Work const& ws, hipStream_t stream)
{
    hipLaunchKernelGGL(bin_scan_kernel, dim3(unsigned(nbatch)), dim3(kScatT), 0, stream, nbins, ws.groups, ws.counts,
                       ws.starts, ws.cursor);
    size_t const lds = scatter_lds(nbins, NX + (W ? 1 : 0));
    auto kern = bin_scatter_kernel<NX, W>;
    hip_check(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  int(lds)),
              "hipFuncSetAttribute");
    int64_t const bpb = (npts + kChunk - 1) / kChunk;
    hipLaunchKernelGGL(kern, dim3(grid_blocks(bpb * nbatch, 1)), dim3(kScatT), lds, stream, nbins, ws.groups, coords,
                       w, npts, bpb, ws.cursor, ws.perm, ws.recs, ws.bins);
}

} // namespace
} // namespace binning
} // namespace ddcx
