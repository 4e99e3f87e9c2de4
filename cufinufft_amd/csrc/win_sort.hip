// setpts for the window kernels (win_device.cuh): the rule that chooses them
// and the order of the points by window.
//
// The bin sort leaves the points in bins.  Here they are counted per window and
// placed in window order, each with what the window kernels need (offsets of the
// first tap, its place inside the window, the input index), so execute streams 20
// bytes per 3D FP32 point (28 with positions and index).  A workgroup takes 1024
// consecutive points of the bin order, which lie in few windows: it counts them
// in an LDS hash table and does one global atomic per window instead of one per
// point (random global atomics run at 2e10 per second).
#include <algorithm>

#include "nufft_launch.h"
#include "win_device.cuh"

namespace cfa {

constexpr int kWinChunk = 1024;  // points per workgroup
constexpr int kWinSlots = 2048;  // hash slots: at most half are used

// PLACE = false: count[key] += the points of each key.  PLACE = true: writes
// the points to start[key] + what is left of count[key], which returns to zero.
template <typename T, int DIM, bool PLACE>
__global__ void __launch_bounds__(512)
k_win_keys(int M, SortedPts sp, WinGeom wg, int *__restrict__ count,
           const int *__restrict__ start, T *__restrict__ xo, unsigned *__restrict__ sho,
           int *__restrict__ ido, long long stride)
{
    constexpr int BT = 512, PP = kWinChunk / BT;
    __shared__ int hk[kWinSlots], hc[kWinSlots];
    const int tid = threadIdx.x;
    for (int k = tid; k < kWinSlots; k += BT) {
        hk[k] = -1;
        hc[k] = 0;
    }
    double v[PP][DIM];
    int id[PP];
#pragma unroll
    for (int j = 0; j < PP; ++j) {
        const int i = min(M - 1, (int)blockIdx.x * kWinChunk + j * BT + tid);
#pragma unroll
        for (int d = 0; d < DIM; ++d) v[j][d] = sp.pos[d * sp.stride + i];
        if (PLACE) id[j] = sp.idx[i];
    }
    __syncthreads();
    int slot[PP], rank[PP];
    unsigned sh[PP];
    T x1[PP][DIM];
#pragma unroll
    for (int j = 0; j < PP; ++j) {
        slot[j] = -1;
        if ((int)blockIdx.x * kWinChunk + j * BT + tid >= M) continue;
        int kw[3] = {0, 0, 0};
        sh[j] = 0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            const int u = win_place<T>(v[j][d], wg.ns, x1[j][d]);
            kw[d] = u / wg.S[d];
            sh[j] |= (unsigned)(u - kw[d] * wg.S[d]) << (8 * d);
        }
        const int key = win_key<DIM>(wg, kw);
        unsigned h = (unsigned)key * 2654435761u >> 21;
        for (;;) {
            const int old = atomicCAS(&hk[h], -1, key);
            if (old == -1 || old == key) break;
            h = (h + 1) & (kWinSlots - 1);
        }
        slot[j] = (int)h;
        rank[j] = atomicAdd(&hc[h], 1);
    }
    __syncthreads();
    for (int k = tid; k < kWinSlots; k += BT) {
        const int n = hc[k];
        if (n == 0) continue;
        if (PLACE)
            hc[k] = start[hk[k]] + atomicSub(&count[hk[k]], n) - n;
        else
            atomicAdd(&count[hk[k]], n);
    }
    if (!PLACE) return;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PP; ++j) {
        if (slot[j] < 0) continue;
        const int o = hc[slot[j]] + rank[j];
        sho[o] = sh[j];
        ido[o] = id[j];
#pragma unroll
        for (int d = 0; d < DIM; ++d) xo[d * stride + o] = x1[j][d];
    }
}

static __global__ void __launch_bounds__(256)
k_win_ranges(int M, int nkeys, int ranges, int *__restrict__ start, const int *__restrict__ used,
             int2 *__restrict__ range)
{
    const int r = blockIdx.x * 256 + threadIdx.x;
    if (r == 0) start[nkeys] = M;
    if (r <= ranges) {
        const int p = win_range_start(start, used, nkeys, M, r, ranges);
        range[r] = make_int2(p, win_key_of(start, nkeys, p));
    }
}

// Where the window kernels beat the per-point ones, the window order's own time
// (25 - 35 us for small sets, 15 - 25 ns per 1000 points) in every call included.
// Measured per-point -> window, setpts and execute, uniform points:
//  3D type 1, 48^3 modes: FP32 ns 5, 4e4 points 180 -> 202 us, 2e5 211 -> 169; ns 6,
//   4e4 199 -> 177, 1e4 170 -> 247; ns 7, 1e4 342 -> 277; FP64 ns 7, 1e4 322 -> 315,
//   ns 10 608 -> 471.  128^3: FP32 ns 6, 3e5 1409 -> 554; FP64 ns 10, 2e6 8520 -> 2128.
//   ns 4: dense grids have too few taps per point (spread alone 0.62 -> 0.68 ms).
//  3D type 2 reads a window's cells once whatever its points: FP32, 48^3, 2e5 points,
//   ns 5 172 -> 168, ns 7 222 -> 199, ns 6, 4e4 156 -> 206; 128^3, 3e5, ns 6 (1.7
//   points per window) 512 -> 504.  FP64 ns 7, 128^3, 3e5 (0.7) 929 -> 1082, 2e6 (4.7)
//   2903 -> 1430; ns 10, 4e4 (0.14) 1007 -> 923, 48^3, 4e4 369 -> 369; ns 13, 48^3, 4e4
//   731 -> 700, 1e4 712 -> 834, 128^3, 3e5 (0.27) 3863 -> 2718.
//  2D type 1: FP32 ns 7, 640^2 modes, 1e6 183 -> 187, 4e6 404 -> 377, ns 6, 4e6 352 ->
//   365; FP64 ns 7, 1e6 240 -> 235, 4e6 561 -> 533; ns 10, 256^2, 3e5 108 -> 97, 640^2,
//   2e5 (5.9 per window) 204 -> 203; ns 13, 640^2, 2e5 (1.9) 226 -> 234, 1e6 (9.7) 345
//   -> 298, 256^2, 1e5 80 -> 98.  32 FP32 transforms, ns 7, 2e6: 3.7 -> 1.5 ms; 4
//   transforms of 2e5: 122 -> 138 us.
//  2D type 2: FP32 ns 7, 640^2, 1e6 182 -> 187, 4e6 445 -> 409, ns 6, 4e6 383 -> 400;
//   4 transforms, 320^2, 2e5, ns 5 118 -> 111, ns 7 160 -> 116; FP64 ns 7, 1e6 222 ->
//   246, 4e6 657 -> 557; ns 10, 256^2, 1e5 78 -> 84, 3e5 116 -> 110, 640^2, 2e5 (5.9)
//   208 -> 189; ns 13, 640^2, 2e5 (1.9) 242 -> 246, 1e6 436 -> 315.
static bool win_pays(int type, int dim, int ns, int elem, int M, int ntr, double per_window)
{
    const bool dbl = elem == 8;
    if (dim == 3 && type == 1) {
        if (ns >= 7) return M >= 10000;
        if (dbl) return M >= 20000;
        return ns == 6 ? M >= 40000 : ns == 5 && M >= 150000;
    }
    if (dim == 3) {
        if (dbl && ns >= 9) return M >= 50000 && per_window >= 0.1;
        if (dbl) return M >= 200000 && per_window >= 4;
        return ns >= 5 && M >= 200000 && per_window >= 1.5;
    }
    const double taps = (double)M * ntr * ns * ns;
    if (dbl && ns >= 9) return per_window >= 5 && taps >= (type == 1 ? 3e7 : 2e7);
    if (type == 1) return per_window >= 50 && taps >= 1.5e8 && (ns >= 7 || ntr >= 4);
    if (per_window < 10) return false;
    if (ntr >= 4 && ns >= 5) return taps >= 2e7;
    return ns >= 7 ? taps >= 1.5e8 : ns == 6 && taps >= 4e8;
}

WinGeom win_choose(int type, int dim, int ns, int elem, const BinGeom &g, int M, int ntr, int ncu)
{
    WinGeom w, none;
    if (dim < 2 || M <= 0) return none;
    if (!(type == 1 ? win_spread_width(dim, ns, elem) : win_interp_width(dim, ns, elem)))
        return none;
    if (!win_windows(type, dim, ns, g.nf, w)) return none;
    if (!win_pays(type, dim, ns, elem, M, ntr, (double)M / w.nkeys))
        return none;
    // One wave per range.  Interp: up to 8 rounds of the waves resident on the
    // device (16 per CU FP32, 8 FP64), no fewer than 128 points each.  Spread: a
    // range flushes a whole window at its end, so ranges grow to 1536 points before
    // there are more than half a round of them, and stop at 4 rounds.  2D spread:
    // one round (half a round: 0.326 -> 0.298 ms, FP32, ns 7, 1e7 points; two rounds
    // cost 32 coils of 2e6 points 1.27 -> 1.49 ms in flushes).
    const int resident = ncu * (elem == 4 ? 16 : 8);
    if (dim == 2 && type == 1)
        w.ranges = std::max(1, std::min(resident, M / 128));
    else if (type == 2)
        w.ranges = std::max(1, std::min(8 * resident, M / 128));
    else
        w.ranges = std::max({1, std::min(resident / 2, M / 128),
                             std::min(4 * resident, M / 1536)});
    return w;
}

// A 2D type-1 plan group spreads by window wherever the kernels are built (the order
// is made with the group): 48 images of 64^2 to 512^2 with up to 1e6 points each,
// FP32, ns 7, took 788 us by the subproblem kernel and 516 us by window (whole
// group), ns 5: 706 and 482; with up to 1e4 points, 2 per window, 527 and 319; 5
// images, 114 and 112; 30 FP64 images, ns 10, up to 3e5 points, 528 and 375.
WinGeom win_member(int ns, int elem, const BinGeom &g, int M, double &work)
{
    WinGeom w, none;
    if (M <= 0 || !win_spread_width(2, ns, elem) || !win_windows(1, 2, ns, g.nf, w)) return none;
    w.ranges = 1;
    work = M + 24.0 * std::min(M, w.nkeys);
    return w;
}

int run_win_clear(const SortBufs &sb, long long keys, const Launch &L)
{
    const long long b = (keys + 255) / 256;
    k_fill_int<<<(unsigned)(b < 4096 ? b : 4096), 256, 0, L.stream>>>(keys, 0, sb.wcount);
    return hipGetLastError() == hipSuccess ? 0 : kErrHip;
}

template <typename T>
int run_win_sort(int dim, int M, const SortBufs &sb, const Launch &L)
{
    const WinGeom &w = sb.win;
    const int nparts = (w.nkeys + kScanChunk - 1) / kScanChunk;
    int2 *part = static_cast<int2 *>(sb.wpart);
    const SortedPts sp{sb.idx, sb.pos, sb.pos_stride};
    const int gc = (M + kWinChunk - 1) / kWinChunk;
    T *x = static_cast<T *>(sb.wx);
    if (dim == 2)
        k_win_keys<T, 2, false><<<gc, 512, 0, L.stream>>>(M, sp, w, sb.wcount, nullptr, nullptr,
                                                          nullptr, nullptr, 0);
    else
        k_win_keys<T, 3, false><<<gc, 512, 0, L.stream>>>(M, sp, w, sb.wcount, nullptr, nullptr,
                                                          nullptr, nullptr, 0);
    // first points, and with a "subproblem" of 2^30 points the used windows
    constexpr int kAny = 1 << 30;
    k_scan_reduce<<<nparts, kScanThreads, 0, L.stream>>>(sb.wcount, w.nkeys, kAny, part);
    k_scan_parts<<<1, kScanThreads, 0, L.stream>>>(part, nparts,
                                                   reinterpret_cast<int *>(part + nparts),
                                                   sb.wused + w.nkeys);
    k_scan_apply<<<nparts, kScanThreads, 0, L.stream>>>(sb.wcount, w.nkeys, kAny, part, sb.wstart,
                                                        sb.wused);
    k_win_ranges<<<w.ranges / 256 + 1, 256, 0, L.stream>>>(M, w.nkeys, w.ranges, sb.wstart,
                                                           sb.wused, sb.wrange);
    if (dim == 2)
        k_win_keys<T, 2, true><<<gc, 512, 0, L.stream>>>(M, sp, w, sb.wcount, sb.wstart, x, sb.wsh,
                                                         sb.widx, sb.pos_stride);
    else
        k_win_keys<T, 3, true><<<gc, 512, 0, L.stream>>>(M, sp, w, sb.wcount, sb.wstart, x, sb.wsh,
                                                         sb.widx, sb.pos_stride);
    return hipGetLastError() == hipSuccess ? 0 : kErrHip;
}

template int run_win_sort<float>(int, int, const SortBufs &, const Launch &);
template int run_win_sort<double>(int, int, const SortBufs &, const Launch &);

}  // namespace cfa
