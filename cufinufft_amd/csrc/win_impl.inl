// Runtime-ns dispatch of the window kernels for one (T, DIM); included by the
// win_spread_<prec><dim>.hip and win_interp_<prec><dim>.hip translation units.
#include <algorithm>

#include "nufft_launch.h"
#include "win_device.cuh"

namespace cfa {

namespace {

inline WinPts win_pts(const SortBufs &sb)
{
    return WinPts{sb.wx, sb.wsh, sb.widx, sb.wstart, sb.wrange, sb.pos_stride};
}
// Workgroups of 4 waves, a range each; whole XCD groups.
inline int win_grid(int ranges)
{
    const int grid = (ranges + 3) / 4;
    return grid >= kNumXcd ? (grid + kNumXcd - 1) / kNumXcd * kNumXcd : grid;
}

template <typename T, int DIM, int NS>
int win_spread_ns(int M, const SortBufs &sb, const cpx<T> *c, cpx<T> *fw, const BinGeom &g,
                  const KerParams<T> &kp, int ntr, long long nftot, const Launch &L)
{
    if constexpr (!win_spread_width(DIM, NS, sizeof(T))) {
        return 1;
    } else {
        const int grid = win_grid(sb.win.ranges);
        constexpr int P = DIM == 2 ? kWinPack / (int)sizeof(cpx<T>) : 1;
        if (DIM == 2 && ntr >= 4 && sb.wc) {
            cpx<T> *pk = static_cast<cpx<T> *>(sb.wc);
            for (int t = 0; t < ntr; t += P) {
                const int nt = std::min(P, ntr - t);
                k_win_pack<T, P><<<(M + 255) / 256, 256, 0, L.stream>>>(M, nt,
                                                                        c + (long long)t * M, pk);
                k_win_spread<T, DIM, NS, P><<<grid, 256, 0, L.stream>>>(
                    win_pts(sb), pk, 1, P, fw + t * nftot, g, sb.win, kp, nt, nftot);
            }
        } else if (DIM == 2 && ntr > 1) {
            k_win_spread<T, DIM, NS, DIM == 2 ? 4 : 1>
                <<<dim3(grid, (ntr + 3) / 4), 256, 0, L.stream>>>(win_pts(sb), c, M, 1, fw, g,
                                                                  sb.win, kp, ntr, nftot);
        } else {
            k_win_spread<T, DIM, NS, 1><<<dim3(grid, ntr), 256, 0, L.stream>>>(
                win_pts(sb), c, M, 1, fw, g, sb.win, kp, ntr, nftot);
        }
        return hipGetLastError() == hipSuccess ? 0 : kErrHip;
    }
}

template <typename T, int DIM, int NS>
int win_interp_ns(int M, const SortBufs &sb, cpx<T> *c, const cpx<T> *fw, const BinGeom &g,
                  const KerParams<T> &kp, int ntr, long long nftot, const Launch &L)
{
    if constexpr (!win_interp_width(DIM, NS, sizeof(T))) {
        return 1;
    } else {
        k_win_interp<T, DIM, NS><<<win_grid(sb.win.ranges), 256, 0, L.stream>>>(
            M, win_pts(sb), c, fw, g, sb.win, kp, ntr, nftot);
        return hipGetLastError() == hipSuccess ? 0 : kErrHip;
    }
}

}  // namespace

#ifndef CFA_NS_CASES
#define CFA_NS_CASES(F) F(4) F(5) F(6) F(7) F(8) F(9) F(10) F(11) F(12) F(13)
#endif

template <typename T, int DIM>
int win_spread_dim(int ns, int M, const SortBufs &sb, const cpx<T> *c, cpx<T> *fw,
                   const BinGeom &g, const KerParams<T> &kp, int ntr, long long nftot,
                   const Launch &L)
{
    switch (ns) {
#define CFA_CASE(N)                                                                          \
    case N:                                                                                  \
        return win_spread_ns<T, DIM, N>(M, sb, c, fw, g, kp, ntr, nftot, L);
        CFA_NS_CASES(CFA_CASE)
#undef CFA_CASE
    }
    return 1;
}

template <typename T>
int win_group_ns(int ns, const void *items, const int2 *map, int waves, const KerParams<T> &kp,
                 const Launch &L)
{
    const WinItem<T> *it = static_cast<const WinItem<T> *>(items);
    switch (ns) {
#define CFA_CASE(N)                                                                          \
    case N:                                                                                  \
        if constexpr (win_spread_width(2, N, sizeof(T)))                                     \
            k_win_spread_group<T, N><<<win_grid(waves), 256, 0, L.stream>>>(it, map, waves,  \
                                                                            kp);             \
        break;
        CFA_NS_CASES(CFA_CASE)
#undef CFA_CASE
    default:
        return 1;
    }
    return hipGetLastError() == hipSuccess ? 0 : kErrHip;
}

template <typename T, int DIM>
int win_interp_dim(int ns, int M, const SortBufs &sb, cpx<T> *c, const cpx<T> *fw,
                   const BinGeom &g, const KerParams<T> &kp, int ntr, long long nftot,
                   const Launch &L)
{
    switch (ns) {
#define CFA_CASE(N)                                                                          \
    case N:                                                                                  \
        return win_interp_ns<T, DIM, N>(M, sb, c, fw, g, kp, ntr, nftot, L);
        CFA_NS_CASES(CFA_CASE)
#undef CFA_CASE
    }
    return 1;
}

}  // namespace cfa

#define CFA_INSTANTIATE_WIN_SPREAD(T, DIM)                                                   \
    template int cfa::win_spread_dim<T, DIM>(int, int, const cfa::SortBufs &,                \
                                             const cfa::cpx<T> *, cfa::cpx<T> *,             \
                                             const cfa::BinGeom &, const cfa::KerParams<T> &, \
                                             int, long long, const cfa::Launch &);
#define CFA_INSTANTIATE_WIN_INTERP(T, DIM)                                                   \
    template int cfa::win_interp_dim<T, DIM>(int, int, const cfa::SortBufs &, cfa::cpx<T> *, \
                                             const cfa::cpx<T> *, const cfa::BinGeom &,      \
                                             const cfa::KerParams<T> &, int, long long,      \
                                             const cfa::Launch &);
