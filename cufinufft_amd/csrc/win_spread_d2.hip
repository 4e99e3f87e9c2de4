// Window spread kernels for double, 2D.
#include "win_impl.inl"
CFA_INSTANTIATE_WIN_SPREAD(double, 2)
namespace cfa {
template <>
int run_win_group<double>(int ns, const void *items, const int2 *map, int waves,
                         const KerParams<double> &kp, const Launch &L)
{
    return win_group_ns<double>(ns, items, map, waves, kp, L);
}
}  // namespace cfa
