// Window spread kernels for float, 2D.
#include "win_impl.inl"
CFA_INSTANTIATE_WIN_SPREAD(float, 2)
namespace cfa {
template <>
int run_win_group<float>(int ns, const void *items, const int2 *map, int waves,
                         const KerParams<float> &kp, const Launch &L)
{
    return win_group_ns<float>(ns, items, map, waves, kp, L);
}
}  // namespace cfa
