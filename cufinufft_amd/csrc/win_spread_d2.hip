// Window spread kernels for double, 2D.
#include "win_impl.inl"
CFA_INSTANTIATE_WIN_SPREAD(double, 2)
