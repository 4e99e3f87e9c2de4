// Window spread kernels for float, 2D.
#include "win_impl.inl"
CFA_INSTANTIATE_WIN_SPREAD(float, 2)
