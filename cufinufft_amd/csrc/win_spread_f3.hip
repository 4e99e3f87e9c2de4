// Window spread kernels for float, 3D.
#include "win_impl.inl"
CFA_INSTANTIATE_WIN_SPREAD(float, 3)
