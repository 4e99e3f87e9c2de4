// Window interp kernels for double, 3D.
#include "win_impl.inl"
CFA_INSTANTIATE_WIN_INTERP(double, 3)
