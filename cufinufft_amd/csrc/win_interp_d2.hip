// Window interp kernels for double, 2D.
#include "win_impl.inl"
CFA_INSTANTIATE_WIN_INTERP(double, 2)
