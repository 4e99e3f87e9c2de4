// Window interp kernels for float, 3D.
#include "win_impl.inl"
CFA_INSTANTIATE_WIN_INTERP(float, 3)
