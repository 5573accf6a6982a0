// okf_fmt_grid.hip -- the launchers (and with them the kernels) of IQ2_XS, IQ2_S, IQ3_XXS.
#include "okf_impl.h"

namespace okf_impl {
OKF_INSTANTIATE(IQ2_XS)
OKF_INSTANTIATE(IQ2_S)
OKF_INSTANTIATE(IQ3_XXS)
}  // namespace okf_impl
