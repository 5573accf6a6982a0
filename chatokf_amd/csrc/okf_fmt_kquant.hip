// okf_fmt_kquant.hip -- the launchers (and with them the kernels) of Q5_K, Q6_K.
#include "okf_impl.h"

namespace okf_impl {
OKF_INSTANTIATE(Q5_K)
OKF_INSTANTIATE(Q6_K)
}  // namespace okf_impl
