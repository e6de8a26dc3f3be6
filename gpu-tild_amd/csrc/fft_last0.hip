// fft_last0.hip -- k_last_reg for axes up to 100 points, one or two types.
#include "fft_last.hpp"

namespace tild {
TILD_LAST_REG_CLASS(0)
}  // namespace tild
