// fft_last1.hip -- k_last_reg for axes up to 100 points, three or four types.
#include "fft_last.hpp"

namespace tild {
TILD_LAST_REG_CLASS(1)
}  // namespace tild
