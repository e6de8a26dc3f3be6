// fft_last3.hip -- k_last_reg for axes up to 100 points, one to four types, for sets that mix them.
#include "fft_last.hpp"

namespace tild {
TILD_LAST_REG_CLASS(3)
}  // namespace tild
