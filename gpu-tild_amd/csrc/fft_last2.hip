// fft_last2.hip -- k_last_reg for longer axes, one or two types (and those of fft_last0.hip).
#include "fft_last.hpp"

namespace tild {
TILD_LAST_REG_CLASS(2)
}  // namespace tild
