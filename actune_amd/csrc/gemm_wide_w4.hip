// The wide-tile kernel (gemm_wide.hpp) for W4 weights.
#include "gemm_wide.hpp"

namespace actune {

void launch_wide_w4(int A, int shape, const LinearArgs& g, hipStream_t st) { launch_wide_width<4>(A, shape, g, st); }

}  // namespace actune
