// digit_wide.hip -- digit_kernel.hpp for 129 to 256 dims (two 128-dim chunks).
#include "digit_kernel.hpp"

namespace msim {
namespace digit {

hipError_t launch_wide2(const ScoreArgs& a, int doc, bool residual, int nt, int reducer, dim3 grid, hipStream_t s) {
  if (doc == kDocSign) {
    if (residual) return hipErrorInvalidValue;
    if (nt == 1) return launch_reducer<kDocSign, false, 1, 2>(a, reducer, grid, s);
    return launch_reducer<kDocSign, false, 2, 2>(a, reducer, grid, s);
  }
  if (residual) {
    if (nt == 1) return launch_reducer<kDocInt4, true, 1, 2>(a, reducer, grid, s);
    return launch_reducer<kDocInt4, true, 2, 2>(a, reducer, grid, s);
  }
  if (nt == 1) return launch_reducer<kDocInt4, false, 1, 2>(a, reducer, grid, s);
  return launch_reducer<kDocInt4, false, 2, 2>(a, reducer, grid, s);
}

}  // namespace digit
}  // namespace msim
