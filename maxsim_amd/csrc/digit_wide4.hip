// digit_wide4.hip -- digit_kernel.hpp for 257 to 512 dims (four 128-dim chunks).
#include "digit_kernel.hpp"

namespace msim {
namespace digit {

hipError_t launch_wide4(const ScoreArgs& a, int doc, bool residual, int nt, int reducer, dim3 grid, hipStream_t s) {
  if (doc == kDocSign) {
    if (residual) return hipErrorInvalidValue;
    if (nt == 1) return launch_reducer<kDocSign, false, 1, 4>(a, reducer, grid, s);
    return launch_reducer<kDocSign, false, 2, 4>(a, reducer, grid, s);
  }
  if (residual) return launch_wide4_residual(a, nt, reducer, grid, s);
  if (nt == 1) return launch_reducer<kDocInt4, false, 1, 4>(a, reducer, grid, s);
  return launch_reducer<kDocInt4, false, 2, 4>(a, reducer, grid, s);
}

}  // namespace digit
}  // namespace msim
