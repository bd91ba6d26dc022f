// digit_raw_wide.hip -- digit_kernel.hpp for int4 streams read as nibbles, dims
// above 128.
#include "digit_kernel.hpp"

namespace msim {
namespace digit {

hipError_t launch_raw_wide(const ScoreArgs& a, bool residual, int reducer, dim3 grid, hipStream_t s) {
  if (a.chunks == 2) {
    if (residual) return launch_reducer<kDocInt4, true, 2, 2, true>(a, reducer, grid, s);
    return launch_reducer<kDocInt4, false, 2, 2, true>(a, reducer, grid, s);
  }
  if (a.chunks != 4) return hipErrorInvalidValue;
  if (residual) return launch_reducer<kDocInt4, true, 2, 4, true>(a, reducer, grid, s);
  return launch_reducer<kDocInt4, false, 2, 4, true>(a, reducer, grid, s);
}

}  // namespace digit
}  // namespace msim
