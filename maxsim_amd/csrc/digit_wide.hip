// digit_wide.hip -- digit_kernel.hpp for dims above 128: two 128-dim chunks up
// to 256 dims (32 query rows per pass), four up to 512 (16 rows).
#include "digit_kernel.hpp"

namespace msim {
namespace digit {

hipError_t launch_wide(const ScoreArgs& a, int doc, bool residual, int nt, int reducer, dim3 grid, hipStream_t s) {
  if (doc == kDocSign && residual) return hipErrorInvalidValue;
  if (a.chunks == 2) {
    if (doc == kDocSign) {
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
  if (a.chunks != 4 || nt != 1) return hipErrorInvalidValue;
  if (doc == kDocSign) return launch_reducer<kDocSign, false, 1, 4>(a, reducer, grid, s);
  if (residual) return launch_reducer<kDocInt4, true, 1, 4>(a, reducer, grid, s);
  return launch_reducer<kDocInt4, false, 1, 4>(a, reducer, grid, s);
}

}  // namespace digit
}  // namespace msim
