// digit_raw_wide.hip -- digit_kernel.hpp for int4 streams read as nibbles, dims
// above 128.  Kernels of 32 rows, and of 16 at four chunks, where the MFMAs of 16
// more rows cost 10 us of 65 (3,000 documents of 512 dims; two chunks: 1 of 41).
#include "digit_kernel.hpp"

namespace msim {
namespace digit {

hipError_t launch_raw_wide(const ScoreArgs& a, bool residual, int nt, int reducer, dim3 grid, hipStream_t s) {
  if (a.chunks == 2) {
    if (residual) return launch_reducer<kDocInt4, true, 2, 2, true>(a, reducer, grid, s);
    return launch_reducer<kDocInt4, false, 2, 2, true>(a, reducer, grid, s);
  }
  if (a.chunks != 4) return hipErrorInvalidValue;
  if (nt == 1) {
    if (residual) return launch_reducer<kDocInt4, true, 1, 4, true>(a, reducer, grid, s);
    return launch_reducer<kDocInt4, false, 1, 4, true>(a, reducer, grid, s);
  }
  if (residual) return launch_reducer<kDocInt4, true, 2, 4, true>(a, reducer, grid, s);
  return launch_reducer<kDocInt4, false, 2, 4, true>(a, reducer, grid, s);
}

}  // namespace digit
}  // namespace msim
