// digit_int4.hip -- digit_kernel.hpp for int4 documents of at most 128 dims.
#include "digit_kernel.hpp"

namespace msim {
namespace digit {

hipError_t launch_int4(const ScoreArgs& a, bool residual, int nt, int reducer, dim3 grid, hipStream_t s) {
  if (residual) {
    if (nt == 1) return launch_reducer<kDocInt4, true, 1, 1>(a, reducer, grid, s);
    if (nt == 2) return launch_reducer<kDocInt4, true, 2, 1>(a, reducer, grid, s);
    return launch_reducer<kDocInt4, true, 4, 1>(a, reducer, grid, s);
  }
  if (nt == 1) return launch_reducer<kDocInt4, false, 1, 1>(a, reducer, grid, s);
  if (nt == 2) return launch_reducer<kDocInt4, false, 2, 1>(a, reducer, grid, s);
  return launch_reducer<kDocInt4, false, 4, 1>(a, reducer, grid, s);
}

}  // namespace digit
}  // namespace msim
