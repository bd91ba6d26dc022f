// digit_wide4r.hip -- digit_kernel.hpp for int4 documents of 257 to 512 dims
// with an int4 residual stream.
#include "digit_kernel.hpp"

namespace msim {
namespace digit {

hipError_t launch_wide4_residual(const ScoreArgs& a, int nt, int reducer, dim3 grid, hipStream_t s) {
  if (nt == 1) return launch_reducer<kDocInt4, true, 1, 4>(a, reducer, grid, s);
  return launch_reducer<kDocInt4, true, 2, 4>(a, reducer, grid, s);
}

}  // namespace digit
}  // namespace msim
