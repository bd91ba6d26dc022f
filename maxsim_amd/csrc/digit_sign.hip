// digit_sign.hip -- digit_kernel.hpp for sign documents of at most 128 dims,
// with or without an int4 residual stream.
#include "digit_kernel.hpp"

namespace msim {
namespace digit {

hipError_t launch_sign(const ScoreArgs& a, bool residual, int nt, int reducer, dim3 grid, hipStream_t s) {
  if (residual) {
    // The binary-prefix + int4-residual format is MaxSim only.
    if (reducer != kRedMax) return hipErrorInvalidValue;
    if (nt == 1) return launch_mode<kDocSign, true, 1, kRedMax, 1>(a, grid, s);
    if (nt == 2) return launch_mode<kDocSign, true, 2, kRedMax, 1>(a, grid, s);
    return launch_mode<kDocSign, true, 4, kRedMax, 1>(a, grid, s);
  }
  if (a.unit_tscale && reducer == kRedMax) {
    if (nt == 1) return launch_mode<kDocSign, false, 1, kRedMax, 1, true>(a, grid, s);
    if (nt == 2) return launch_mode<kDocSign, false, 2, kRedMax, 1, true>(a, grid, s);
    return launch_mode<kDocSign, false, 4, kRedMax, 1, true>(a, grid, s);
  }
  if (nt == 1) return launch_reducer<kDocSign, false, 1, 1>(a, reducer, grid, s);
  if (nt == 2) return launch_reducer<kDocSign, false, 2, 1>(a, reducer, grid, s);
  return launch_reducer<kDocSign, false, 4, 1>(a, reducer, grid, s);
}

}  // namespace digit
}  // namespace msim
