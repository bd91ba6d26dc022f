// digit_raw.hip -- digit_kernel.hpp for int4 streams read as nibbles, at most 128
// dims.  (No kernel of 16 rows: it is bound by memory and the decoding, 8 tokens
// take what 32 do.)
#include "digit_kernel.hpp"

namespace msim {
namespace digit {

hipError_t launch_raw(const ScoreArgs& a, int doc, bool residual, int nt, int reducer, dim3 grid, hipStream_t s) {
  if (a.chunks > 1) return doc == kDocSign ? hipErrorInvalidValue : launch_raw_wide(a, residual, nt, reducer, grid, s);
  if (doc == kDocSign) {
    if (!residual || reducer != kRedMax) return hipErrorInvalidValue;
    if (nt <= 2) return launch_mode<kDocSign, true, 2, kRedMax, 1, false, true>(a, grid, s);
    return launch_mode<kDocSign, true, 4, kRedMax, 1, false, true>(a, grid, s);
  }
  if (residual) {
    if (nt <= 2) return launch_reducer<kDocInt4, true, 2, 1, true>(a, reducer, grid, s);
    return launch_reducer<kDocInt4, true, 4, 1, true>(a, reducer, grid, s);
  }
  if (nt <= 2) return launch_reducer<kDocInt4, false, 2, 1, true>(a, reducer, grid, s);
  return launch_reducer<kDocInt4, false, 4, 1, true>(a, reducer, grid, s);
}

}  // namespace digit
}  // namespace msim
