// RMSNorm launch shapes for many rows of any width (norm_tail.h), in a file of their own so that they
// compile beside the others.
#include "norm_tail.h"

namespace hyle_hip {

bool launch_norm_tail_rms(Elem type, const NormParams &p, const void *x, const void *w, void *y,
                          hipStream_t stream) {
  return run_tail_typed<false>(type, p, Bound{x, w, nullptr, y}, stream);
}

}  // namespace hyle_hip
