// The quantize kernels on float32 input.
#include "quantize_core.h"

namespace aqtx {
int launch_quantize_f32(const QArgs& a, int reduce, int partitionable, int64_t nscales, hipStream_t st) {
  return dispatch<float>(a, reduce, partitionable, nscales, st);
}
}  // namespace aqtx
