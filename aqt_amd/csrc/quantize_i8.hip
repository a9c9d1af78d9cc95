// The quantize kernels on int8 input.
#include "quantize_core.h"

namespace aqtx {
int launch_quantize_i8(const QArgs& a, int reduce, int partitionable, int64_t nscales, hipStream_t st) {
  return dispatch<int8_t>(a, reduce, partitionable, nscales, st);
}
}  // namespace aqtx
