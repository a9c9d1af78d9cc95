// The quantize kernels on bf16 input.
#include "quantize_core.h"

namespace aqtx {
int launch_quantize_bf16(const QArgs& a, int reduce, int partitionable, int64_t nscales, hipStream_t st) {
  return dispatch<uint16_t>(a, reduce, partitionable, nscales, st);
}
}  // namespace aqtx
