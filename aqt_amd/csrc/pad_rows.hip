// Rows of a contraction operand copied to 16-byte aligned rows whose length is a multiple of 16, the added bytes zero.
// What the MFMA kernels load in 16-byte pieces may then have any contraction length and any start: a zero byte is the
// value 0 in int8, e4m3 and e5m2 alike, so the longer contraction has the same products.
// Bound by HBM bytes on large operands (each read once, written once), by the launch on small ones; both operands
// of a contraction go in one launch.  A thread moves one 16-byte piece: the store is aligned, the load is one
// unaligned 16-byte load, the last piece of a row byte by byte.
// 1999 x 3001 outputs, k = 1030 (int8): this copy and the MFMA kernel take 27 us, one thread per output element, which
// reads both operands a byte at a time, 21.9 ms; 128 x 128 x 129: 8 against 12 us.
#include "common.h"

namespace aqtx {
namespace {

struct PadSide {
  const uint8_t* src;
  uint8_t* dst;
  int64_t rows, ld, stride;  // of src, in bytes
};

struct PadArgs {
  PadSide side[2];
  int64_t k;
  int32_t pieces;  // 16-byte pieces of an output row
};

__global__ __launch_bounds__(256) void pad_rows_kernel(const PadArgs a) {
  const PadSide& s = a.side[blockIdx.z];
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = i / a.pieces;
  if (row >= s.rows) return;
  const int64_t k0 = (i - row * a.pieces) * 16;
  const uint8_t* src = s.src + blockIdx.y * s.stride + row * s.ld + k0;
  uint4 v = make_uint4(0u, 0u, 0u, 0u);
  if (k0 + 16 <= a.k) {
    __builtin_memcpy(&v, src, 16);
  } else {
    uint32_t w[4] = {0u, 0u, 0u, 0u};
    const int left = (int)(a.k - k0);
#pragma unroll
    for (int e = 0; e < 15; ++e)
      if (e < left) w[e >> 2] |= (uint32_t)src[e] << (8 * (e & 3));
    v = make_uint4(w[0], w[1], w[2], w[3]);
  }
  *reinterpret_cast<uint4*>(s.dst + ((int64_t)blockIdx.y * s.rows * a.pieces + i) * 16) = v;
}

}  // namespace
}  // namespace aqtx

using namespace aqtx;

extern "C" int aqtx_pad_rows(int64_t batch, int64_t k, const void* a, int64_t rows_a, int64_t lda, int64_t stride_a,
                             void* a_out, const void* b, int64_t rows_b, int64_t ldb, int64_t stride_b, void* b_out,
                             void* stream) {
  clear_error();
  AQTX_REQUIRE(batch >= 0 && k >= 0 && rows_a >= 0 && rows_b >= 0, "aqtx_pad_rows: negative shape");
  AQTX_REQUIRE(lda >= k && (b_out == nullptr || ldb >= k), "aqtx_pad_rows: leading dimension smaller than the row length");
  AQTX_REQUIRE(batch <= 65535 && k < (1ll << 31) - 16, "aqtx_pad_rows: shape too large for one launch");
  const int64_t pieces = (k + 15) / 16, rows = b_out != nullptr && rows_b > rows_a ? rows_b : rows_a;
  if (batch == 0 || rows == 0 || k == 0) return 0;
  AQTX_REQUIRE((rows_a == 0 || (a != nullptr && a_out != nullptr)) && (b_out == nullptr || rows_b == 0 || b != nullptr),
               "aqtx_pad_rows: NULL buffer");
  AQTX_REQUIRE(((uintptr_t)a_out % 16) == 0 && ((uintptr_t)b_out % 16) == 0, "aqtx_pad_rows: outputs must be 16-byte aligned");
  const int64_t blocks = (rows * pieces + 255) / 256;
  AQTX_REQUIRE(rows < (1ll << 40) && blocks < (1ll << 31), "aqtx_pad_rows: shape too large for one launch");
  PadArgs g{};
  g.side[0] = PadSide{reinterpret_cast<const uint8_t*>(a), reinterpret_cast<uint8_t*>(a_out), rows_a, lda, stride_a};
  g.side[1] = PadSide{reinterpret_cast<const uint8_t*>(b), reinterpret_cast<uint8_t*>(b_out), b_out != nullptr ? rows_b : 0, ldb, stride_b};
  g.k = k;
  g.pieces = (int32_t)pieces;
  pad_rows_kernel<<<dim3((unsigned)blocks, (unsigned)batch, b_out != nullptr ? 2 : 1), 256, 0, reinterpret_cast<hipStream_t>(stream)>>>(g);
  AQTX_HIP_CHECK_LAUNCH("pad_rows_kernel");
  return 0;
}
