// Row offsets of a ragged contraction's groups from their sizes, and zeros in the output rows behind the last group.
// Bound by its launch: one takes the place of five of a few us each (zeros, cumulative sum, copies, clamp), and of a
// fill of the whole output, 30 us for 8192 x 14336 bf16 values, of which the contraction overwrites the rows of all groups.
// (Two bytes a lane, as rows of any length need, fill as fast as memory takes them: nothing but 8192 x 14336 int32 zeros, no
// row in any group, 102 us with the empty contraction; 100 with torch's fill and the launches it replaced.)
#include "common.h"

namespace aqtx {
namespace {

// Every block finds the covered rows itself.  Up to 128 groups: inclusive sums over one wave, 64 at a time.  More: eight sizes a thread, 2048
// at a time (64 at a time are a chain of a load and seven sums for each 64, 16 us for 2000 groups).
template <bool MANY>
__global__ __launch_bounds__(256) void ragged_prepare_kernel(const int32_t* __restrict__ sizes, int64_t groups, int64_t m,
                                                             int32_t* __restrict__ offsets, uint16_t* __restrict__ c, int64_t row_halves) {
  constexpr int kPer = MANY ? 8 : 1, kWaves = MANY ? 4 : 1;
  __shared__ int64_t wave_sum[kWaves], wave_most[kWaves];
  const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
  if (MANY || wave == 0) {
    int64_t before = 0, most = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) offsets[0] = 0;
    for (int64_t g0 = 0; g0 < groups; g0 += 64 * kWaves * kPer) {
      const int64_t mine = g0 + (int64_t)threadIdx.x * kPer;
      int32_t size[kPer];
      int64_t sum = 0;
#pragma unroll
      for (int u = 0; u < kPer; ++u) size[u] = mine + u < groups ? sizes[mine + u] : 0;
#pragma unroll
      for (int u = 0; u < kPer; ++u) sum += size[u];
      const int64_t own = sum;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int64_t up = __shfl_up(sum, off, 64);
        if (lane >= off) sum += up;
      }
      int64_t at = before + sum - own;
      if constexpr (MANY) {
        if (lane == 63) wave_sum[wave] = sum;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
          if (w < wave) at += wave_sum[w];
          before += wave_sum[w];
        }
      } else {
        before += __shfl(sum, 63, 64);
      }
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        at += size[u];
        int64_t end = (int64_t)(int32_t)at;
        if (end > m) end = m;
        if (mine + u < groups) {
          if (blockIdx.x == 0) offsets[mine + u + 1] = (int32_t)end;
          if (end > most) most = end;
        }
      }
      if constexpr (MANY) __syncthreads();  // the sums have been read
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const int64_t other = __shfl_xor(most, off, 64);
      most = other > most ? other : most;
    }
    if (lane == 0) wave_most[wave] = most;
  }
  __syncthreads();
  int64_t covered = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) covered = wave_most[w] > covered ? wave_most[w] : covered;
  const int64_t first = covered * row_halves, total = m * row_halves, stride = (int64_t)gridDim.x * 256;
  for (int64_t i = first + (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += stride) c[i] = 0;
}

}  // namespace
}  // namespace aqtx

using namespace aqtx;

extern "C" int aqtx_ragged_prepare(const int32_t* sizes, int64_t groups, int64_t m, int32_t* offsets, void* c,
                                   int64_t row_bytes, void* stream) {
  clear_error();
  AQTX_REQUIRE(groups >= 0 && m >= 0 && m < (1ll << 31) && row_bytes >= 0 && row_bytes % 2 == 0,
               "aqtx_ragged_prepare: negative or too large shape, or odd row bytes");
  AQTX_REQUIRE(offsets != nullptr && (sizes != nullptr || groups == 0) && (c != nullptr || m * row_bytes == 0),
               "aqtx_ragged_prepare: NULL buffer");
  AQTX_REQUIRE(((uintptr_t)sizes % 4) == 0 && ((uintptr_t)offsets % 4) == 0 && ((uintptr_t)c % 2) == 0,
               "aqtx_ragged_prepare: buffers are not element aligned");
  int64_t blocks = (m * (row_bytes / 2) + 256 * 64 - 1) / (256 * 64);
  blocks = blocks < 1 ? 1 : blocks > 1024 ? 1024 : blocks;
  const auto kernel = groups <= 128 ? ragged_prepare_kernel<false> : ragged_prepare_kernel<true>;
  kernel<<<dim3((unsigned)blocks), 256, 0, reinterpret_cast<hipStream_t>(stream)>>>(sizes, groups, m, offsets,
                                                                                    reinterpret_cast<uint16_t*>(c), row_bytes / 2);
  AQTX_HIP_CHECK_LAUNCH("ragged_prepare_kernel");
  return 0;
}
