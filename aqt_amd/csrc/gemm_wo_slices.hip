// aqtx_gemm_weight_only with k in slices, for a long k over few output tiles: 128 x 256 tiles of float32 partial sums, one
// slab a slice, and a launch that adds the slabs in slice order and dequantizes.  Without slices those shapes run on 64 x 64
// tiles, whose workgroups read each operand many times over and walk all of k: 256 x 4096 x 14336 in 94 us.
//
// The weight goes straight from memory into the operand registers.  A wave owns 64 columns of the tile for all 128 rows, so
// no other wave needs its part of the weight: it loads those int8 values (three stages ahead) and widens them
// between the matrix instructions, and LDS holds the bf16 rows of A alone, which arrive by direct loads.  (A weight widened
// on its way to LDS costs two LDS writes per 16 bytes and fragment reads of both operands by every wave; all of k
// on this tile without slices, the two are level: 500 x 14336 x 4096 in 75 us, from fragment order 68 and 72.)
// Bound by neither the matrix cores (a stage of 64 k has 1024 cycles of them and takes about 2000) nor memory: one wave a SIMD
// issues 130 vector instructions a stage next to them.  With slices / without, us, weights from HBM:
//   k = 14336: 65 x 4096 columns 36.5 / 90.5, 256 x 4096 51 / 94, 512 x 4096 80 / 109, 512 x 1024 37 / 74, 256 x 8192 82 / 111
//   k = 8192: 65 x 1024 24.4 / 40.0, 512 x 2048 37 / 44, 512 x 4096 53 / 61;  k = 6144: 256 x 4096 33.9 / 36.0
#include "gemm_core.h"

namespace aqtx {
namespace {

typedef int v2i __attribute__((ext_vector_type(2)));

constexpr int WTM = 128, WTN = 256, WBK = 64;       // rows, columns, k of a stage
constexpr int kWRow = WBK * 2, kWTile = WTM * kWRow;  // A in LDS: 128 bytes a row, 16 KiB a stage
constexpr int kWBuffers = 4, kWAhead = 3;

// A 16-byte load leaves lane (r, 0) with k 0..15 of weight row r and lane (r, 1) with k 16..31, and a matrix instruction
// wants k 0..7 | 8..15 of the two (then 16..23 | 24..31): two exchanges between the halves of the wave.
__device__ __forceinline__ void split_halves(const v4i x, v2i& first, v2i& second) {
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const auto s = __builtin_amdgcn_permlane32_swap((uint32_t)x[d], (uint32_t)x[d + 2], false, false);
    first[d] = (int)s[0];
    second[d] = (int)s[1];
  }
}
// 8 int8 values (k order) -> 8 bf16 values: the upper half of a value's float32 form is the result, exactly.
__device__ __forceinline__ v4i widen8(const v2i x) {
  v4i w;
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const uint32_t f0 = __float_as_uint((float)(int8_t)x[d]), f1 = __float_as_uint((float)(int8_t)(x[d] >> 8));
    const uint32_t f2 = __float_as_uint((float)(int8_t)(x[d] >> 16)), f3 = __float_as_uint((float)(x[d] >> 24));
    w[2 * d] = (int)__builtin_amdgcn_perm(f1, f0, 0x07060302u);
    w[2 * d + 1] = (int)__builtin_amdgcn_perm(f3, f2, 0x07060302u);
  }
  return w;
}

// Workgroup z of the grid contracts k in [z * k_chunk, (z + 1) * k_chunk) and leaves float32 sums in slab z.
template <bool FRAG>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2)))
void gemm_wo_slices_kernel(const GemmArgs g_in) {
  GemmArgs g = g_in;
  // objects of their own, so that the compiler can tell a fragment read of one from a request in flight into another
  __shared__ __attribute__((aligned(1024))) uint8_t ring0[kWTile], ring1[kWTile], ring2[kWTile], ring3[kWTile];
  auto ring = [&](const int b) -> uint8_t* { return b == 0 ? ring0 : b == 1 ? ring1 : b == 2 ? ring2 : ring3; };
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, lh = lane >> 5;
  int tm, tn;
  tile_of_block(blockIdx.x, g.tiles_m, g.tiles_n, tm, tn);
  const int64_t bz = blockIdx.y;
  const int64_t m0 = (int64_t)tm * WTM, n0 = (int64_t)tn * WTN;
  const int64_t kb = (int64_t)blockIdx.z * g.k_chunk;  // a multiple of 64
  g.a += kb * 2;
  g.b += FRAG ? kb * 16 : kb;  // 64 bytes of a row = one KiB step
  g.k = (g.k - kb) < g.k_chunk ? (g.k - kb) : g.k_chunk;
  const int64_t rows_a = (g.m - m0) < WTM ? (g.m - m0) : WTM;
  const int64_t rows_b = (g.n - n0) < WTN ? (g.n - n0) : WTN;
  const int k = (int)g.k;
  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(g.a + bz * g.stride_a + m0 * g.lda), 0, (int)((rows_a - 1) * g.lda + 2 * g.k), kBufferRsrcWord3);
  const __amdgpu_buffer_rsrc_t rsrc_b = FRAG
      ? __builtin_amdgcn_make_buffer_rsrc((void*)(g.b + (n0 / 16) * (int64_t)g.b_steps * 1024), 0,
                                          (int)((rows_b + 15) / 16 * g.b_steps * 1024), kBufferRsrcWord3)
      : __builtin_amdgcn_make_buffer_rsrc((void*)(g.b + bz * g.stride_b + n0 * g.ldb), 0,
                                          (int)((rows_b - 1) * g.ldb + g.k), kBufferRsrcWord3);
  constexpr int kOutside = 0x7FFFFFF0;  // reads as zero

  // A: a request covers 8 rows x 128 B, four a wave; lane l asks for the chunk that belongs at position l & 7 of row l >> 3
  // (position p of row r holds chunk p ^ f(r)).  B: load (nb, h) is 16 k of each row of 32-column block nb.  The row and
  // chunk of a load are in its vector offset, which the buffer's range check covers; the scalar offset (the stage's k) is
  // not range checked, the mask on k covers it.
  int avo[4], akp[4], bvo[2][2], bkp[2];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = wave * 32 + j * 8 + (lane >> 3), r = row & 31;
    const int c = (lane & 7) ^ ((r ^ (r >> 3)) & 7);
    akp[j] = c * 8;
    avo[j] = row * (int)g.lda + c * 16;
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int q = 2 * h + lh;
    bkp[h] = 16 * q;
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      const int row = wave * 64 + nb * 32 + lr;
      bvo[nb][h] = FRAG ? (row >> 4) * g.b_steps * 1024 + (q * 16 + (row & 15)) * 16 : row * (int)g.ldb + q * 16;
    }
  }
  v4i raw[kWBuffers][2][2];
  auto request_a = [&](uint8_t* buf, const int j, const int k0) {
    const int vo = k0 + akp[j] < k ? avo[j] : kOutside;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, AQTX_LDS_PTR(buf + (wave * 32 + j * 8) * kWRow), 16, vo, k0 * 2, 0, 0);
  };
  auto request_b = [&](const int set, const int nb, const int h, const int k0) {
    const int vo = k0 + bkp[h] < k ? bvo[nb][h] : kOutside;
    raw[set][nb][h] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_b, vo, FRAG ? k0 * 16 : k0, 0);
  };
  constexpr int kRequests = 8;  // of a wave and stage

  int fo[4];  // fragment of k step ks of a 32-row block: chunk 2 ks + lh of row lr
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) fo[ks] = lr * kWRow + (((2 * ks + lh) ^ ((lr ^ (lr >> 3)) & 7)) << 4);

  v16f acc[4][2];
#pragma unroll
  for (int im = 0; im < 4; ++im)
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[im][nb][r] = 0.0f;

  const int nstages = (k + WBK - 1) / WBK;
#pragma unroll
  for (int d = 0; d < kWAhead; ++d) {
#pragma unroll
    for (int j = 0; j < 4; ++j) request_a(ring(d), j, d * WBK);
#pragma unroll
    for (int i = 0; i < 4; ++i) request_b(d, i >> 1, i & 1, d * WBK);
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kWAhead - 1) * kRequests) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  // Stage s computes from buffer and register set s % 4 and requests stage s + 3 (past the end of k: zeros nobody uses)
  // into those that stage s - 1 left at its barrier.  Requests complete in order: before its barrier a wave waits until all
  // but those of stages s + 2 and s + 3 have landed, and behind the barrier everybody's have.
  auto stage = [&](const int s, auto set_c) {
    constexpr int SET = decltype(set_c)::value, NEXT = (SET + kWAhead) % kWBuffers;
    const uint8_t* st = ring(SET);
    const int k_next = (s + kWAhead) * WBK;
    // (not a use of these registers moves above the barrier, where it would wait for the requests in flight behind them)
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(raw[SET][i >> 1][i & 1]));
    v2i half[2][2][2];  // [column block][of its two loads][first, second]
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      v4i fa[4], fb[2];
#pragma unroll
      for (int im = 0; im < 4; ++im) fa[im] = *reinterpret_cast<const v4i*>(st + im * 32 * kWRow + fo[ks]);
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        if ((ks & 1) == 0) split_halves(raw[SET][nb][ks >> 1], half[nb][ks >> 1][0], half[nb][ks >> 1][1]);
        fb[nb] = widen8(half[nb][ks >> 1][ks & 1]);
      }
      request_a(ring(NEXT), ks, k_next);
      request_b(NEXT, ks >> 1, ks & 1, k_next);
#pragma unroll
      for (int im = 0; im < 4; ++im)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) acc[im][nb] = MmaBf16W8::mma(fb[nb], fa[im], acc[im][nb]);
    }
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((kWAhead - 1) * kRequests) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  int s = 0;
  for (; s + 4 <= nstages; s += 4) {
    stage(s, std::integral_constant<int, 0>{});
    stage(s + 1, std::integral_constant<int, 1>{});
    stage(s + 2, std::integral_constant<int, 2>{});
    stage(s + 3, std::integral_constant<int, 3>{});
  }
  if (s < nstages) stage(s, std::integral_constant<int, 0>{});
  if (s + 1 < nstages) stage(s + 1, std::integral_constant<int, 1>{});
  if (s + 2 < nstages) stage(s + 2, std::integral_constant<int, 2>{});
  // the requests past the end of k write zeros to the buffers: they have to land before the epilogue's use of them
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  // ---- lane holds C[m = im*32 + lr][n = wave*64 + nb*32 + 8q + 4lh + e], register 4q + e of block (im, nb); a wave passes
  // 32 rows at a time through a buffer of its own, so that the stores are 16 bytes a lane along rows
  constexpr int kRowBytes = 64 * 4, kPitch = kRowBytes + 16, kLanesPerRow = kRowBytes / 16, kRowsPerPass = 64 / kLanesPerRow;
  static_assert(32 * kPitch <= kWTile, "32 rows of a wave fit its buffer");
  uint8_t* mine = ring(wave);
  float* slab = reinterpret_cast<float*>(g.slabs) + ((int64_t)blockIdx.z * gridDim.y + bz) * g.m * g.n;
  const bool vec = g.n % 4 == 0;
#pragma unroll
  for (int im = 0; im < 4; ++im) {
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const v16f& v = acc[im][nb];
        *reinterpret_cast<float4*>(mine + lr * kPitch + (nb * 32 + 8 * q + 4 * lh) * 4) =
            make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
      }
    const int pr = lane / kLanesPerRow, pc = lane % kLanesPerRow;
#pragma unroll
    for (int it = 0; it < 32 / kRowsPerPass; ++it) {
      const int r = it * kRowsPerPass + pr;
      const float4 val = *reinterpret_cast<const float4*>(mine + r * kPitch + pc * 16);
      const int64_t mm = m0 + im * 32 + r, nn = n0 + wave * 64 + pc * 4;
      if (mm >= g.m || nn >= g.n) continue;
      float* dst = slab + mm * g.n + nn;
      if (vec) {
        *reinterpret_cast<float4*>(dst) = val;
      } else {
        const float o[4] = {val.x, val.y, val.z, val.w};
        for (int e = 0; e < 4 && nn + e < g.n; ++e) dst[e] = o[e];
      }
    }
  }
}

// Adds the slabs in slice order and dequantizes: eight columns a thread.
template <int EPI>
__global__ __launch_bounds__(256) void sum_slabs_wo_kernel(const GemmArgs g) {
  const int64_t mm = blockIdx.y, bz = blockIdx.z, n8 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
  if (n8 >= g.n) return;
  const int nv = g.n - n8 < 8 ? (int)(g.n - n8) : 8;
  const int64_t slab = (int64_t)gridDim.z * g.m * g.n, at = (bz * g.m + mm) * g.n + n8;
  const float* slabs = reinterpret_cast<const float*>(g.slabs);
  const bool vec = nv == 8 && g.n % 4 == 0;
  float v[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  for (int z = 0; z < g.k_split; ++z) {
    const float* src = slabs + z * slab + at;
    if (vec) {
      const float4 a = *reinterpret_cast<const float4*>(src), b = *reinterpret_cast<const float4*>(src + 4);
      v[0] += a.x; v[1] += a.y; v[2] += a.z; v[3] += a.w;
      v[4] += b.x; v[5] += b.y; v[6] += b.z; v[7] += b.w;
    } else {
      for (int e = 0; e < nv; ++e) v[e] += src[e];
    }
  }
  const float* cs = g.col_scale != nullptr ? g.col_scale + bz * g.stride_cs + n8 : nullptr;
  uint16_t* dst = reinterpret_cast<uint16_t*>(g.c) + bz * g.stride_c + mm * g.ldc + n8;
  for (int e = 0; e < nv; ++e) dst[e] = bf16_bits(dequant_value<EPI, false>(v[e], 1.0f, cs != nullptr ? cs[e] : 1.0f));
}

}  // namespace

// Slices of k for a plan, 1 = none: workgroups for the chip's 256 CUs, at most 16 slices.  Fewer than four are level with the
// kernels that walk all of k (512 x 8192 x 14336 142 us and 139), and so are four at k = 6144 (512 x 4096 47 and 47); a
// shorter k is not cut.
int gemm_weight_only_k_slices(const aqtx_gemm_plan* p) {
  if (p->tuning != 0 || p->k_split != 0 || p->k < 6144) return 1;
  const int64_t tiles = ((p->m + WTM - 1) / WTM) * ((p->n + WTN - 1) / WTN) * p->batch;
  const int64_t s = 256 / tiles;
  return s < 4 ? 1 : s > 16 ? 16 : (int)s;
}

int launch_gemm_weight_only_slices(const aqtx_gemm_plan* p, const void* a, const void* b, const float* col_scale, void* c,
                                   int slices, hipStream_t st) {
  GemmArgs g = make_gemm_args(p, a, b, nullptr, col_scale, c, nullptr);
  g.lda *= 2; g.stride_a *= 2;  // A in bytes (k stays a count)
  g.b_steps = (int)((p->k + 63) / 64);
  g.tiles_m = (int)((p->m + WTM - 1) / WTM);
  g.tiles_n = (int)((p->n + WTN - 1) / WTN);
  g.k_chunk = ((p->k + slices - 1) / slices + WBK - 1) / WBK * WBK;
  g.k_split = (int)((p->k + g.k_chunk - 1) / g.k_chunk);
  g.slabs = reinterpret_cast<int32_t*>(p->k_split_workspace);
  const dim3 grid((unsigned)(g.tiles_m * g.tiles_n), (unsigned)p->batch, (unsigned)g.k_split);
  if (p->b_layout == AQTX_W_FRAGMENTS) gemm_wo_slices_kernel<true><<<grid, 256, 0, st>>>(g);
  else gemm_wo_slices_kernel<false><<<grid, 256, 0, st>>>(g);
  const dim3 sgrid((unsigned)((p->n + 2047) / 2048), (unsigned)p->m, (unsigned)p->batch);
  // epilogue 4: first product bf16 (no row scale), second f32
  if (p->col_scale_dtype != AQTX_BF16) sum_slabs_wo_kernel<4><<<sgrid, 256, 0, st>>>(g);
  else sum_slabs_wo_kernel<0><<<sgrid, 256, 0, st>>>(g);
  AQTX_HIP_CHECK_LAUNCH("gemm_wo_slices_kernel");
  return 0;
}

}  // namespace aqtx
