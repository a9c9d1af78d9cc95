// Abs-max calibration + quantization kernels (gfx950), compiled once per input type
// (quantize_f32.hip, quantize_bf16.hip, quantize_i8.hip); the C entry points are in quantize.hip.
//
// One operand of the quantized dot_general goes through
//   scale = absmax / quant_bound            (calibration.py:117-157)
//   t     = x * (1 / scale)                 (aqt_tensor.py:125-159)
//   t     = t + noise; clip; round; cast    (int_numerics.py:81-111,
//                                            fp8_numerics.py:36-123)
// with every intermediate rounded to the dtype the reference holds it in.  Two
// launch shapes cover the layouts:
//   * "rows": the reduced axis is the contiguous one.  A segment (one row, or one
//     subchannel group of a row) is loaded once into registers by 16, 64 or 256
//     lanes, reduced with wavefront shuffles (+LDS across the four waves),
//     quantized from registers and stored: one HBM read, one write.
//   * "tile": the reduced axis is the strided one (or the whole tensor).  A
//     column abs-max pass (atomic max on the float bit pattern) is followed by a
//     128x64 tile pass that quantizes and, on request, writes the transposed
//     layout through LDS so that the consumer GEMM finds its contraction axis
//     contiguous.
#pragma once
#include "common.h"
#include <type_traits>

#include "threefry.h"

namespace aqtx {

struct QArgs {
  const void* x;
  const float* prescale;
  void* q;
  float* scale;
  uint16_t* scale_bf16;  // optional second copy of the computed scales as bf16 elements
  uint32_t* ws_absmax;
  float* ws_inv;
  // Arrival counts of the abs-max blocks, zero on entry and exit, one per group of blocks that share scales: the last
  // block of a group turns its maxima into scales.  NULL: finalize_scales_kernel does, in a launch of its own.
  uint32_t* ws_arrived;
  int64_t batch, rows, cols;
  int64_t L;        // rows kernel: segment length
  int64_t nseg;     // rows kernel: number of segments
  int64_t G;        // tile kernels: group length along rows
  int64_t ngroups;  // tile kernels: rows / G
  int64_t ssb, ssg, ssc;  // tile kernels: scale index strides
  int64_t nsb, nsr, nsc;  // noise counter strides
  int64_t psb;            // prescale batch stride
  float quant_bound, clip_bound;
  BitGen gen;
  const uint32_t* key_dev;  // optional: the two key words in device memory (replace gen.k0 / gen.k1)
  int noise;
  int ps_mode;
  int transpose_out;
  int out_dtype;
  int cbf;  // compute dtype is bf16
  int sbf;  // scale dtype is bf16
  int scale_given;
  const uint16_t* given_bf16;  // given scales as bf16 elements, read where they lie (NULL: in `scale`)
  int ws_zeroed;  // the abs-max words of the workspace are zero on entry
  int scale_only; // the scales are all that is asked for (a calibration on its own): nothing reads or writes q
  int once_shift; // columns: calibrated and quantized in one pass, with so many threads a row (as a shift); -1: not
  int even_odd8;  // rows kernel: bytes of each group of 8 outputs stored as elements 0,2,4,6,1,3,5,7
  // Partial maxima of |q| along the axis that carries the scales, one byte per position of the reduced axis and
  // part (aqtx_quant_plan::other_axis_absmax): written by a launch (oa_out), or read in place of an abs-max pass
  // over this input (oa_in).
  uint8_t* oa_out;
  const uint8_t* oa_in;
  int64_t oa_in_parts;
};

// Blocks of the row kernel that also writes column maxima, each walking rows: seven per CU of the largest part, as
// many as its registers (67 with 16 running maxima) let a CU hold (measured on 8192 rows of 4096 bf16 values, 21 us
// without the maxima: 62 us with 256 blocks, 40 with 512, 30 with 1024).
constexpr int64_t kColmaxBlocks = 7 * 256;

constexpr int kTileR = 128, kTileC = 64;

// Column abs-max: a block takes 64 lanes x 8 columns (1 where there are fewer than 8) and 64 rows of them.
constexpr int kAbsRowChunk = 64, kAbsColLanes = 64;
inline int64_t absmax_col_groups(int64_t cols) {
  const int64_t width = kAbsColLanes * (cols >= 8 ? 8 : 1);
  return (cols + width - 1) / width;
}

// Columns in one pass (quant_cols_once_kernel): rows a thread, by the bytes of a value (64 registers of values), and threads
// a row (as a shift), 2 to 16.
template <int ESZ> constexpr int kOnceRows = ESZ == 2 ? 16 : 8;
constexpr int kOnceMaxShift = 4;
// The shift, or -1 where calibration and quantization stay launches of their own: columns beyond a block's registers, and
// row maxima, whose parts are 64 columns, beyond those of 8 threads a row.  Few threads a row while that gives the chip two
// blocks a CU, but a wave a block: 4096 x 4096 bf16 14.5 us with 2 and 17.6 with 4, 8 entries of 4096 x 14336 444 and 421,
// 128 x 16384 with 2 8, with 4 5.3.  Calibration and quantization in launches of their own / in one, us:
//   bf16     16 x 2048 9.8 / 5.6, 512 x 512 8.2 / 5.1, 1030 x 3001 11.2 / 7.0, 2048 x 64 8.6 / 6.1, 2048 x 16384 36.1 / 23.2,
//            4096 x 1024 10.7 / 9.3, 4096 x 4096 21.8 / 14.5, 4096 x 14336 52 / 41, 8 entries of it 477 / 421
//   float32  128 x 512 8.5 / 3.9, 512 x 2048 9.0 / 4.4, 1024 x 8192 19.0 / 9.4, 2048 x 2048 11.7 / 7.0, 2048 x 8192 28.1 / 19.5
inline int cols_once_shift(int esz, int64_t batch, int64_t rows, int64_t cols, bool row_maxima) {
  const int R = esz == 2 ? 16 : 8;
  const int64_t groups = (rows + R - 1) / R;
  if (rows < R || cols < 8 || groups > 256) return -1;
  if (row_maxima) return groups <= 128 ? 3 : -1;
  int shift = 1;
  while (shift < kOnceMaxShift && (groups << shift) < 64) ++shift;
  while (shift < kOnceMaxShift && (groups << (shift + 1)) <= 1024 && batch * (cols >> (shift + 4)) >= 512) ++shift;
  return shift;
}

// Launches the passes of one plan for one input type.
int launch_quantize_f32(const QArgs& a, int reduce, int partitionable, int64_t nscales, hipStream_t st);
int launch_quantize_bf16(const QArgs& a, int reduce, int partitionable, int64_t nscales, hipStream_t st);
int launch_quantize_i8(const QArgs& a, int reduce, int partitionable, int64_t nscales, hipStream_t st);

namespace {

// Kernel-side copy of the arguments with the PRNG key taken from device memory when the caller
// passed it there (a traced key under XLA, a key updated on the device between graph replays).
__device__ __forceinline__ QArgs with_device_key(const QArgs& in) {
  QArgs a = in;
  if (in.key_dev != nullptr) {
    a.gen.k0 = in.key_dev[0];
    a.gen.k1 = in.key_dev[1];
  }
  return a;
}

// The computed scale goes out as float32 and, when the caller keeps its scales in bf16, once
// more as bf16 elements (the value is already rounded to bf16, so the narrowing is exact).
__device__ __forceinline__ void store_scale(const QArgs& a, int64_t i, float v) {
  a.scale[i] = v;
  if (a.scale_bf16 != nullptr) a.scale_bf16[i] = (uint16_t)(__float_as_uint(v) >> 16);
}

// A scale the caller gives.
__device__ __forceinline__ float given_scale(const QArgs& a, int64_t i) {
  return a.given_bf16 != nullptr ? __uint_as_float((uint32_t)a.given_bf16[i] << 16) : a.scale[i];
}

// ---- typed vector loads ------------------------------------------------------
// Eight values at any element boundary: one vector load each (two for float32) whatever the alignment, so rows of
// any length take the same path.
template <typename V> __device__ __forceinline__ V load_unaligned(const void* p) {
  V v;
  __builtin_memcpy(&v, p, sizeof(V));
  return v;
}
__device__ __forceinline__ void store8(uint8_t* p, uint2 v) { __builtin_memcpy(p, &v, 8); }
template <typename T> struct Loader;
template <> struct Loader<float> {
  static __device__ __forceinline__ void load8(const float* p, float* v) {
    const float4 a = load_unaligned<float4>(p);
    const float4 b = load_unaligned<float4>(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  }
  static __device__ __forceinline__ float load1(const float* p) { return *p; }
};
template <> struct Loader<uint16_t> {  // bf16 bit patterns
  static __device__ __forceinline__ void load8(const uint16_t* p, float* v) {
    const uint4 a = load_unaligned<uint4>(p);
    v[0] = __uint_as_float(a.x << 16); v[1] = __uint_as_float(a.x & 0xFFFF0000u);
    v[2] = __uint_as_float(a.y << 16); v[3] = __uint_as_float(a.y & 0xFFFF0000u);
    v[4] = __uint_as_float(a.z << 16); v[5] = __uint_as_float(a.z & 0xFFFF0000u);
    v[6] = __uint_as_float(a.w << 16); v[7] = __uint_as_float(a.w & 0xFFFF0000u);
  }
  static __device__ __forceinline__ float load1(const uint16_t* p) {
    return __uint_as_float(((uint32_t)*p) << 16);
  }
};
template <> struct Loader<int8_t> {
  static __device__ __forceinline__ void load8(const int8_t* p, float* v) {
    const uint2 a = load_unaligned<uint2>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] = (float)(int8_t)((a.x >> (8 * i)) & 0xFF);
      v[4 + i] = (float)(int8_t)((a.y >> (8 * i)) & 0xFF);
    }
  }
  static __device__ __forceinline__ float load1(const int8_t* p) { return (float)*p; }
};

__device__ __forceinline__ float rnd(float x, int bf) { return bf ? round_bf16(x) : x; }

// scale and reciprocal scale from the abs-max (calibration.py:145-157,
// aqt_tensor.py:151-155).
__device__ __forceinline__ void scale_from_absmax(float amax, const QArgs& a, float& scale,
                                                  float& inv) {
  if (amax == 0.0f) amax = 1.0f;
  float s = rnd(amax / a.quant_bound, a.cbf);
  s = rnd(s, a.sbf);
  float i = rnd(1.0f / s, a.sbf);
  if (isinf(i)) i = 1.0f;
  scale = s;
  inv = i;
}

__device__ __forceinline__ float inv_of_scale(float scale, const QArgs& a) {
  float i = rnd(1.0f / scale, a.sbf);
  if (isinf(i)) i = 1.0f;
  return i;
}

__device__ __forceinline__ float apply_prescale(float v, float ps, const QArgs& a) {
  // aqt_dot_general.py:714-720: lhs * scale_t.astype(lhs.dtype)
  return rnd(v * rnd(ps, a.cbf), a.cbf);
}

// The value after scaling, noise and clipping, still a float.
__device__ __forceinline__ float scaled_noisy_clipped(float v, float inv, uint64_t ctr,
                                                      const QArgs& a) {
  const int tbf = a.cbf & a.sbf;  // promote(x.dtype, scale.dtype)
  float t = rnd(v * inv, tbf);
  if (a.noise == AQTX_NOISE_JAX_UNIFORM) {
    const uint32_t bits = a.gen.draw(ctr);
    float u = __uint_as_float((bits >> 9) | 0x3F800000u) - 1.0f;
    u = fmaxf(0.0f, u);
    t = rnd(t + (u - 0.5f), tbf);
  } else if (a.noise == AQTX_NOISE_CUSTOM1) {
    const uint32_t bits = a.gen.draw(ctr);
    const float f = __uint_as_float((bits << 7) | 0x3F800000u);
    t = rnd(t + (f - 1.49999237060546875f), tbf);  // 1.5 - 2^-17
  } else if (a.noise == AQTX_NOISE_FP8_MANTISSA) {
    const int mant = (a.out_dtype == AQTX_E4M3) ? 3 : 2;
    const uint32_t bits = a.gen.draw(ctr);
    if (tbf) {
      const uint32_t mask = (1u << (7 - mant)) - 1u;
      uint32_t u = __float_as_uint(t) >> 16;
      u = ((u + (bits & mask)) & ~mask) & 0xFFFFu;
      t = __uint_as_float(u << 16);
    } else {
      const uint32_t mask = (1u << (23 - mant)) - 1u;
      uint32_t u = __float_as_uint(t);
      u = (u + (bits & mask)) & ~mask;
      t = __uint_as_float(u);
    }
  }
  t = fminf(fmaxf(t, -a.clip_bound), a.clip_bound);
  return t;
}

// float (already clipped) -> output byte
__device__ __forceinline__ uint32_t to_qbyte(float t, int out_dtype) {
  if (out_dtype == AQTX_E4M3) {
    return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(t, t, 0, false) & 0xFFu;
  } else if (out_dtype == AQTX_E5M2) {
    return (uint32_t)__builtin_amdgcn_cvt_pk_bf8_f32(t, t, 0, false) & 0xFFu;
  }
  return (uint32_t)((int)rintf(t)) & 0xFFu;
}

// ---- compile-time specialisations of the element pipeline ------------------------------
// SPEC 0: every flag is read from QArgs at run time (any dtype / numerics).
// SPEC 1: bf16 values, bf16 scale, integer out (int8, or int4 in an int8 byte), round to nearest
//         even (the forward operands).
// SPEC 3: bf16 values, bf16 scale, fp8 out (e4m3fn or e5m2), no noise.
// SPEC 5: SPEC 3 + fp8 mantissa stochastic rounding, 16-bit draws of the original layout.
// SPEC 2: SPEC 1 + jax.random.uniform noise in the original threefry counter layout (the
//         gradient-side operands).  With PAIR the two elements that share one threefry block
//         (indices i and i + total/2) are produced by the same thread from a single block.
// SPEC 6, 7: SPEC 1 and SPEC 2 with float32 values and scales (no intermediate is rounded).  On SPEC 0 a float32
//         layer was bound by the run-time flags and the 64-bit noise counters: 8.4 million gradients with noise took
//         131 us (tiles; 18 on SPEC 7) and 32 us (rows; 19), 8.4 million activations without it 23 us (11 on SPEC 6),
//         and the step of a 4096 x 512 -> 2048 -> 512 block 852 us (374).
constexpr bool spec_is_f32(int spec) { return spec == 6 || spec == 7; }
constexpr bool spec_has_uniform_noise(int spec) { return spec == 2 || spec == 7; }
template <int SPEC>
__device__ __forceinline__ float spec_scale(float v, float inv, const QArgs& a) {
  if constexpr (SPEC == 0) return rnd(v * inv, a.cbf & a.sbf);
  if constexpr (spec_is_f32(SPEC)) return v * inv;
  return round_bf16(v * inv);
}
__device__ __forceinline__ float uniform_noise(uint32_t bits) {
  // jax.random.uniform: f = bitcast(bits >> 9 | 0x3F800000) in [1, 2), u = f - 1, max(0, u); then
  // the centring of JaxUniform, u - 0.5.  f - 1 and u - 0.5 are exact (multiples of 2^-23 below 1)
  // and u >= 0, so the three steps equal the single exact subtraction f - 1.5.  The shift-and-or
  // is one funnel shift of {0x7F, bits} by 9.
  const uint32_t f = __builtin_amdgcn_alignbit(0x7Fu, bits, 9);
  return __uint_as_float(f) - 1.5f;
}
// Rounds two floats to bf16 (ties to even) in place: the packed conversion of (0, x) leaves bf16(x) in the upper half of the
// word over zeros, rounded and widened in one instruction (both in one conversion take three). The time of the noise kernels is
// their vector instructions: with the byte permutes of pack4, 186 -> 176 us (rows) and 193 -> 189 (columns) at bf16 8192 x 14336.
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void round_bf16_pair(float& a, float& b) {
  a = __builtin_bit_cast(float, __builtin_convertvector(f32x2_t{0.0f, a}, bf16x2_t));
  b = __builtin_bit_cast(float, __builtin_convertvector(f32x2_t{0.0f, b}, bf16x2_t));
}
template <int SPEC>
__device__ __forceinline__ uint32_t spec_finish(float t, const QArgs& a) {
  // clip, round half to even, cast (int_numerics.py:99-110; fp8_numerics.py:112-123)
  if constexpr (SPEC == 0 || SPEC == 3 || SPEC == 5) {
    t = fminf(fmaxf(t, -a.clip_bound), a.clip_bound);
    return to_qbyte(t, a.out_dtype);
  }
  // clip in one median-of-three; round half to even and convert in one addition: after
  // t + 1.5 * 2^23 the low mantissa bits are the two's complement of the rounded integer
  // (|t| <= 127 here)
  t = __builtin_amdgcn_fmed3f(t, -a.clip_bound, a.clip_bound);
  return __float_as_uint(t + 12582912.0f) & 0xFFu;
}
// fp_mantissa_round on a bf16 value (fp8_numerics.py:36-64): add the masked random bits to the
// bit pattern, clear the low mantissa bits.  The sum stays in the upper half, where the value is: fewer instructions
// than by shifts down and up, with the rounding before it (fp8 with noise, tile kernel, bf16 8192 x 14336 by one scale:
// 179 -> 168 us with its abs-max).
__device__ __forceinline__ float bf16_mantissa_sr(float t, uint32_t bits, uint32_t mask) {
  const uint32_t hi = mask << 16;
  return __uint_as_float((__float_as_uint(t) + ((bits << 16) & hi)) & ~hi);
}
// scale -> (noise) -> clip/round/cast for one element
template <int SPEC>
__device__ __forceinline__ uint32_t spec_quant(float v, float inv, uint64_t ctr, const QArgs& a) {
  if constexpr (SPEC == 0) {
    return to_qbyte(scaled_noisy_clipped(v, inv, ctr, a), a.out_dtype);
  } else {
    float t = spec_scale<SPEC>(v, inv, a);
    if constexpr (SPEC == 2) t = round_bf16(t + uniform_noise(a.gen.word_original((uint32_t)ctr)));
    if constexpr (SPEC == 7) t = t + uniform_noise(a.gen.word_original((uint32_t)ctr));
    if constexpr (SPEC == 5) {
      const uint32_t w = a.gen.word_original((uint32_t)(ctr >> 1));
      t = bf16_mantissa_sr(t, (ctr & 1) ? (w >> 16) : w, a.out_dtype == AQTX_E4M3 ? 0xFu : 0x1Fu);
    }
    return spec_finish<SPEC>(t, a);
  }
}
// The same for the noiseless integer pipelines (SPEC 0 with integer out, SPEC 1, SPEC 6), which also hands out the clipped
// value before rounding: |q| = rint(|t|) and rint is monotonic, so a maximum of |q| can be kept as a maximum of
// |t| (one instruction per element) and rounded once at the end.
template <int SPEC>
__device__ __forceinline__ uint32_t spec_quant_mag(float v, float inv, uint64_t ctr, const QArgs& a, float& t_clipped) {
  static_assert(SPEC == 0 || SPEC == 1 || SPEC == 6, "noiseless integer pipelines");
  if constexpr (SPEC == 0) {
    t_clipped = scaled_noisy_clipped(v, inv, ctr, a);
    return to_qbyte(t_clipped, a.out_dtype);
  } else {
    t_clipped = __builtin_amdgcn_fmed3f(spec_scale<SPEC>(v, inv, a), -a.clip_bound, a.clip_bound);
    return __float_as_uint(t_clipped + 12582912.0f) & 0xFFu;
  }
}
// the pair (i, i + half) from one threefry block (SPEC 2 and 7, original layout, i < half)
template <int SPEC>
__device__ __forceinline__ void pair_quant(float v0, float inv0, float v1, float inv1, uint32_t i,
                                           const QArgs& a, uint32_t& q0, uint32_t& q1) {
  const U2 bits = threefry2x32(a.gen.k0, a.gen.k1, i, i + a.gen.half);
  static_assert(spec_has_uniform_noise(SPEC), "pipelines with one 32-bit draw per element");
  float t0 = v0 * inv0, t1 = v1 * inv1;
  if constexpr (SPEC == 2) round_bf16_pair(t0, t1);
  t0 += uniform_noise(bits.x);
  t1 += uniform_noise(bits.y);
  if constexpr (SPEC == 2) round_bf16_pair(t0, t1);
  q0 = spec_finish<SPEC>(t0, a);
  q1 = spec_finish<SPEC>(t1, a);
}
template <int SPEC>
__device__ __forceinline__ float spec_prescale(float v, float ps, const QArgs& a) {
  if constexpr (SPEC == 0) return apply_prescale(v, ps, a);
  if constexpr (spec_is_f32(SPEC)) return v * ps;
  return round_bf16(v * round_bf16(ps));
}
template <int SPEC>
__device__ __forceinline__ void spec_scale_from_absmax(float amax, const QArgs& a, float& scale, float& inv) {
  if constexpr (SPEC == 0) {
    scale_from_absmax(amax, a, scale, inv);
  } else {
    constexpr bool bf = !spec_is_f32(SPEC);
    if (amax == 0.0f) amax = 1.0f;
    scale = round_to<bf>(amax / a.quant_bound);
    inv = round_to<bf>(1.0f / scale);
    if (isinf(inv)) inv = 1.0f;
  }
}

template <int LANES>
__device__ __forceinline__ float segment_max(float v, float* smem) {
  constexpr int W = LANES < 64 ? LANES : 64;
#pragma unroll
  for (int off = W / 2; off > 0; off >>= 1) v = nanmax(v, __shfl_xor(v, off, W));
  if constexpr (LANES >= 256) {  // the segment is the whole block
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) smem[wave] = v;
    __syncthreads();
    v = nanmax(nanmax(smem[0], smem[1]), nanmax(smem[2], smem[3]));
    if constexpr (LANES == 512) v = nanmax(v, nanmax(nanmax(smem[4], smem[5]), nanmax(smem[6], smem[7])));
  }
  return v;
}

// Eight row values kept in registers between the abs-max pass and the quantize pass.  bf16
// inputs of the specialised pipelines stay packed two per register (the prescaled value is
// rounded to bf16 as well), which halves the registers a row costs and doubles the waves per SIMD.
template <bool PACKED> struct RowVals;
template <> struct RowVals<false> {
  float f[8];
  __device__ __forceinline__ void put(const float* t) {
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = t[e];
  }
  __device__ __forceinline__ void get(float* t) const {
#pragma unroll
    for (int e = 0; e < 8; ++e) t[e] = f[e];
  }
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = 0.0f;
  }
};
template <> struct RowVals<true> {
  uint32_t w[4];
  __device__ __forceinline__ void put(const float* t) {  // t[e] are bf16-representable
#pragma unroll
    for (int i = 0; i < 4; ++i)
      w[i] = __builtin_amdgcn_perm(__float_as_uint(t[2 * i + 1]), __float_as_uint(t[2 * i]), 0x07060302u);
  }
  __device__ __forceinline__ void get(float* t) const {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      t[2 * i] = __uint_as_float(w[i] << 16);
      t[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
    }
  }
  __device__ __forceinline__ void zero() { w[0] = w[1] = w[2] = w[3] = 0u; }
};
typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));
// max of the two bf16 magnitudes of `w` against the running packed maxima: magnitudes of
// floats order like unsigned integers
__device__ __forceinline__ uint32_t packed_absmax(uint32_t m, uint32_t w) {
  const u16x2_t a = __builtin_bit_cast(u16x2_t, m), b = __builtin_bit_cast(u16x2_t, w & 0x7FFF7FFFu);
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(a, b));
}

// Eight output bytes -> two words, in element order or as elements 0,2,4,6 | 1,3,5,7.
// (Byte permutes of the low bytes, which need no masking first; a branch and no selects, which were a select a value.)
__device__ __forceinline__ uint32_t pack4(uint32_t q0, uint32_t q1, uint32_t q2, uint32_t q3) {
  return __builtin_amdgcn_perm(__builtin_amdgcn_perm(q3, q2, 0x0c0c0400u), __builtin_amdgcn_perm(q1, q0, 0x0c0c0400u), 0x05040100u);
}
__device__ __forceinline__ uint2 pack8(const uint32_t (&q)[8], int even_odd8) {
  if (even_odd8) {
    asm volatile("");
    return make_uint2(pack4(q[0], q[2], q[4], q[6]), pack4(q[1], q[3], q[5], q[7]));
  }
  return make_uint2(pack4(q[0], q[1], q[2], q[3]), pack4(q[4], q[5], q[6], q[7]));
}
// Transposes 4 x 4 bytes: words of rows -> words of columns (half an instruction a byte, where gathering a column's bytes
// next to the row's by shifts took one).
__device__ __forceinline__ void transpose4(const uint32_t (&r)[4], uint32_t (&c)[4]) {
  const uint32_t a = __builtin_amdgcn_perm(r[1], r[0], 0x05010400u), b = __builtin_amdgcn_perm(r[3], r[2], 0x05010400u);
  const uint32_t d = __builtin_amdgcn_perm(r[1], r[0], 0x07030602u), e = __builtin_amdgcn_perm(r[3], r[2], 0x07030602u);
  c[0] = __builtin_amdgcn_perm(b, a, 0x05040100u);
  c[1] = __builtin_amdgcn_perm(b, a, 0x07060302u);
  c[2] = __builtin_amdgcn_perm(e, d, 0x05040100u);
  c[3] = __builtin_amdgcn_perm(e, d, 0x07060302u);
}

// quant_cols_once_kernel: maxima of magnitudes (bf16: two to a word) and the eight values of a row's registers.
template <typename TIn> __device__ __forceinline__ uint32_t once_max(uint32_t x, uint32_t y) {
  if constexpr (sizeof(TIn) == 2)
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2_t, x), __builtin_bit_cast(u16x2_t, y)));
  return x > y ? x : y;
}
template <typename TIn, int W> __device__ __forceinline__ void once_unpack(const uint4 (&w)[W], float (&v)[8]) {
  if constexpr (sizeof(TIn) == 2) {
    const uint32_t x[4] = {w[0].x, w[0].y, w[0].z, w[0].w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = __uint_as_float(x[i] << 16);
      v[2 * i + 1] = __uint_as_float(x[i] & 0xFFFF0000u);
    }
  } else {
#pragma unroll
    for (int h = 0; h < W; ++h) {
      v[4 * h] = __uint_as_float(w[h].x); v[4 * h + 1] = __uint_as_float(w[h].y);
      v[4 * h + 2] = __uint_as_float(w[h].z); v[4 * h + 3] = __uint_as_float(w[h].w);
    }
  }
}

// ---- rows kernel: reduced axis contiguous -------------------------------------
// PAIR (SPEC 2 and 7): the block owns segment s and segment s + nseg/2, whose elements share
// threefry blocks; requires whole rows as segments and the natural noise layout.
// A block is 256 threads, or 512 (LANES = 512: one long segment per block, half the row values per
// thread, so that six waves fit a SIMD: the stochastic pipeline is bound by vector instruction
// issue: one in 2.1 ns from a lone wave, in 1.1 to 1.8 from several).
// The bound of four waves a SIMD goes to pipelines that fit 128 registers.  int8 values of the bf16 pipelines, held as
// floats, do not: two paired rows of eight pieces need 182, and spill 196 bytes a lane under the bound (300 rows of 9000
// with noise: 17.7 us, 12.8 without it; 2048 of 16384: 59 and 55).
// COLMAX (whole rows as segments, one per block, no PAIR): the grid is smaller than the number of rows, a block
// walks rows blockIdx.x, + gridDim.x, ... and keeps, per column it owns, the largest |q| it wrote; at the end it
// stores them as row blockIdx.x of QArgs::oa_out ([gridDim.x][cols] bytes): what a later pass that calibrates the
// quantized values over the rows needs instead of reading them again.
template <typename TIn, int LANES, int ITERS, int SPEC, bool PAIR, bool COLMAX = false>
__global__ __launch_bounds__(LANES == 512 ? 512 : 256,
                             (COLMAX && ITERS <= 2 && SPEC == 1) ? 7 : LANES == 512 ? 3
                             : !COLMAX && ((sizeof(TIn) == 2 && SPEC != 0) || spec_is_f32(SPEC)) ? 4 : 1)
void quant_rows_kernel(const QArgs a_in) {
  const QArgs a = with_device_key(a_in);
  constexpr int VEC = 8;
  constexpr int NT = LANES == 512 ? 512 : 256;
  constexpr int SEG_PER_BLOCK = NT / LANES;
  constexpr int NSET = PAIR ? 2 : 1;
  static_assert(!COLMAX || (!PAIR && SEG_PER_BLOCK == 1), "column maxima: one whole row per block");
  __shared__ float smem[NSET][NT / 64];
  const int tid = threadIdx.x;
  const int lane = tid % LANES;
  const int64_t nseg_grid = PAIR ? a.nseg / 2 : a.nseg;
  // A last piece that would hang over the end starts eight before it (values met twice give the same bytes and the same
  // maximum).  In 32 bits (a segment holds at most 16384 values): one minimum a piece.
  const int len = (int)a.L;
  auto has_piece = [&](int it) { return (it * LANES + lane) * VEC < len; };
  // (64 bits on the run-time pipeline, whose noise counters are: 10000 rows of 2048 float32 values to e4m3 23.1 us, 24.8
  // with its piece positions in 32)
  auto piece_at = [&](int it) -> std::conditional_t<SPEC == 0, int64_t, int> {
    const int j = (it * LANES + lane) * VEC;
    return j < len - VEC ? j : len - VEC;
  };
  float colmax[COLMAX ? ITERS : 1][VEC];  // largest clipped |x / scale| per column (rounded at the end)
  if constexpr (COLMAX) {
#pragma unroll
    for (int it = 0; it < ITERS; ++it)
#pragma unroll
      for (int e = 0; e < VEC; ++e) colmax[it][e] = 0.0f;
  }
  for (int64_t blk = blockIdx.x;; blk += gridDim.x) {
  if constexpr (COLMAX) {
    if (blk >= nseg_grid) break;  // uniform over the block
  }
  const int64_t seg0 = blk * SEG_PER_BLOCK + tid / LANES;
  const bool active = seg0 < nseg_grid;
  const int64_t segs_per_row = a.cols / a.L;

  constexpr bool PACKED = (sizeof(TIn) == 2) && (SPEC != 0);
  static_assert(!(sizeof(TIn) == 2 && spec_is_f32(SPEC)), "bf16 input is held in bf16");
  RowVals<PACKED> v[NSET][ITERS];
  float scale[NSET], inv[NSET];
  int64_t grow[NSET], col0[NSET];
#pragma unroll
  for (int s = 0; s < NSET; ++s) {
    const int64_t seg = seg0 + (int64_t)s * nseg_grid;
    grow[s] = active ? seg / segs_per_row : 0;  // b * rows + r
    col0[s] = active ? (seg % segs_per_row) * a.L : 0;
    const int64_t b = grow[s] / a.rows, r = grow[s] % a.rows;
    const TIn* xp = reinterpret_cast<const TIn*>(a.x) + grow[s] * a.cols + col0[s];
    const float* psv = a.prescale + b * a.psb;
    float row_ps = 1.0f;
    if (a.ps_mode == AQTX_PRESCALE_PER_ROW) row_ps = psv[r];
    float amax = 0.0f;
    uint32_t amax_packed = 0u;
#pragma clang loop unroll(full)
    for (int it = 0; it < ITERS; ++it) {
      const auto j0 = piece_at(it);
      if (active && has_piece(it)) {
        bool stored = false;
        if constexpr (PACKED) {
          if (a.ps_mode == AQTX_PRESCALE_NONE) {  // the loaded words are the stored form
            const uint4 raw = load_unaligned<uint4>(xp + j0);
            v[s][it].w[0] = raw.x; v[s][it].w[1] = raw.y; v[s][it].w[2] = raw.z; v[s][it].w[3] = raw.w;
#pragma unroll
            for (int i = 0; i < 4; ++i) amax_packed = packed_absmax(amax_packed, v[s][it].w[i]);
            stored = true;
          }
        }
        if (!stored) {
          float t[VEC];
          Loader<TIn>::load8(xp + j0, t);
          if (a.ps_mode == AQTX_PRESCALE_PER_ROW) {
#pragma unroll
            for (int e = 0; e < VEC; ++e) t[e] = spec_prescale<SPEC>(t[e], row_ps, a);
          } else if (a.ps_mode == AQTX_PRESCALE_PER_COL) {
            float ps[8];
            Loader<float>::load8(psv + col0[s] + j0, ps);
#pragma unroll
            for (int e = 0; e < VEC; ++e) t[e] = spec_prescale<SPEC>(t[e], ps[e], a);
          }
          v[s][it].put(t);
          if constexpr (PACKED) {  // the values are bf16 by now: two magnitudes per integer max
#pragma unroll
            for (int i = 0; i < 4; ++i) amax_packed = packed_absmax(amax_packed, v[s][it].w[i]);
          } else {
#pragma unroll
            for (int e = 0; e < VEC; ++e) amax = absmax_step(amax, t[e]);
          }
        }
      } else {
        v[s][it].zero();
      }
    }
    if constexpr (PACKED)
      amax = nanmax(amax, nanmax(__uint_as_float(amax_packed << 16), __uint_as_float(amax_packed & 0xFFFF0000u)));
    amax = segment_max<LANES>(amax, smem[s]);
    if (a.scale_given) {
      scale[s] = active ? given_scale(a, seg) : 1.0f;
      inv[s] = inv_of_scale(scale[s], a);
    } else {
      spec_scale_from_absmax<SPEC>(amax, a, scale[s], inv[s]);
      if (active && lane == 0) store_scale(a, seg, scale[s]);
    }
  }

  if (a.scale_only) return;
  uint8_t* qp0 = reinterpret_cast<uint8_t*>(a.q) + grow[0] * a.cols + col0[0];
  if constexpr (PAIR) {
    uint8_t* qp1 = reinterpret_cast<uint8_t*>(a.q) + grow[1] * a.cols + col0[1];
    const uint32_t ctr_row = (uint32_t)(grow[0] * a.cols);  // natural layout: index of (row, 0)
#pragma clang loop unroll(full)
    for (int it = 0; it < ITERS; ++it) {
      const auto j0 = piece_at(it);
      if (active && has_piece(it)) {
        uint32_t q0[VEC], q1[VEC];
        float t0[VEC], t1[VEC];
        v[0][it].get(t0);
        v[1][it].get(t1);
#pragma unroll
        for (int e = 0; e < VEC; ++e)
          pair_quant<SPEC>(t0[e], inv[0], t1[e], inv[1], ctr_row + (uint32_t)(j0 + e), a, q0[e], q1[e]);
        store8(qp0 + j0, pack8(q0, a.even_odd8));
        store8(qp1 + j0, pack8(q1, a.even_odd8));
      }
    }
  } else {
    const int64_t b = grow[0] / a.rows, r = grow[0] % a.rows;
    const uint64_t ctr_row = (uint64_t)(b * a.nsb + r * a.nsr + col0[0] * a.nsc);
#pragma clang loop unroll(full)
    for (int it = 0; it < ITERS; ++it) {
      const auto j0 = piece_at(it);
      if (active && has_piece(it)) {
        uint32_t q[VEC];
        float t[VEC];
        v[0][it].get(t);
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          if constexpr (COLMAX) {
            float tc;
            q[e] = spec_quant_mag<SPEC>(t[e], inv[0], ctr_row + (uint64_t)((int64_t)(j0 + e) * a.nsc), a, tc);
            colmax[it][e] = fmaxf(colmax[it][e], fabsf(tc));
          } else {
            q[e] = spec_quant<SPEC>(t[e], inv[0], ctr_row + (uint64_t)((int64_t)(j0 + e) * a.nsc), a);
          }
        }
        store8(qp0 + j0, pack8(q, a.even_odd8));
      }
    }
  }
  if constexpr (!COLMAX) break;
  __syncthreads();  // the next row's abs-max goes through the same LDS words
  }
  if constexpr (COLMAX) {
#pragma clang loop unroll(full)
    for (int it = 0; it < ITERS; ++it) {
      const auto j0 = piece_at(it);
      if (has_piece(it)) {
        uint32_t m[VEC];
#pragma unroll
        for (int e = 0; e < VEC; ++e) m[e] = (uint32_t)(int)rintf(colmax[it][e]);
        *reinterpret_cast<uint2*>(a.oa_out + (int64_t)blockIdx.x * a.cols + j0) = pack8(m, 0);
      }
    }
  }
}

// Generic rows kernel: segments shorter than 8 or longer than 16384, and others (element_rows_ahead); one wave per
// segment, two reads.
template <typename TIn>
__global__ __launch_bounds__(256) void quant_rows_generic_kernel(const QArgs a_in) {
  const QArgs a = with_device_key(a_in);
  const int lane = threadIdx.x & 63;
  const int64_t seg = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (seg >= a.nseg) return;  // the whole wave leaves together; no barrier below
  const int64_t segs_per_row = a.cols / a.L;
  const int64_t grow = seg / segs_per_row;
  const int64_t col0 = (seg % segs_per_row) * a.L;
  const int64_t b = grow / a.rows, r = grow % a.rows;
  const TIn* xp = reinterpret_cast<const TIn*>(a.x) + grow * a.cols + col0;
  auto value = [&](int64_t j) {
    float v = Loader<TIn>::load1(xp + j);
    if (a.ps_mode == AQTX_PRESCALE_PER_ROW) v = apply_prescale(v, a.prescale[b * a.psb + r], a);
    else if (a.ps_mode == AQTX_PRESCALE_PER_COL) v = apply_prescale(v, a.prescale[b * a.psb + col0 + j], a);
    return v;
  };
  float amax = 0.0f;
  for (int64_t j = lane; j < a.L; j += 64) amax = absmax_step(amax, value(j));
  amax = segment_max<64>(amax, nullptr);
  float scale, inv;
  if (a.scale_given) {
    scale = given_scale(a, seg);
    inv = inv_of_scale(scale, a);
  } else {
    scale_from_absmax(amax, a, scale, inv);
    if (lane == 0) store_scale(a, seg, scale);
  }
  if (a.scale_only) return;
  uint8_t* qp = reinterpret_cast<uint8_t*>(a.q) + grow * a.cols + col0;
  const uint64_t ctr_row = (uint64_t)(b * a.nsb + r * a.nsr + col0 * a.nsc);
  for (int64_t j = lane; j < a.L; j += 64) {
    const float t = scaled_noisy_clipped(value(j), inv, ctr_row + (uint64_t)(j * a.nsc), a);
    qp[j] = (uint8_t)to_qbyte(t, a.out_dtype);
  }
}

// ---- tile kernels: reduced axis strided (or the whole tensor) -------------------

__global__ void fill_u32_kernel(uint32_t* p, int64_t n, uint32_t v) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}


// What the last block of a group finds out: whether every block of it has merged its maxima.  The atomics are
// read-modify-writes, carried out at the memory side of the per-XCD L2s, and every thread has waited for the value its
// own returned before the barrier in front of the count, so the exchange needs no fence (each of the group's words is
// read by one more read-modify-write).
__device__ __forceinline__ bool last_arrival(uint32_t* arrived, uint32_t blocks, int* flag) {
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t before = __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *flag = before + 1u == blocks;
    if (before + 1u == blocks) __hip_atomic_fetch_and(arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  return *flag != 0;
}

// Merges one maximum; the wait for the returned value orders it before last_arrival's count.
__device__ __forceinline__ void merge_absmax(uint32_t* word, float m) {
  const uint32_t before = __hip_atomic_fetch_max(word, __float_as_uint(m), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("" ::"v"(before));
}

// Scale (output) and reciprocal scale (workspace) of index i from the merged maximum, whose word goes back to zero.
__device__ __forceinline__ void finalize_merged(const QArgs& a, int64_t i) {
  const uint32_t w = __hip_atomic_fetch_and(a.ws_absmax + i, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  float scale, inv;
  scale_from_absmax(__uint_as_float(w), a, scale, inv);
  store_scale(a, i, scale);
  a.ws_inv[i] = inv;
}

// Scale (output) and reciprocal scale (workspace) of index i from a maximum that nothing is merged with.
__device__ __forceinline__ void finalize_alone(const QArgs& a, int64_t i, float m) {
  float scale, inv;
  scale_from_absmax(m, a, scale, inv);
  store_scale(a, i, scale);
  a.ws_inv[i] = inv;
}

// Column abs-max: block = WAVES waves x (64 lanes x VEC cols); the waves interleave
// over the rows of one chunk, partial maxima meet in LDS and leave through one
// atomic max per column (|x| >= 0, so the float bit pattern orders like a uint).
// Bound by HBM bytes on large inputs, by the latency of loads, atomics and launches on small ones.  A wave requests four
// rows before it uses the first (bf16 without a prescale).  FOLD, for launches of few blocks: 16 waves in each, whose one
// round of requests is the whole chunk, and the last block of a column group to arrive computes its scales (QArgs::ws_arrived),
// which spares finalize_scales_kernel, 4 to 5 us mostly of gap: 512 to 2048 columns take 6-12 us instead of 9-14 and that
// launch.  On a chip full of blocks both cost more than they give, as blocks wait at barriers and for the atomics' returns:
// 8192 x 14336 with a prescale 61-88 us against 57 and the launch.  Chunks of 16 rows, for more blocks, take four times the
// atomics (4096 x 2048 float32: 22 us against 12).  A group of one chunk has its scales from its block, with no atomics.
template <typename TIn, int VEC, bool FOLD>
__global__ __launch_bounds__(FOLD ? 1024 : 256) void absmax_cols_kernel(const QArgs a) {
  constexpr int WAVES = FOLD ? 16 : 4;
  constexpr int WIDTH = kAbsColLanes * VEC;
  __shared__ float smem[WAVES][WIDTH];
  __shared__ int last;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // a lane's columns; where eight would hang over the end, the last eight of the row (met twice: same maximum)
  auto columns_at = [&](int64_t l) -> int64_t {
    const int64_t c = (int64_t)blockIdx.x * WIDTH + l * VEC;
    return c >= a.cols ? a.cols : c + VEC <= a.cols ? c : a.cols - VEC;
  };
  const int64_t c0 = columns_at(lane);
  const int64_t chunks_per_group = (a.G + kAbsRowChunk - 1) / kAbsRowChunk;
  const int64_t g = blockIdx.y / chunks_per_group;
  const int64_t chunk = blockIdx.y % chunks_per_group;
  const int64_t b = blockIdx.z;
  const int64_t r_begin = g * a.G + chunk * kAbsRowChunk;
  int64_t r_end = r_begin + kAbsRowChunk;
  if (r_end > (g + 1) * a.G) r_end = (g + 1) * a.G;
  constexpr int AHEAD = 4;  // rows of a wave in flight
  float m[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) m[e] = 0.0f;
  if (c0 < a.cols) {
    const TIn* xb = reinterpret_cast<const TIn*>(a.x) + b * a.rows * a.cols + c0;
    bool done = false;
    if constexpr (VEC == 8 && sizeof(TIn) == 2) {
      if (a.ps_mode == AQTX_PRESCALE_NONE) {  // bf16 magnitudes order like unsigned integers, two per instruction
        done = true;
        uint32_t mw[4] = {0u, 0u, 0u, 0u};
        auto meet = [&](const uint4& w) {
          mw[0] = packed_absmax(mw[0], w.x); mw[1] = packed_absmax(mw[1], w.y);
          mw[2] = packed_absmax(mw[2], w.z); mw[3] = packed_absmax(mw[3], w.w);
        };
        int64_t r = r_begin + wave;
        for (; r + WAVES * (AHEAD - 1) < r_end; r += WAVES * AHEAD) {
          uint4 w[AHEAD];
#pragma unroll
          for (int u = 0; u < AHEAD; ++u) w[u] = load_unaligned<uint4>(xb + (r + WAVES * u) * a.cols);
#pragma unroll
          for (int u = 0; u < AHEAD; ++u) meet(w[u]);
        }
        for (; r < r_end; r += WAVES) meet(load_unaligned<uint4>(xb + r * a.cols));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          m[2 * i] = __uint_as_float(mw[i] << 16);
          m[2 * i + 1] = __uint_as_float(mw[i] & 0xFFFF0000u);
        }
      }
    }
    if (!done) {
      float ps[VEC];
#pragma unroll
      for (int e = 0; e < VEC; ++e) ps[e] = 1.0f;
      if (a.ps_mode == AQTX_PRESCALE_PER_COL) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) ps[e] = a.prescale[b * a.psb + c0 + e];
      }
      for (int64_t r = r_begin + wave; r < r_end; r += WAVES) {
        float v[VEC];
        if constexpr (VEC == 8) Loader<TIn>::load8(xb + r * a.cols, v);
        else v[0] = Loader<TIn>::load1(xb + r * a.cols);
        if (a.ps_mode == AQTX_PRESCALE_PER_ROW) {
          const float rp = a.prescale[b * a.psb + r];
#pragma unroll
          for (int e = 0; e < VEC; ++e) v[e] = apply_prescale(v[e], rp, a);
        } else if (a.ps_mode == AQTX_PRESCALE_PER_COL) {
#pragma unroll
          for (int e = 0; e < VEC; ++e) v[e] = apply_prescale(v[e], ps[e], a);
        }
#pragma unroll
        for (int e = 0; e < VEC; ++e) m[e] = absmax_step(m[e], v[e]);
      }
    }
  }
#pragma unroll
  for (int e = 0; e < VEC; ++e) smem[wave][lane * VEC + e] = m[e];
  __syncthreads();
  for (int i = threadIdx.x; i < WIDTH; i += 64 * WAVES) {
    const int64_t first = columns_at(i / VEC), c = first + i % VEC;
    // (columns a last group of fewer than eight borrows from the group before it belong to that one's blocks)
    if (first < a.cols && c >= (int64_t)blockIdx.x * WIDTH) {
      float mm = smem[0][i];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) mm = nanmax(mm, smem[w][i]);
      const int64_t index = b * a.ssb + g * a.ssg + c * a.ssc;
      if (chunks_per_group == 1) finalize_alone(a, index, mm);
      else if constexpr (FOLD) merge_absmax(a.ws_absmax + index, mm);
      else atomicMax(a.ws_absmax + index, __float_as_uint(mm));
    }
  }
  if constexpr (FOLD) {
    if (chunks_per_group == 1) return;
    if (!last_arrival(a.ws_arrived + (b * a.ngroups + g) * gridDim.x + blockIdx.x, (uint32_t)chunks_per_group, &last)) return;
    const int64_t end = (int64_t)(blockIdx.x + 1) * WIDTH;
    for (int64_t c = (int64_t)blockIdx.x * WIDTH + threadIdx.x; c < end && c < a.cols; c += 64 * WAVES)
      finalize_merged(a, b * a.ssb + g * a.ssg + c * a.ssc);
  }
}

// Whole-tensor abs-max per batch entry (one entry for the whole batch where the batch shares its scale).  An entry of one
// block has its scale from it, with no atomics.
template <typename TIn, int THREADS>
__global__ __launch_bounds__(THREADS) void absmax_all_kernel(const QArgs a) {
  __shared__ float smem[THREADS / 64];
  __shared__ int last;
  const int64_t b = blockIdx.y;
  const int64_t n = a.rows * a.cols;
  const TIn* xb = reinterpret_cast<const TIn*>(a.x) + b * n;
  float m = 0.0f;
  if (n >= 8 && (a.ps_mode == AQTX_PRESCALE_NONE || a.cols % 8 == 0)) {
    // 8 elements per lane and load (with a prescale: of one row); the last eight of the entry are met twice where their
    // number is no multiple of 8
    const int64_t stride = (int64_t)gridDim.x * THREADS * 8;
    const int64_t j0 = ((int64_t)blockIdx.x * THREADS + threadIdx.x) * 8;
    bool done = false;
    if constexpr (sizeof(TIn) == 2) {
      if (a.ps_mode == AQTX_PRESCALE_NONE) {
        done = true;
        uint32_t mw[4] = {0u, 0u, 0u, 0u};
#pragma unroll 4
        for (int64_t j = j0; j < n; j += stride) {
          const uint4 w = load_unaligned<uint4>(xb + (j + 8 <= n ? j : n - 8));
          mw[0] = packed_absmax(mw[0], w.x); mw[1] = packed_absmax(mw[1], w.y);
          mw[2] = packed_absmax(mw[2], w.z); mw[3] = packed_absmax(mw[3], w.w);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
          m = nanmax(m, nanmax(__uint_as_float(mw[i] << 16), __uint_as_float(mw[i] & 0xFFFF0000u)));
      }
    }
    if (!done) {
#pragma unroll 4
      for (int64_t j = j0; j < n; j += stride) {
        const int64_t i = j + 8 <= n ? j : n - 8;
        float v[8];
        Loader<TIn>::load8(xb + i, v);
        if (a.ps_mode == AQTX_PRESCALE_PER_ROW) {
          const float rp = a.prescale[b * a.psb + i / a.cols];
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = apply_prescale(v[e], rp, a);
        } else if (a.ps_mode == AQTX_PRESCALE_PER_COL) {
          float ps[8];
          Loader<float>::load8(a.prescale + b * a.psb + i % a.cols, ps);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = apply_prescale(v[e], ps[e], a);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) m = absmax_step(m, v[e]);
      }
    }
  } else {
    for (int64_t i = (int64_t)blockIdx.x * THREADS + threadIdx.x; i < n; i += (int64_t)gridDim.x * THREADS) {
      float v = Loader<TIn>::load1(xb + i);
      if (a.ps_mode == AQTX_PRESCALE_PER_ROW) v = apply_prescale(v, a.prescale[b * a.psb + i / a.cols], a);
      else if (a.ps_mode == AQTX_PRESCALE_PER_COL) v = apply_prescale(v, a.prescale[b * a.psb + i % a.cols], a);
      m = absmax_step(m, v);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = nanmax(m, __shfl_xor(m, off, 64));
  if ((threadIdx.x & 63) == 0) smem[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < THREADS / 64; ++w) m = nanmax(m, smem[w]);
  }
  const uint32_t blocks = a.ssb != 0 ? gridDim.x : gridDim.x * gridDim.y;
  if (blocks == 1) {
    if (threadIdx.x == 0) finalize_alone(a, b * a.ssb, m);
    return;
  }
  if (threadIdx.x == 0) merge_absmax(a.ws_absmax + b * a.ssb, m);
  if (a.ws_arrived == nullptr) return;
  if (last_arrival(a.ws_arrived + b * a.ssb, blocks, &last) && threadIdx.x == 0) finalize_merged(a, b * a.ssb);
}

// abs-max bit patterns -> scale (output) and reciprocal scale (workspace).
__global__ void finalize_scales_kernel(const QArgs a, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float scale, inv;
  if (a.scale_given) {
    scale = given_scale(a, i);
    inv = inv_of_scale(scale, a);
  } else {
    scale_from_absmax(__uint_as_float(a.ws_absmax[i]), a, scale, inv);
    a.ws_absmax[i] = 0u;  // the abs-max words leave as they have to arrive: zero
    store_scale(a, i, scale);
  }
  a.ws_inv[i] = inv;
}

// Partial maxima of |x| (bytes, [parts][n], written by an earlier launch next to the int8 values this one reads)
// -> scale (output) and reciprocal scale (workspace), in place of the abs-max pass and finalize_scales_kernel.
// A block takes 16 scales: thread t folds the 16 bytes of parts t, t + 256, ... (as eight pairs of 16-bit lanes,
// two maxima per instruction), the threads meet through wave shuffles and LDS.  (64 scales per block, whose loads
// use whole 64-byte sectors, leave 64 blocks for 4096 scales and measured slower: 11.6 against 8.1 us on average
// over 1792 and 224 parts.)
typedef unsigned short u16x2_max_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pk_max_u16(uint32_t x, uint32_t y) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2_max_t, x),
                                                                __builtin_bit_cast(u16x2_max_t, y)));
}
__global__ __launch_bounds__(256) void finalize_partials_kernel(const QArgs a, int64_t n) {
  __shared__ uint32_t smax[4][8];
  const int64_t c0 = (int64_t)blockIdx.x * 16;  // n is a multiple of 16 here
  uint32_t m[8];  // m[2 i] = bytes 0 and 2 of word i in 16-bit lanes, m[2 i + 1] = bytes 1 and 3
#pragma unroll
  for (int i = 0; i < 8; ++i) m[i] = 0u;
  for (int64_t p = threadIdx.x; p < a.oa_in_parts; p += 256) {
    const uint4 w = *reinterpret_cast<const uint4*>(a.oa_in + p * n + c0);
    const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      m[2 * i] = pk_max_u16(m[2 * i], ww[i] & 0x00FF00FFu);
      m[2 * i + 1] = pk_max_u16(m[2 * i + 1], (ww[i] >> 8) & 0x00FF00FFu);
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m[i] = pk_max_u16(m[i], (uint32_t)__shfl_xor((int)m[i], off, 64));
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int i = 0; i < 8; ++i) smax[wave][i] = m[i];
  }
  __syncthreads();
  if (threadIdx.x < 16) {
    // column c0 + t is byte t % 4 of word t / 4: lane (t % 4) / 2 of m[2 (t / 4) + t % 2]
    const int t = threadIdx.x, i = 2 * (t >> 2) + (t & 1), hi = (t >> 1) & 1;
    uint32_t v = pk_max_u16(pk_max_u16(smax[0][i], smax[1][i]), pk_max_u16(smax[2][i], smax[3][i]));
    v = hi ? v >> 16 : v & 0xFFFFu;
    float scale, inv;
    scale_from_absmax((float)v, a, scale, inv);
    store_scale(a, c0 + t, scale);
    a.ws_inv[c0 + t] = inv;
  }
}


// Columns in one pass: a block owns 8 << tshift whole columns, reads them once into registers, finds their scales and
// writes the quantized values; no abs-max launch, no workspace, no second read.  A thread holds kOnceRows consecutive rows of
// 8 columns, so the bytes of a column (transposed output) leave as one 16-byte (float32: 8-byte) store a thread, 64 lanes together
// covering whole lines.  Bound by HBM bytes: one read and one write.
// ROWMAX (8 threads a row): see quant_tile_kernel.
template <typename TIn, int SPEC, bool ROWMAX>
__global__ __launch_bounds__(1024) void quant_cols_once_kernel(const QArgs a, const int tshift) {
  constexpr int R = kOnceRows<sizeof(TIn)>, W = 8 * sizeof(TIn) / 16;
  __shared__ __attribute__((aligned(16))) uint32_t smax[16][8 << kOnceMaxShift];
  __shared__ __attribute__((aligned(16))) float sinv[8 << kOnceMaxShift];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int T = 1 << tshift, width = 8 << tshift, slot = tid & (T - 1);
  // Blocks of part of a line (2 or 4 threads a row): those of one line go to blocks i, i + 8, ..., which share an XCD.
  int cb = blockIdx.x;
  const int sib = 3 - tshift > 0 ? 3 - tshift : 0;
  if (cb < ((int)gridDim.x & -(8 << sib))) cb = (cb & -(8 << sib)) | ((cb & 7) << sib) | ((cb >> 3) & ((1 << sib) - 1));
  // a thread's columns and rows; where they would hang over the end, the last ones (met twice: the same bytes twice)
  auto columns_at = [&](int t) -> int64_t {
    const int64_t c = (int64_t)cb * width + t * 8;
    return c >= a.cols ? a.cols : c + 8 <= a.cols ? c : a.cols - 8;
  };
  const int64_t c0 = columns_at(slot);
  int64_t r0 = (int64_t)(tid >> tshift) * R;
  const bool active = c0 < a.cols && r0 < a.rows;
  if (r0 + R > a.rows) r0 = a.rows - R;
  const int64_t b = blockIdx.y;
  uint4 w[R][W];
  if (active) {
    const TIn* p = reinterpret_cast<const TIn*>(a.x) + (b * a.rows + r0) * a.cols + c0;
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
      for (int h = 0; h < W; ++h) w[j][h] = load_unaligned<uint4>(p + j * a.cols + h * (8 / W));
  } else {
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
      for (int h = 0; h < W; ++h) w[j][h] = make_uint4(0, 0, 0, 0);
  }
  // magnitudes order like unsigned integers, NaN above infinity
  uint32_t m[4 * W];
#pragma unroll
  for (int i = 0; i < 4 * W; ++i) m[i] = 0u;
#pragma unroll
  for (int j = 0; j < R; ++j)
#pragma unroll
    for (int h = 0; h < W; ++h) {
      const uint32_t x[4] = {w[j][h].x, w[j][h].y, w[j][h].z, w[j][h].w};
#pragma unroll
      for (int i = 0; i < 4; ++i) m[4 * h + i] = once_max<TIn>(m[4 * h + i], sizeof(TIn) == 2 ? x[i] & 0x7FFF7FFFu : x[i] & 0x7FFFFFFFu);
    }
  for (int off = T; off < 64; off <<= 1)
#pragma unroll
    for (int i = 0; i < 4 * W; ++i) m[i] = once_max<TIn>(m[i], (uint32_t)__shfl_xor((int)m[i], off, 64));
  if (lane < T) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      smax[wave][lane * 8 + e] = sizeof(TIn) == 2 ? ((e & 1) ? m[e >> 1] & 0xFFFF0000u : m[e >> 1] << 16) : m[e];
  }
  __syncthreads();
  for (int i = tid; i < width; i += blockDim.x) {
    const int64_t first = columns_at(i >> 3), c = first + (i & 7);
    if (first < a.cols) {
      uint32_t mm = smax[0][i];
      for (int v = 1; v < ((int)blockDim.x >> 6); ++v) mm = mm > smax[v][i] ? mm : smax[v][i];
      float scale, inv;
      spec_scale_from_absmax<SPEC>(__uint_as_float(mm), a, scale, inv);
      store_scale(a, b * a.ssb + c * a.ssc, scale);
      sinv[i] = inv;
    }
  }
  __syncthreads();
  if (!active) return;  // (ROWMAX: whole rows of the block's threads at a time)
  float inv[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) inv[e] = sinv[slot * 8 + e];
  uint8_t* q = reinterpret_cast<uint8_t*>(a.q) + b * a.rows * a.cols;
  uint32_t out[8][R / 4], rmax[R / 4];
#pragma unroll
  for (int i = 0; i < R / 4; ++i) {
    rmax[i] = 0u;
#pragma unroll
    for (int e = 0; e < 8; ++e) out[e][i] = 0u;
  }
#pragma unroll
  for (int j = 0; j < R; ++j) {
    float v[8], rm = 0.0f;
    once_unpack<TIn>(w[j], v);
    uint32_t qv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if constexpr (ROWMAX) {
        float tc;
        qv[e] = spec_quant_mag<SPEC>(v[e], inv[e], 0, a, tc);
        rm = fmaxf(rm, fabsf(tc));
      } else {
        qv[e] = spec_quant<SPEC>(v[e], inv[e], 0, a);
      }
      out[e][j >> 2] |= qv[e] << (8 * (j & 3));
    }
    if constexpr (ROWMAX) {
#pragma unroll
      for (int off = 1; off < 8; off <<= 1) rm = fmaxf(rm, __shfl_xor(rm, off, 64));
      rmax[j >> 2] |= (uint32_t)(int)rintf(rm) << (8 * (j & 3));
    }
    __builtin_amdgcn_sched_barrier(0);  // row after row, so that their bytes take the registers of the values
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) __builtin_memcpy(q + (c0 + e) * a.rows + r0, out[e], R);
  if constexpr (ROWMAX) {
    if (slot == 0) __builtin_memcpy(a.oa_out + (int64_t)cb * a.rows + r0, rmax, R);
  }
}

// 128x64 tile: thread (rg = tid/8, cc = tid%8) owns rows 4*rg..+3, cols 8*cc..+7; with RPT = 1, a 32x64 tile and one row.
// PAIR (SPEC 2 and 7, and SPEC 5 with value 1): 1 = the block also owns the tile `rows/2` further down (natural noise
// layout), 2 = the tile `cols/2` further right (noise counters of the transposed tensor); the
// two tiles' elements share threefry blocks.
// ROWMAX (no PAIR; every tile interior): the block also finds, for each of its 128 rows, the largest |q| among its 64
// columns, and stores them as bytes rows r0.. of row blockIdx.x of QArgs::oa_out ([column tiles][rows]).
template <typename TIn, int SPEC, int PAIR, bool ROWMAX = false, int RPT = 4>
__global__ __launch_bounds__(256) void quant_tile_kernel(const QArgs a_in) {
  static_assert(!ROWMAX || (PAIR == 0 && RPT == 4), "row maxima: one tile per block");
  static_assert(RPT == 4 || RPT == 1, "rows a thread");
  constexpr int TR = 32 * RPT, TPAD = TR + 4;  // rows of the tile; LDS bytes a column
  const QArgs a = with_device_key(a_in);
  constexpr int NSET = PAIR ? 2 : 1;
  __shared__ uint32_t lds[NSET][kTileC * TPAD / 4];
  const int tid = threadIdx.x;
  const int cc = tid & 7, rg = tid >> 3;
  const int64_t b = blockIdx.z;
  const TIn* xb = reinterpret_cast<const TIn*>(a.x) + b * a.rows * a.cols;
  uint8_t* qb = reinterpret_cast<uint8_t*>(a.q) + b * a.rows * a.cols;
  int64_t r0[NSET], c0[NSET];
  r0[0] = (int64_t)blockIdx.y * TR;
  c0[0] = (int64_t)blockIdx.x * kTileC;
  // the first tile of a pair stays inside the first half of the paired axis
  const int64_t row_lim = PAIR == 1 ? a.rows / 2 : a.rows;
  const int64_t col_lim = PAIR == 2 ? a.cols / 2 : a.cols;
  // A last tile that would hang over the end moves back inside (values two blocks meet give the same bytes in both), so
  // that every tile of a tensor of at least one tile takes the branch-free path.  SPEC 5 draws for pairs of columns
  // that start at an even one.  (1999 x 1030, 1999 x 3001 and 1030 x 3001 values with byte and element accesses on every
  // tile: 24, 36 and 18 us, the first two with noise; now 15, 26 and 7.)
  if (r0[0] + TR > row_lim && row_lim >= TR) r0[0] = row_lim - TR;
  if (c0[0] + kTileC > col_lim && col_lim >= kTileC && (SPEC != 5 || col_lim % 2 == 0)) c0[0] = col_lim - kTileC;
  if constexpr (PAIR == 1) { r0[1] = r0[0] + a.rows / 2; c0[1] = c0[0]; }
  if constexpr (PAIR == 2) { r0[1] = r0[0]; c0[1] = c0[0] + a.cols / 2; }

  uint32_t words[NSET][2][RPT];  // words[s][h][j] = bytes of cols c+4*h..c+4*h+3 at row RPT*rg+j
#pragma unroll
  for (int s = 0; s < NSET; ++s)
#pragma unroll
    for (int j = 0; j < RPT; ++j) words[s][0][j] = words[s][1][j] = 0u;

  // Tiles that lie wholly inside the tensor (and inside the first half of a paired axis) take a
  // branch-free path with vector loads of the reciprocal scales and the pre-scale factors.
  const bool interior = (r0[0] + TR <= row_lim) && (c0[0] + kTileC <= col_lim) && a.ssc <= 1;
  // Every lane of the tile that has values has eight: one decision for the tile, before each lane's own (64 x 64 values
  // with noise and one scale 15.3 us; 18.8 with the lanes' decision alone).
  const bool whole = a.cols % 8 == 0 && col_lim % 8 == 0;
  // Given scales: the tile's reciprocals are computed here (LDS), where the rows of a column share one
  __shared__ float inv_lds[NSET][kTileC];
  const bool inv_here = a.scale_given && a.ngroups == 1;
  if (inv_here) {
    if (tid < kTileC) {
#pragma unroll
      for (int s = 0; s < NSET; ++s) {
        const int64_t c = c0[s] + tid;
        inv_lds[s][tid] = c < a.cols ? inv_of_scale(given_scale(a, b * a.ssb + c * a.ssc), a) : 1.0f;
      }
    }
    __syncthreads();
  }
  uint32_t rowmax = 0u;  // ROWMAX: byte j = largest |q| of row r0 + 4 * rg + j among the tile's 64 columns
  auto rows = [&](auto fast_tag) {
    constexpr bool FAST = decltype(fast_tag)::value;
    float ps_col[NSET][8];
    if constexpr (FAST) {
      if (a.ps_mode == AQTX_PRESCALE_PER_COL) {
#pragma unroll
        for (int s = 0; s < NSET; ++s) Loader<float>::load8(a.prescale + b * a.psb + c0[s] + cc * 8, ps_col[s]);
      }
    }
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      const int64_t rl = r0[0] + rg * RPT + j;  // position inside the first tile's half
      const int64_t cl = c0[0] + cc * 8;
      if (FAST || (rl < row_lim && cl < col_lim)) {
        const int nvalid = FAST ? 8 : ((col_lim - cl) >= 8 ? 8 : (int)(col_lim - cl));
        float x[NSET][8], inv[NSET][8];
#pragma unroll
        for (int s = 0; s < NSET; ++s) {
          const int64_t r = r0[s] + rg * RPT + j, c = c0[s] + cc * 8;
          if (FAST || whole) {
            Loader<TIn>::load8(xb + r * a.cols + c, x[s]);
          } else if (nvalid == 8) {
            Loader<TIn>::load8(xb + r * a.cols + c, x[s]);
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
              x[s][e] = e < nvalid ? Loader<TIn>::load1(xb + r * a.cols + c + e) : 0.0f;
          }
          const int64_t sbase = b * a.ssb + (r / a.G) * a.ssg;
          if (a.ps_mode == AQTX_PRESCALE_PER_ROW) {
            const float rp = a.prescale[b * a.psb + r];
#pragma unroll
            for (int e = 0; e < 8; ++e) x[s][e] = spec_prescale<SPEC>(x[s][e], rp, a);
          } else if (a.ps_mode == AQTX_PRESCALE_PER_COL) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              if constexpr (FAST) x[s][e] = spec_prescale<SPEC>(x[s][e], ps_col[s][e], a);
              else if (e < nvalid) x[s][e] = spec_prescale<SPEC>(x[s][e], a.prescale[b * a.psb + c + e], a);
            }
          }
          if (inv_here) {
#pragma unroll
            for (int e = 0; e < 8; ++e) inv[s][e] = inv_lds[s][cc * 8 + e];
          } else if constexpr (FAST) {
            if (a.ssc == 0) {
              const float v = a.ws_inv[sbase];
#pragma unroll
              for (int e = 0; e < 8; ++e) inv[s][e] = v;
            } else {
              Loader<float>::load8(a.ws_inv + sbase + c, inv[s]);
            }
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) inv[s][e] = e < nvalid ? a.ws_inv[sbase + (c + e) * a.ssc] : 1.0f;
          }
        }
        uint32_t qs[NSET][8];
#pragma unroll
        for (int s = 0; s < NSET; ++s)
#pragma unroll
          for (int e = 0; e < 8; ++e) qs[s][e] = 0u;
        U2 wbits{0u, 0u};  // SPEC 5: the 32-bit word(s) two neighbouring elements draw their 16 bits from
        float rm = 0.0f;   // ROWMAX: largest clipped |x / scale| of this row among this thread's 8 columns
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          if (FAST || e < nvalid) {
            uint32_t qv[NSET];
            if constexpr (SPEC == 5) {
              // 16-bit draws: elements 2w and 2w+1 share word w; with PAIR the block (w, w + half)
              // also serves the same two elements of the tile rows/2 further down.
              const uint32_t sr_mask = a.out_dtype == AQTX_E4M3 ? 0xFu : 0x1Fu;
              const uint64_t ctr = (uint64_t)(b * a.nsb + rl * a.nsr + (cl + e) * a.nsc);
              if ((e & 1) == 0) {
                if constexpr (PAIR) {
                  wbits = threefry2x32(a.gen.k0, a.gen.k1, (uint32_t)(ctr >> 1), (uint32_t)(ctr >> 1) + a.gen.half);
                } else {
                  wbits.x = a.gen.word_original((uint32_t)(ctr >> 1));
                }
              }
              const int sh = (e & 1) * 16;
#pragma unroll
              for (int s = 0; s < NSET; ++s) {
                float t = round_bf16(x[s][e] * inv[s][e]);
                t = bf16_mantissa_sr(t, (s == 0 ? wbits.x : wbits.y) >> sh, sr_mask);
                qv[s] = spec_finish<5>(t, a);
              }
            } else if constexpr (PAIR) {
              const uint32_t i = (uint32_t)((r0[0] + rg * RPT + j) * a.nsr + (c0[0] + cc * 8 + e) * a.nsc);
              pair_quant<SPEC>(x[0][e], inv[0][e], x[1][e], inv[1][e], i, a, qv[0], qv[1]);
            } else if constexpr (ROWMAX) {
              float tc;
              qv[0] = spec_quant_mag<SPEC>(x[0][e], inv[0][e], 0, a, tc);
              rm = fmaxf(rm, fabsf(tc));
            } else {
              const uint64_t ctr = (uint64_t)(b * a.nsb + rl * a.nsr + (cl + e) * a.nsc);
              qv[0] = spec_quant<SPEC>(x[0][e], inv[0][e], ctr, a);
            }
#pragma unroll
            for (int s = 0; s < NSET; ++s) qs[s][e] = qv[s];
          }
        }
        uint32_t w[NSET][2];
#pragma unroll
        for (int s = 0; s < NSET; ++s) {
          const uint2 v = pack8(qs[s], 0);
          w[s][0] = words[s][0][j] = v.x;
          w[s][1] = words[s][1][j] = v.y;
        }
        if constexpr (ROWMAX) {
          // every tile is interior here, so all lanes are in this branch: the 8 threads of a row (consecutive lanes)
          // meet by shuffles; rint(max |t|) = max |q|
#pragma unroll
          for (int off = 1; off < 8; off <<= 1) rm = fmaxf(rm, __shfl_xor(rm, off, 64));
          rowmax |= (uint32_t)(int)rintf(rm) << (8 * j);
        }
        if (!a.transpose_out) {
#pragma unroll
          for (int s = 0; s < NSET; ++s) {
            const int64_t r = r0[s] + rg * RPT + j, c = c0[s] + cc * 8;
            if (FAST || whole) {
              store8(qb + r * a.cols + c, make_uint2(w[s][0], w[s][1]));
            } else if (nvalid == 8) {
              store8(qb + r * a.cols + c, make_uint2(w[s][0], w[s][1]));
            } else {
              for (int e = 0; e < nvalid; ++e)
                qb[r * a.cols + c + e] = (uint8_t)(w[s][e >> 2] >> (8 * (e & 3)));
            }
          }
        }
      }
    }
  };
  if (interior) rows(std::true_type{});
  else rows(std::false_type{});
  if constexpr (ROWMAX) {
    if (cc == 0)
      *reinterpret_cast<uint32_t*>(a.oa_out + ((int64_t)blockIdx.x * a.rows + r0[0] + rg * 4)) = rowmax;
  }
  if (!a.transpose_out) return;  // uniform across the block

  // Transposed write: LDS holds each tile as [col][row bytes], row stride TPAD B.
#pragma unroll
  for (int s = 0; s < NSET; ++s)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if constexpr (RPT == 4) {
        uint32_t col4[4];
        transpose4(words[s][h], col4);
#pragma unroll
        for (int e = 0; e < 4; ++e) lds[s][((cc * 8 + 4 * h + e) * TPAD + rg * 4) / 4] = col4[e];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          reinterpret_cast<uint8_t*>(lds[s])[(cc * 8 + 4 * h + e) * TPAD + rg] = (uint8_t)(words[s][h][0] >> (8 * e));
      }
    }
  __syncthreads();
  // thread -> 16-byte chunks of the [64][TR] byte tile
  constexpr int CH = TR / 16, ITEMS = kTileC * CH;
#pragma unroll
  for (int s = 0; s < NSET; ++s) {
#pragma unroll
    for (int h = 0; h < (ITEMS + 255) / 256; ++h) {
      if (ITEMS < 256 && tid >= ITEMS) break;
      const int col = (tid + 256 * h) / CH, chunk = (tid + 256 * h) % CH;
      const int64_t gc_l = c0[0] + col, gr_l = r0[0] + chunk * 16;  // bounds in first-tile terms
      const int64_t gc = c0[s] + col, gr = r0[s] + chunk * 16;
      if (gc_l < col_lim && gr_l < row_lim) {
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = lds[s][(col * TPAD + chunk * 16) / 4 + i];
        uint8_t* dst = qb + gc * a.rows + gr;
        const int64_t lim = row_lim - gr_l;
        if (lim >= 16) {
          const uint4 v = make_uint4(w[0], w[1], w[2], w[3]);
          __builtin_memcpy(dst, &v, 16);
        } else {
          const int nv = (int)lim;
          for (int i = 0; i < nv; ++i) dst[i] = (uint8_t)(w[i >> 2] >> (8 * (i & 3)));
        }
      }
    }
  }
}

// ---- host side ---------------------------------------------------------------------

// Which compile-time specialisation (see spec_quant) serves this plan.
int spec_of(const QArgs& a, int partitionable) {
  if (a.cbf && a.sbf && (a.out_dtype == AQTX_E4M3 || a.out_dtype == AQTX_E5M2)) {
    if (a.noise == AQTX_NOISE_NONE) return 3;
    if (a.noise == AQTX_NOISE_FP8_MANTISSA && !partitionable && a.gen.width == 16 && a.nsc == 1 &&
        a.nsr % 2 == 0 && a.nsb % 2 == 0)
      return 5;  // neighbouring elements draw from one word, starting at an even counter
    return 0;
  }
  if (a.cbf != a.sbf || !(a.out_dtype == AQTX_I8 || a.out_dtype == AQTX_I4)) return 0;
  if (a.noise == AQTX_NOISE_NONE) return a.cbf ? 1 : 6;
  if (a.noise == AQTX_NOISE_JAX_UNIFORM && !partitionable) return a.cbf ? 2 : 7;
  return 0;
}

template <typename TIn, int SPEC>
int launch_rows_colmax(const QArgs& a, hipStream_t st) {
  const int64_t L = a.L;
  const int64_t blocks = a.nseg < kColmaxBlocks ? a.nseg : kColmaxBlocks;  // = aqtx_quantize_other_axis_parts: rows of oa_out
#define AQTX_ROWS_CM(ITERS)                                                                                  \
  {                                                                                                          \
    quant_rows_kernel<TIn, 256, ITERS, SPEC, false, true><<<dim3((unsigned)blocks), 256, 0, st>>>(a);        \
    AQTX_HIP_CHECK_LAUNCH("quant_rows_kernel, column maxima");                                               \
    return 0;                                                                                                \
  }
  if (L <= 2048) AQTX_ROWS_CM(1)
  if (L <= 4096) AQTX_ROWS_CM(2)
  AQTX_ROWS_CM(4)
#undef AQTX_ROWS_CM
}

template <typename TIn, int SPEC, bool PAIR>
int launch_rows_spec(const QArgs& a, hipStream_t st) {
  const int64_t L = a.L;
  const int64_t nseg = PAIR ? a.nseg / 2 : a.nseg;
#define AQTX_ROWS(LANES, ITERS)                                                        \
  {                                                                                    \
    constexpr int kThreads = LANES == 512 ? 512 : 256;                                 \
    const int64_t blocks = (nseg + (kThreads / LANES) - 1) / (kThreads / LANES);       \
    quant_rows_kernel<TIn, LANES, ITERS, SPEC, PAIR><<<dim3((unsigned)blocks), kThreads, 0, st>>>(a); \
    AQTX_HIP_CHECK_LAUNCH("quant_rows_kernel");                                        \
    return 0;                                                                          \
  }
  if (L <= 128) AQTX_ROWS(16, 1)
  if (L <= 512) AQTX_ROWS(64, 1)
  if (L <= 2048) AQTX_ROWS(256, 1)
  if (L <= 4096) AQTX_ROWS(256, 2)
  if (L <= 8192) AQTX_ROWS(256, 4)
  if constexpr ((SPEC == 2 && sizeof(TIn) == 2) || SPEC == 7) AQTX_ROWS(512, 4)
  else AQTX_ROWS(256, 8)
#undef AQTX_ROWS
}

// Whether segments whose length is no multiple of 8 go to the kernel with a wave per segment and an element a lane.  Pieces
// of 8 are ahead where loads and stores are what a row costs (1000 rows of 1001 bf16 values 4.3 us against 9.5) and beyond
// 2048 values always.  They lose where a lane's eight draws or conversions follow one another with too few rows to hide
// it, and where rows are many and leave most lanes of a launch shape (128, 512, 2048 values) without a piece.  The lines
// lie where the two measured alike; pieces / elements in us at either side of them, by pipeline:
//   typed, no noise     570 values: 1000 rows 4.2 / 6.6, 10000 15.8 / 14.0; 700: 10000 16.0 / 16.9
//   run time, no noise  20 values: 1000 rows 4.6 / 3.7, 8200 4.6 / 5.7; 129: 40000 24.4 / 23.2; 700: 4000 10.3 / 9.1; 1001: 10.5 / 16.1
//   noise, paired rows  10 values: 10000 rows 13.5 / 7.5, 30000 14.6 / 16.6; 31: 1000 5.2 / 3.9, 8200 6.1 / 6.9; 100: 1000
//                       5.2 / 4.4, 4000 5.3 / 5.9; 129: 100 5.3 / 5.1, 4000 6.6 / 7.3; 570: 1000 6.9 / 8.5, 10000 29.2 / 25.4
//   noise otherwise     10 values: 30000 rows 17.2 / 16.4, 40000 19.6 / 20.9; 31: 10000 8.3 / 7.5, 30000 15.4 / 16.7; 100: 1000
//                       5.9 / 4.4, 8200 8.0 / 8.8; 300: 10000 19.3 / 16.9; 511: 19.7 / 23.4; 700: 1000 7.6 / 9.8, 4000 19.8 / 15.5
inline bool element_rows_ahead(const QArgs& a, int spec, bool paired) {
  const int64_t L = a.L, n = a.nseg;
  if (L % 8 == 0 || L > 2048 || a.even_odd8) return false;
  struct Lines {
    int64_t below16, below64, below128;     // fewer segments than this of a length below 16, 64, 128
    int64_t mid_length, mid_segments;       // lengths beyond 128 below, and fewer segments than
    int64_t long_length, long_segments;     // lengths beyond 512 below, and at least so many segments
  };
  constexpr int64_t kAny = INT64_MAX;
  constexpr Lines kTyped{0, 0, 0, 0, 0, 640, 4096}, kRunTime{4096, 4096, 2048, 160, kAny, 800, 2048},
      kPaired{20480, 6144, 2048, 256, 2048, 640, 4096}, kNoise{32768, 16384, 4096, 400, kAny, 1024, 2048};
  const Lines& l = a.noise == AQTX_NOISE_NONE ? (spec != 0 ? kTyped : kRunTime) : paired ? kPaired : kNoise;
  if (L < 128) return n < (L < 16 ? l.below16 : L < 64 ? l.below64 : l.below128);
  if (L < 512) return L < l.mid_length && n < l.mid_segments;
  return L < l.long_length && n >= l.long_segments;
}

template <typename TIn>
int launch_rows(const QArgs& a, int partitionable, hipStream_t st) {
  const int64_t L = a.L;
  AQTX_REQUIRE(!a.even_odd8 || (L % 8 == 0 && a.cols % 8 == 0 && L <= 16384),
               "aqtx_quantize: out_k_order = EVEN_ODD8 needs cols and group to be multiples of 8 and "
               "segments of at most 16384");
  const int spec = spec_of(a, partitionable);
  // one threefry block serves elements i and i + total/2: pair whole rows when the noise counters follow the
  // natural [batch*rows, cols] order
  const bool natural = a.nsc == 1 && a.nsr == a.cols && (a.batch == 1 || a.nsb == a.rows * a.cols) &&
                       L == a.cols && (a.nseg % 2 == 0);
  if (L < 8 || L > 16384 || element_rows_ahead(a, spec, natural && spec_has_uniform_noise(spec))) {
    const int64_t blocks = (a.nseg + 3) / 4;
    quant_rows_generic_kernel<TIn><<<dim3((unsigned)blocks), 256, 0, st>>>(a);
    AQTX_HIP_CHECK_LAUNCH("quant_rows_generic_kernel");
    return 0;
  }
  // (oa_out: the caller has checked rows_colmax_ok: noise none, so spec is 1, 6 or 0; float input is held in the
  // compute dtype, so the bf16 pipelines never meet float32 input nor the float32 ones bf16 input)
  if constexpr (sizeof(TIn) != 4) {
    if (spec == 1) return a.oa_out != nullptr ? launch_rows_colmax<TIn, 1>(a, st) : launch_rows_spec<TIn, 1, false>(a, st);
    if (spec == 2) return natural ? launch_rows_spec<TIn, 2, true>(a, st) : launch_rows_spec<TIn, 2, false>(a, st);
    if (spec == 3) return launch_rows_spec<TIn, 3, false>(a, st);
    if (spec == 5) return launch_rows_spec<TIn, 5, false>(a, st);
  }
  if constexpr (sizeof(TIn) != 2) {
    if (spec == 6) return a.oa_out != nullptr ? launch_rows_colmax<TIn, 6>(a, st) : launch_rows_spec<TIn, 6, false>(a, st);
    if (spec == 7) return natural ? launch_rows_spec<TIn, 7, true>(a, st) : launch_rows_spec<TIn, 7, false>(a, st);
  }
  return a.oa_out != nullptr ? launch_rows_colmax<TIn, 0>(a, st) : launch_rows_spec<TIn, 0, false>(a, st);
}

template <typename TIn>
int launch_tiles(const QArgs& a, int reduce, int partitionable, int64_t nscales, hipStream_t st) {
  if constexpr (sizeof(TIn) != 1) {
    if (a.once_shift >= 0) {
      const int R = kOnceRows<sizeof(TIn)>, shift = a.once_shift;
      const int threads = (int)((((a.rows + R - 1) / R << shift) + 63) / 64 * 64);
      const dim3 grid((unsigned)((a.cols + (8 << shift) - 1) / (8 << shift)), (unsigned)a.batch);
      constexpr int kInt = sizeof(TIn) == 2 ? 1 : 6;
      if (a.oa_out != nullptr) quant_cols_once_kernel<TIn, kInt, true><<<grid, threads, 0, st>>>(a, shift);
      else quant_cols_once_kernel<TIn, kInt, false><<<grid, threads, 0, st>>>(a, shift);
      AQTX_HIP_CHECK_LAUNCH("quant_cols_once_kernel");
      return 0;
    }
  }
  if (a.oa_in != nullptr) {
    finalize_partials_kernel<<<dim3((unsigned)(nscales / 16)), 256, 0, st>>>(a, nscales);
    AQTX_HIP_CHECK_LAUNCH("finalize_partials_kernel");
  } else {
  bool folded = false;  // the abs-max launch leaves the scales itself
  if (!a.scale_given) {
    if (!a.ws_zeroed) {
      fill_u32_kernel<<<dim3((unsigned)((nscales + 255) / 256)), 256, 0, st>>>(a.ws_absmax, nscales, 0u);
      AQTX_HIP_CHECK_LAUNCH("fill_u32_kernel");
    }
    if (reduce == AQTX_REDUCE_ALL || reduce == AQTX_REDUCE_ALL_BATCH) {
      // Every block ends in two atomics (its maximum and its arrival).  Atomics on one address take turns (about 10 ns
      // each, measured), and so do those on the neighbouring words of the batch entries, which share a cache line: 32
      // entries x 98 blocks took 31 us for 26 MB.  So the launch as a whole aims at one block per 96 KiB of input (the
      // time to stream that much), but at least 64 where there are values for them (small tensors are bound by latency)
      // and at most 512, two of 16 waves on each CU; a batch of more entries has one block for each.  (Calibrated and
      // quantized, against blocks of 4 waves for 48 KiB each, 256 to 2048 of them, and a launch for the scales: bf16 64 x
      // 64 9.6 and 10.3 us, 2048 x 2048 10.6 and 13.4, 8192 x 4096 33.7 and 45.4, 256 entries of 64 x 64 10.9 and 11.0.)
      QArgs whole = a;
      if (reduce == AQTX_REDUCE_ALL_BATCH && a.ps_mode == AQTX_PRESCALE_NONE) {  // the entries follow one another
        whole.rows = a.batch * a.rows;
        whole.batch = 1;
      }
      const int64_t values = whole.rows * whole.cols;
      int64_t nblk = (values + 1024 * 8 - 1) / (1024 * 8);
      const int64_t total_bytes = whole.batch * values * (int64_t)sizeof(TIn);
      int64_t cap_total = total_bytes / (96 << 10);
      cap_total = cap_total < 64 ? 64 : cap_total > 512 ? 512 : cap_total;
      const int64_t cap = whole.batch >= cap_total ? 1 : cap_total / whole.batch;
      if (nblk > cap) nblk = cap;
      if (nblk < 1) nblk = 1;
      folded = a.ws_arrived != nullptr || (nblk == 1 && (whole.batch == 1 || a.ssb != 0));
      const dim3 grid((unsigned)nblk, (unsigned)whole.batch);
      // many small entries: blocks of 4 waves, more of which a CU holds at a time
      if (whole.batch >= 512 && values <= 16384) absmax_all_kernel<TIn, 256><<<grid, 256, 0, st>>>(whole);
      else absmax_all_kernel<TIn, 1024><<<grid, 1024, 0, st>>>(whole);
      AQTX_HIP_CHECK_LAUNCH("absmax_all_kernel");
    } else {
      const dim3 grid((unsigned)absmax_col_groups(a.cols), (unsigned)(a.ngroups * ((a.G + kAbsRowChunk - 1) / kAbsRowChunk)), (unsigned)a.batch);
      // Folded up to two blocks of 16 waves a CU, one round of the chip, and small inputs up to four.  Float values without a
      // prescale are bound by HBM bytes from 8 million on: there only where few blocks share a set of scales.  Calibration and
      // quantization, folded / not, us:
      //   bf16           8192 x 512 12.1 / 12.1, 2048 x 4096 15.7 / 14.8, 4096 x 4096 24.4 / 21.6 (groups of 64 rows 20.5 / 22.3),
      //                  512 x 32768 21.3 / 21.7, 4096 x 5120 28.5 / 24.1
      //   float32        8192 x 512 13.7 / 16.7, 256 x 64 x 64 11.7 / 14.5, 8192 x 1024 21.5 / 21.2, 513 x 16383 24.3 / 26.5,
      //                  4096 x 4096 31.4 / 28.4
      //   bf16 prescaled 2048 x 4096 18.9 / 21.4, 4096 x 4096 27.3 / 28.4, 4608 x 4096 33.7 / 31.5; 50000 x 64 27.1 / 31.0
      //   int8           2048 x 4096 16.3 / 17.4, 4096 x 4096 24.1 / 24.1, 4096 x 5120 28.6 / 25.9; 50000 x 64 24.7 / 27.0
      const int64_t blocks = (int64_t)grid.x * grid.y * grid.z, values = a.batch * a.rows * a.cols;
      const bool bytes_bound = sizeof(TIn) != 1 && a.ps_mode == AQTX_PRESCALE_NONE && values >= (8 << 20) && a.G > 16 * kAbsRowChunk;
      const bool alone = a.G <= kAbsRowChunk;  // (a block has all rows of its columns)
      folded = a.cols >= 8 && (alone ? blocks <= 512
                                     : a.ws_arrived != nullptr && !bytes_bound && blocks <= (values < (4 << 20) ? 1023 : 512));
      if (a.cols < 8) absmax_cols_kernel<TIn, 1, false><<<grid, 256, 0, st>>>(a);
      else if (folded) absmax_cols_kernel<TIn, 8, true><<<grid, 1024, 0, st>>>(a);
      else absmax_cols_kernel<TIn, 8, false><<<grid, 256, 0, st>>>(a);
      folded |= alone;
      AQTX_HIP_CHECK_LAUNCH("absmax_cols_kernel");
    }
  }
  // (given scales shared by whole columns: the tile kernel takes their reciprocals itself)
  if (a.scale_given ? a.ngroups != 1 : !folded) {
    finalize_scales_kernel<<<dim3((unsigned)((nscales + 255) / 256)), 256, 0, st>>>(a, nscales);
    AQTX_HIP_CHECK_LAUNCH("finalize_scales_kernel");
  }
  }
  if (a.scale_only) return 0;
  const int spec = spec_of(a, partitionable);
  auto grid_for = [&](int pair) {
    const int64_t rows = pair == 1 ? a.rows / 2 : a.rows, cols = pair == 2 ? a.cols / 2 : a.cols;
    return dim3((unsigned)((cols + kTileC - 1) / kTileC), (unsigned)((rows + kTileR - 1) / kTileR),
                (unsigned)a.batch);
  };
  auto low_grid_for = [&](int pair) {
    const int64_t rows = pair == 1 ? a.rows / 2 : a.rows;
    dim3 g = grid_for(pair);
    g.y = (unsigned)((rows + kTileR / 4 - 1) / (kTileR / 4));
    return g;
  };
  // With noise a thread's values are a serial chain of a hundred instructions each, so few tiles are cut to 32 rows, for four
  // times the waves.  Float32 values up to two tall tiles a CU, narrower ones up to eight; where HBM bounds the large ones the
  // short rows of a transposed tile lose.  Calibrated and quantized, tall / low, us:
  //   bf16     64 x 64 14.2 / 7.0, 512 x 1024 14.5 / 8.9, 1024 x 2048 15.4 / 11.0, 2048 x 2048 16.6 / 14.4,
  //            4096 x 4096 36.9 / 35.1, 8192 x 4096 (2048 tiles) 61.0 / 59.4; to fp8 64 x 64 17.8 / 7.4,
  //            2048 x 2048 19.8 / 14.1, 8192 x 4096 57.9 / 53.6, 8192 x 14336 168 / 198
  //   int8     512 x 1024 15.4 / 9.9, 4096 x 4096 38.6 / 37.1, 8192 x 4096 60.9 / 58.8, two entries of it (8192 tiles) 164 / 166
  //   float32  64 x 64 16.4 / 7.4, 1024 x 2048 15.9 / 11.5, 1999 x 3001 32.0 / 28.4, 2048 x 4096 (512 tiles) 27.8 / 27.5, 4096 x 4096 39.9 / 41.0,
  //            8192 x 14336 249 / 296
  auto low = [&](int pair) {
    const dim3 g = grid_for(pair);
    return (int64_t)g.x * g.y * g.z <= (sizeof(TIn) == 4 ? 512 : 2048);
  };
#define AQTX_TILE(SPEC, PAIR, ...) quant_tile_kernel<TIn, SPEC, PAIR, ##__VA_ARGS__><<<grid_for(PAIR), 256, 0, st>>>(a)
#define AQTX_NOISE_TILE(SPEC, PAIR)                                                                        \
  {                                                                                                      \
    if (low(PAIR)) quant_tile_kernel<TIn, SPEC, PAIR, false, 1><<<low_grid_for(PAIR), 256, 0, st>>>(a);  \
    else AQTX_TILE(SPEC, PAIR);                                                                          \
  }
  // pair the two elements of each threefry block: i and i + total/2 lie rows/2 apart when the noise counters are
  // row-major over [rows, cols], cols/2 apart when over [cols, rows]
  auto uniform = [&](auto tag) {
    constexpr int S = decltype(tag)::value;
    const bool natural = a.batch == 1 && a.nsc == 1 && a.nsr == a.cols && (a.rows % 2 == 0);
    const bool transposed = a.batch == 1 && a.nsr == 1 && a.nsc == a.rows && (a.cols % 2 == 0);
    if (natural) AQTX_NOISE_TILE(S, 1)
    else if (transposed) AQTX_NOISE_TILE(S, 2)
    else AQTX_NOISE_TILE(S, 0)
  };
  bool done = false;  // (oa_out: the caller has checked tiles_rowmax_ok: noise none, so spec is 1, 6 or 0)
  if constexpr (sizeof(TIn) != 4) {  // the bf16 pipelines
    done = true;
    if (spec == 1 && a.oa_out != nullptr) {
      AQTX_TILE(1, 0, true);
    } else if (spec == 1) {
      AQTX_TILE(1, 0);
    } else if (spec == 2) {
      uniform(std::integral_constant<int, 2>{});
    } else if (spec == 3) {
      AQTX_TILE(3, 0);
    } else if (spec == 5) {
      // half of a threefry block would be thrown away unless the tile rows/2 further down, whose elements draw
      // from the other half, is quantized by the same workgroup
      const bool natural = a.batch == 1 && a.nsr == a.cols && (a.rows % 2 == 0);
      if (natural) AQTX_NOISE_TILE(5, 1)
      else AQTX_NOISE_TILE(5, 0)
    } else {
      done = false;
    }
  }
  if constexpr (sizeof(TIn) != 2) {  // the float32 ones
    if (!done) {
      done = true;
      if (spec == 6 && a.oa_out != nullptr) AQTX_TILE(6, 0, true);
      else if (spec == 6) AQTX_TILE(6, 0);
      else if (spec == 7) uniform(std::integral_constant<int, 7>{});
      else done = false;
    }
  }
  if (!done) {
    if (a.oa_out != nullptr) AQTX_TILE(0, 0, true);
    else AQTX_TILE(0, 0);
  }
#undef AQTX_NOISE_TILE
#undef AQTX_TILE
  AQTX_HIP_CHECK_LAUNCH("quant_tile_kernel");
  return 0;
}

template <typename TIn>
int dispatch(const QArgs& a, int reduce, int partitionable, int64_t nscales, hipStream_t st) {
  if (reduce == AQTX_REDUCE_COLS) return launch_rows<TIn>(a, partitionable, st);
  return launch_tiles<TIn>(a, reduce, partitionable, nscales, st);
}

}  // namespace
}  // namespace aqtx
