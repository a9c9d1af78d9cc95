// C entry points of the quantize kernels (quantize_core.h), of one-scale dequantization and of the random bits.
#include "quantize_core.h"

namespace aqtx {
namespace {

__global__ void random_bits_kernel(BitGen gen, int64_t n, void* out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t v = gen.draw((uint64_t)i);
  if (gen.width == 16) reinterpret_cast<uint16_t*>(out)[i] = (uint16_t)v;
  else reinterpret_cast<uint32_t*>(out)[i] = v;
}

// out[b, r, c] = cast(q) * scale (aqt_tensor.py:179-183), one thread per element.
template <typename TOut>
__global__ void dequant_kernel(const QArgs a, int fp8_kind) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t per_b = a.rows * a.cols;
  if (i >= a.batch * per_b) return;
  const int64_t b = i / per_b, rc = i % per_b, r = rc / a.cols, c = rc % a.cols;
  const uint8_t* qb = reinterpret_cast<const uint8_t*>(a.x) + b * per_b;
  const uint8_t raw = a.transpose_out ? qb[c * a.rows + r] : qb[rc];
  float v;
  if (fp8_kind == AQTX_E4M3) v = __builtin_amdgcn_cvt_f32_fp8((int)raw, 0);
  else if (fp8_kind == AQTX_E5M2) v = __builtin_amdgcn_cvt_f32_bf8((int)raw, 0);
  else v = (float)(int8_t)raw;
  const float s = a.scale[b * a.ssb + (r / a.G) * a.ssg + (c / a.L) * a.ssc];
  v = rnd(v, a.cbf);
  v = rnd(v * s, a.cbf & a.sbf);
  v = rnd(v, a.cbf);
  if constexpr (sizeof(TOut) == 2) reinterpret_cast<uint16_t*>(a.q)[i] = bf16_bits(v);
  else reinterpret_cast<float*>(a.q)[i] = v;
}

// ---- host side ---------------------------------------------------------------------

int validate(const aqtx_quant_plan* p) {
  AQTX_REQUIRE(p != nullptr, "aqtx_quantize: plan is NULL");
  AQTX_REQUIRE(p->in_dtype == AQTX_F32 || p->in_dtype == AQTX_BF16 || p->in_dtype == AQTX_I8,
               "aqtx_quantize: unsupported in_dtype %d", p->in_dtype);
  AQTX_REQUIRE(is_float_dtype(p->compute_dtype),
               "aqtx_quantize: compute_dtype must be f32 or bf16, got %d", p->compute_dtype);
  AQTX_REQUIRE(p->in_dtype == AQTX_I8 || p->in_dtype == p->compute_dtype,
               "aqtx_quantize: float input must be held in compute_dtype (in %d, compute %d)",
               p->in_dtype, p->compute_dtype);
  AQTX_REQUIRE(is_float_dtype(p->scale_dtype),
               "aqtx_quantize: scale_dtype must be f32 or bf16, got %d", p->scale_dtype);
  AQTX_REQUIRE(p->out_dtype == AQTX_I8 || p->out_dtype == AQTX_I4 || p->out_dtype == AQTX_E4M3 ||
                   p->out_dtype == AQTX_E5M2,
               "aqtx_quantize: unsupported out_dtype %d", p->out_dtype);
  AQTX_REQUIRE(p->batch >= 0 && p->rows >= 0 && p->cols >= 0, "aqtx_quantize: negative shape");
  AQTX_REQUIRE(p->reduce >= AQTX_REDUCE_COLS && p->reduce <= AQTX_REDUCE_ALL_BATCH,
               "aqtx_quantize: unknown reduce mode %d", p->reduce);
  AQTX_REQUIRE(p->group >= 0, "aqtx_quantize: negative group");
  if (p->group > 0) {
    AQTX_REQUIRE(p->reduce == AQTX_REDUCE_COLS || p->reduce == AQTX_REDUCE_ROWS,
                 "aqtx_quantize: group needs REDUCE_COLS or REDUCE_ROWS");
    const int64_t axis = p->reduce == AQTX_REDUCE_COLS ? p->cols : p->rows;
    AQTX_REQUIRE(axis % p->group == 0,
                 "aqtx_quantize: group %lld does not divide the reduced axis %lld",
                 (long long)p->group, (long long)axis);
  }
  AQTX_REQUIRE(!(p->transpose_out && p->reduce == AQTX_REDUCE_COLS),
               "aqtx_quantize: transpose_out is not supported with REDUCE_COLS");
  AQTX_REQUIRE(p->noise >= AQTX_NOISE_NONE && p->noise <= AQTX_NOISE_FP8_MANTISSA,
               "aqtx_quantize: unknown noise kind %d", p->noise);
  const bool fp8 = p->out_dtype == AQTX_E4M3 || p->out_dtype == AQTX_E5M2;
  AQTX_REQUIRE(!(p->noise == AQTX_NOISE_FP8_MANTISSA && !fp8),
               "aqtx_quantize: mantissa noise needs an fp8 out_dtype");
  AQTX_REQUIRE(!((p->noise == AQTX_NOISE_JAX_UNIFORM || p->noise == AQTX_NOISE_CUSTOM1) && fp8),
               "aqtx_quantize: additive noise needs an integer out_dtype");
  if (p->noise != AQTX_NOISE_NONE) {
    AQTX_REQUIRE(p->noise_total > 0 && p->noise_total < (int64_t)0xFFFFFFFFll,
                 "aqtx_quantize: noise_total %lld out of range (1 .. 2^32-2)",
                 (long long)p->noise_total);
  }
  AQTX_REQUIRE(p->prescale >= AQTX_PRESCALE_NONE && p->prescale <= AQTX_PRESCALE_PER_COL,
               "aqtx_quantize: unknown prescale mode %d", p->prescale);
  AQTX_REQUIRE(p->quant_bound > 0.0f && p->clip_bound > 0.0f,
               "aqtx_quantize: bounds must be positive");
  return 0;
}

int64_t scale_count(const aqtx_quant_plan* p) {
  switch (p->reduce) {
    case AQTX_REDUCE_COLS: return p->batch * p->rows * (p->group ? p->cols / p->group : 1);
    case AQTX_REDUCE_ROWS: return p->batch * (p->group ? p->rows / p->group : 1) * p->cols;
    case AQTX_REDUCE_ALL: return p->batch;
    default: return 1;
  }
}

int noise_width(const aqtx_quant_plan* p) {
  if (p->noise == AQTX_NOISE_CUSTOM1) return 16;
  if (p->noise == AQTX_NOISE_FP8_MANTISSA)
    return (p->compute_dtype == AQTX_BF16 && p->scale_dtype == AQTX_BF16) ? 16 : 32;
  return 32;
}

// Whether the row kernels can leave column maxima of |q| behind for this plan: whole rows of 520 to 8192
// aligned values as segments, one batch entry, integer values rounded to nearest.
bool rows_colmax_ok(const aqtx_quant_plan* p) {
  return p->reduce == AQTX_REDUCE_COLS && p->batch == 1 && p->group == 0 && !p->transpose_out &&
         p->noise == AQTX_NOISE_NONE && (p->out_dtype == AQTX_I8 || p->out_dtype == AQTX_I4) &&
         p->out_k_order == AQTX_K_NATURAL && p->cols % 8 == 0 && p->cols > 512 && p->cols <= 8192 && p->rows > 0;
}

// Whether the tile kernel can leave row maxima of |q| behind for this plan: one scale per column over whole
// columns, every 128 x 64 tile inside the tensor, one batch entry, integer values rounded to nearest.
bool tiles_rowmax_ok(const aqtx_quant_plan* p) {
  return p->reduce == AQTX_REDUCE_ROWS && p->batch == 1 && p->group == 0 && p->noise == AQTX_NOISE_NONE &&
         (p->out_dtype == AQTX_I8 || p->out_dtype == AQTX_I4) && p->rows > 0 && p->cols > 0 &&
         p->rows % kTileR == 0 && p->cols % kTileC == 0;
}

// Threads a row (as a shift) with which the columns of this plan are calibrated and quantized in one pass, or -1: new scales
// of whole columns, transposed output, the compile-time integer pipelines without noise or prescale, and a size that cols_once_shift takes.
int once_shift_of(const aqtx_quant_plan* p, bool row_maxima) {
  if (p->reduce != AQTX_REDUCE_ROWS || !p->transpose_out || (p->group != 0 && p->group != p->rows) || p->scale_given || p->noise != AQTX_NOISE_NONE ||
      p->prescale != AQTX_PRESCALE_NONE || p->compute_dtype != p->in_dtype || p->scale_dtype != p->in_dtype)
    return -1;
  if ((p->in_dtype != AQTX_BF16 && p->in_dtype != AQTX_F32) || (p->out_dtype != AQTX_I8 && p->out_dtype != AQTX_I4)) return -1;
  return cols_once_shift(p->in_dtype == AQTX_BF16 ? 2 : 4, p->batch, p->rows, p->cols, row_maxima);
}

}  // namespace
}  // namespace aqtx

using namespace aqtx;

// A few very long rows (one scale per image of a convolution's input, say) would leave most of
// the chip idle in the row kernels, which give a row to one wave or workgroup.  Such a plan is the
// same computation as one scale per batch entry of [batch * rows][cols / c][c]: the whole-tensor
// path, which spreads every entry over many workgroups.  Returns true and fills `q` if `p` is
// such a plan.
static bool long_rows_as_batches(const aqtx_quant_plan* p, aqtx_quant_plan* q) {
  if (p->reduce != AQTX_REDUCE_COLS || p->group != 0 || p->transpose_out || p->prescale != AQTX_PRESCALE_NONE ||
      p->out_k_order != AQTX_K_NATURAL)
    return false;
  if (p->batch <= 0 || p->rows <= 0 || p->batch * p->rows > 512 || p->cols < 16384) return false;
  if (p->noise != AQTX_NOISE_NONE && p->batch > 1 && p->noise_stride_batch != p->rows * p->noise_stride_row)
    return false;
  int64_t c = 0;
  for (int64_t cand = 1024; cand >= 64; cand /= 2) {
    if (p->cols % cand == 0) { c = cand; break; }
  }
  if (c == 0) return false;
  *q = *p;
  q->batch = p->batch * p->rows;
  q->rows = p->cols / c;
  q->cols = c;
  q->reduce = AQTX_REDUCE_ALL;
  q->noise_stride_batch = p->noise_stride_row;
  q->noise_stride_row = c * p->noise_stride_col;
  return true;
}

extern "C" int64_t aqtx_quantize_other_axis_parts(const aqtx_quant_plan* p) {
  aqtx_quant_plan alt;
  if (p == nullptr || p->scale_given || long_rows_as_batches(p, &alt)) return 0;
  if (rows_colmax_ok(p)) return p->rows < kColmaxBlocks ? p->rows : kColmaxBlocks;
  if (tiles_rowmax_ok(p)) return p->cols / kTileC;
  return 0;
}

extern "C" size_t aqtx_quantize_workspace_bytes(const aqtx_quant_plan* p) {
  aqtx_quant_plan alt;
  if (p != nullptr && long_rows_as_batches(p, &alt)) return aqtx_quantize_workspace_bytes(&alt);
  if (p == nullptr || p->reduce == AQTX_REDUCE_COLS) return 0;
  if (p->batch < 0 || p->rows < 0 || p->cols < 0 || p->group < 0) return 0;
  if (p->reduce < AQTX_REDUCE_ROWS || p->reduce > AQTX_REDUCE_ALL_BATCH) return 0;
  if (p->group > 0 && (p->reduce != AQTX_REDUCE_ROWS || p->rows % p->group != 0)) return 0;
  return (size_t)scale_count(p) * 8;
}

// scale_only: q is neither read nor written (aqtx_calibrate).  given_bf16: the given scales (aqtx_quantize_given).
static int quantize_impl(const aqtx_quant_plan* p, const void* x, const float* prescale, void* q, float* scale, bool scale_only,
                         const uint16_t* given_bf16, void* workspace, size_t workspace_bytes, void* stream) {
  if (int rc = validate(p)) return rc;
  aqtx_quant_plan alt;
  if (long_rows_as_batches(p, &alt))
    return quantize_impl(&alt, x, prescale, q, scale, scale_only, given_bf16, workspace, workspace_bytes, stream);
  const int64_t total = p->batch * p->rows * p->cols;
  if (total == 0) return 0;
  AQTX_REQUIRE(x != nullptr && (q != nullptr || scale_only) && (scale != nullptr || given_bf16 != nullptr),
               "aqtx_quantize: NULL buffer");
  AQTX_REQUIRE(!scale_only || (p->noise == AQTX_NOISE_NONE && !p->scale_given && p->other_axis_absmax == nullptr),
               "aqtx_calibrate (scale_only) goes without noise, a given scale and other_axis_absmax");
  AQTX_REQUIRE((p->prescale == AQTX_PRESCALE_NONE) == (prescale == nullptr),
               "aqtx_quantize: prescale pointer does not match plan->prescale");
  AQTX_REQUIRE(p->batch <= 65535, "aqtx_quantize: batch %lld exceeds 65535", (long long)p->batch);
  const size_t need = aqtx_quantize_workspace_bytes(p);
  AQTX_REQUIRE(workspace_bytes >= need && (need == 0 || workspace != nullptr),
               "aqtx_quantize: workspace too small (%zu < %zu)", workspace_bytes, need);
  AQTX_REQUIRE(((uintptr_t)x % 16) == 0 && ((uintptr_t)q % 16) == 0 &&
                   ((uintptr_t)scale % 4) == 0 &&
                   (prescale == nullptr || ((uintptr_t)prescale % 16) == 0) &&
                   (workspace == nullptr || ((uintptr_t)workspace % 4) == 0),
               "aqtx_quantize: x, q and prescale must be 16-byte aligned");

  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int64_t nscales = scale_count(p);
  QArgs a{};
  a.x = x; a.prescale = prescale; a.q = q; a.scale = scale;
  a.scale_bf16 = (p->scale_typed != nullptr && p->scale_dtype == AQTX_BF16 && !p->scale_given)
                     ? reinterpret_cast<uint16_t*>(p->scale_typed) : nullptr;
  a.scale_only = scale_only;
  a.given_bf16 = given_bf16;
  a.batch = p->batch; a.rows = p->rows; a.cols = p->cols;
  a.nsb = p->noise_stride_batch; a.nsr = p->noise_stride_row; a.nsc = p->noise_stride_col;
  a.quant_bound = p->quant_bound; a.clip_bound = p->clip_bound;
  a.noise = p->noise; a.ps_mode = p->prescale; a.psb = p->prescale_stride_batch;
  a.transpose_out = p->transpose_out; a.out_dtype = p->out_dtype;
  a.cbf = p->compute_dtype == AQTX_BF16; a.sbf = p->scale_dtype == AQTX_BF16;
  a.scale_given = p->scale_given;
  a.ws_zeroed = p->workspace_zeroed;
  a.once_shift = scale_only ? -1 : once_shift_of(p, p->other_axis_absmax != nullptr);
  if (p->other_axis_absmax != nullptr) {
    AQTX_REQUIRE(aqtx_quantize_other_axis_parts(p) > 0,
                 "aqtx_quantize: this plan cannot write other_axis_absmax (aqtx_quantize_other_axis_parts is 0)");
    AQTX_REQUIRE(((uintptr_t)p->other_axis_absmax % 8) == 0, "aqtx_quantize: other_axis_absmax must be 8-byte aligned");
    a.oa_out = reinterpret_cast<uint8_t*>(p->other_axis_absmax);
  }
  if (p->absmax_partials != nullptr) {
    AQTX_REQUIRE(p->in_dtype == AQTX_I8 && p->reduce == AQTX_REDUCE_ROWS && p->group == 0 && p->batch == 1 &&
                     !p->scale_given && p->prescale == AQTX_PRESCALE_NONE && p->absmax_parts > 0 && p->cols % 16 == 0 &&
                     ((uintptr_t)p->absmax_partials % 16) == 0,
                 "aqtx_quantize: absmax_partials (16-byte aligned) go with int8 input, AQTX_REDUCE_ROWS over whole columns (a "
                 "multiple of 16 of them), one batch entry, no prescale and no given scale");
    a.oa_in = reinterpret_cast<const uint8_t*>(p->absmax_partials);
    a.oa_in_parts = p->absmax_parts;
  }
  AQTX_REQUIRE(p->out_k_order == AQTX_K_NATURAL || p->out_k_order == AQTX_K_EVEN_ODD8,
               "aqtx_quantize: unknown out_k_order %d", p->out_k_order);
  if (p->out_k_order == AQTX_K_EVEN_ODD8) {
    AQTX_REQUIRE(p->reduce == AQTX_REDUCE_COLS && !p->transpose_out &&
                     (p->out_dtype == AQTX_I8 || p->out_dtype == AQTX_I4),
                 "aqtx_quantize: out_k_order = EVEN_ODD8 needs AQTX_REDUCE_COLS, an integer out_dtype and no transpose_out");
    a.even_odd8 = 1;
  }
  if (p->noise != AQTX_NOISE_NONE) {
    a.gen = make_bitgen(p->key, p->noise_total, noise_width(p), p->partitionable);
    a.key_dev = p->key_device;
    AQTX_REQUIRE(((uintptr_t)p->key_device % 4) == 0, "aqtx_quantize: key_device is not 4-byte aligned");
  }
  if (p->reduce == AQTX_REDUCE_COLS) {
    a.L = p->group ? p->group : p->cols;
    a.nseg = nscales;
  } else {
    a.ws_absmax = reinterpret_cast<uint32_t*>(workspace);
    // A workspace kept across calls holds the abs-max words (zero between calls) in its first
    // half and the reciprocal scales in its second, whatever the number of scales of a call.
    a.ws_inv = reinterpret_cast<float*>(workspace) +
               (p->workspace_zeroed ? (int64_t)(workspace_bytes / 8) : nscales);
    if (p->reduce == AQTX_REDUCE_ROWS) {
      a.G = p->group ? p->group : p->rows;
      a.ngroups = p->rows / a.G;
      a.ssb = a.ngroups * p->cols; a.ssg = p->cols; a.ssc = 1;
    } else {
      a.G = p->rows; a.ngroups = 1;
      a.ssb = p->reduce == AQTX_REDUCE_ALL ? 1 : 0; a.ssg = 0; a.ssc = 0;
    }
    // Room behind the abs-max words of a kept workspace (zero like them): the arrival counts of the abs-max blocks, one per
    // set of scales that they share: a column group of its blocks, a batch entry, or the whole batch
    const int64_t groups = p->reduce == AQTX_REDUCE_ROWS  ? p->batch * a.ngroups * absmax_col_groups(p->cols)
                           : p->reduce == AQTX_REDUCE_ALL ? p->batch
                                                          : 1;
    if (p->workspace_zeroed && (int64_t)(workspace_bytes / 8) >= nscales + groups) a.ws_arrived = a.ws_absmax + (workspace_bytes / 8) - groups;
    const int64_t grid_y = p->reduce != AQTX_REDUCE_ROWS
                               ? (p->rows + kTileR - 1) / kTileR
                               : a.ngroups * ((a.G + kAbsRowChunk - 1) / kAbsRowChunk);
    AQTX_REQUIRE(grid_y <= 65535 && (p->rows + kTileR - 1) / kTileR <= 65535,
                 "aqtx_quantize: too many rows for one launch (%lld)", (long long)p->rows);
  }
  switch (p->in_dtype) {
    case AQTX_F32: return launch_quantize_f32(a, p->reduce, p->partitionable, nscales, st);
    case AQTX_BF16: return launch_quantize_bf16(a, p->reduce, p->partitionable, nscales, st);
    default: return launch_quantize_i8(a, p->reduce, p->partitionable, nscales, st);
  }
}

extern "C" int aqtx_quantize(const aqtx_quant_plan* p, const void* x, const float* prescale,
                             void* q, float* scale, void* workspace, size_t workspace_bytes,
                             void* stream) {
  clear_error();
  return quantize_impl(p, x, prescale, q, scale, false, nullptr, workspace, workspace_bytes, stream);
}

extern "C" int aqtx_quantize_given(const aqtx_quant_plan* p, const void* x, const float* prescale, void* q,
                                   const void* scale, void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  AQTX_REQUIRE(p != nullptr && p->scale_given, "aqtx_quantize_given: plan is NULL or has no scale_given");
  if (p->scale_dtype != AQTX_BF16)
    return quantize_impl(p, x, prescale, q, reinterpret_cast<float*>(const_cast<void*>(scale)), false, nullptr, workspace,
                         workspace_bytes, stream);
  AQTX_REQUIRE(((uintptr_t)scale % 2) == 0, "aqtx_quantize_given: scale is not element aligned");
  return quantize_impl(p, x, prescale, q, nullptr, false, reinterpret_cast<const uint16_t*>(scale), workspace, workspace_bytes,
                       stream);
}

extern "C" int aqtx_calibrate(const aqtx_quant_plan* p, const void* x, const float* prescale, float* scale, void* workspace,
                              size_t workspace_bytes, void* stream) {
  clear_error();
  return quantize_impl(p, x, prescale, nullptr, scale, true, nullptr, workspace, workspace_bytes, stream);
}

extern "C" int aqtx_dequantize(const aqtx_quant_plan* p, const void* q, const float* scale,
                               void* out, void* stream) {
  clear_error();
  if (int rc = validate(p)) return rc;
  AQTX_REQUIRE(p->in_dtype != AQTX_I8, "aqtx_dequantize: in_dtype names the float result dtype");
  const int64_t total = p->batch * p->rows * p->cols;
  if (total == 0) return 0;
  AQTX_REQUIRE(q != nullptr && scale != nullptr && out != nullptr, "aqtx_dequantize: NULL buffer");
  if (!p->transpose_out && p->group == 0) {
    // q in the order of the result and one scale per row, per column or per (batch) tensor: the
    // 16-columns-per-lane kernel of aqtx_scale_cast, same arithmetic
    aqtx_scale_plan sp{};
    sp.in_dtype = p->out_dtype; sp.out_dtype = p->in_dtype;
    sp.batch = p->batch; sp.rows = p->rows; sp.cols = p->cols;
    sp.factors = 1; sp.factor_dtype[0] = p->scale_dtype;
    if (p->reduce == AQTX_REDUCE_COLS) {
      sp.factor_axis[0] = AQTX_FACTOR_ROWS; sp.factor_stride_b[0] = p->rows;
    } else if (p->reduce == AQTX_REDUCE_ROWS) {
      sp.factor_axis[0] = AQTX_FACTOR_COLS; sp.factor_stride_b[0] = p->cols;
    } else {
      sp.rows = 1; sp.cols = p->rows * p->cols;
      sp.factor_axis[0] = AQTX_FACTOR_ROWS; sp.factor_stride_b[0] = p->reduce == AQTX_REDUCE_ALL ? 1 : 0;
    }
    return aqtx_scale_cast(&sp, q, scale, nullptr, out, stream);
  }
  QArgs a{};
  a.x = q; a.q = out; a.scale = const_cast<float*>(scale);
  a.batch = p->batch; a.rows = p->rows; a.cols = p->cols;
  a.transpose_out = p->transpose_out;
  a.cbf = p->in_dtype == AQTX_BF16; a.sbf = p->scale_dtype == AQTX_BF16;
  // scale index = b*ssb + (r/G)*ssg + (c/L)*ssc
  if (p->reduce == AQTX_REDUCE_COLS) {
    a.L = p->group ? p->group : p->cols; a.G = 1;
    const int64_t per_row = p->cols / a.L;
    a.ssb = p->rows * per_row; a.ssg = per_row; a.ssc = 1;
  } else if (p->reduce == AQTX_REDUCE_ROWS) {
    a.G = p->group ? p->group : p->rows; a.L = 1;
    a.ssb = (p->rows / a.G) * p->cols; a.ssg = p->cols; a.ssc = 1;
  } else {
    a.G = p->rows; a.L = p->cols; a.ssb = p->reduce == AQTX_REDUCE_ALL ? 1 : 0; a.ssg = 0; a.ssc = 0;
  }
  const int fp8_kind = (p->out_dtype == AQTX_E4M3 || p->out_dtype == AQTX_E5M2) ? p->out_dtype : 0;
  const unsigned blocks = (unsigned)((total + 255) / 256);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (p->in_dtype == AQTX_BF16) dequant_kernel<uint16_t><<<dim3(blocks), 256, 0, st>>>(a, fp8_kind);
  else dequant_kernel<float><<<dim3(blocks), 256, 0, st>>>(a, fp8_kind);
  AQTX_HIP_CHECK_LAUNCH("dequant_kernel");
  return 0;
}

extern "C" int aqtx_random_bits(const uint32_t key_host[2], int64_t n, int32_t bit_width,
                                int32_t partitionable, void* out, void* stream) {
  clear_error();
  AQTX_REQUIRE(key_host != nullptr, "aqtx_random_bits: key is NULL");
  AQTX_REQUIRE(bit_width == 16 || bit_width == 32, "aqtx_random_bits: bit_width must be 16 or 32");
  AQTX_REQUIRE(n >= 0 && n < (int64_t)0xFFFFFFFFll, "aqtx_random_bits: n out of range");
  if (n == 0) return 0;
  AQTX_REQUIRE(out != nullptr, "aqtx_random_bits: out is NULL");
  BitGen gen = make_bitgen(key_host, n, bit_width, partitionable);
  random_bits_kernel<<<dim3((unsigned)((n + 255) / 256)), 256, 0,
                       reinterpret_cast<hipStream_t>(stream)>>>(gen, n, out);
  AQTX_HIP_CHECK_LAUNCH("random_bits_kernel");
  return 0;
}

namespace aqtx {
namespace {
// word i of the 2 * num words of jax.random.split(key, num)
AQTX_HD uint32_t split_word(uint32_t k0, uint32_t k1, uint32_t num, int partitionable, uint32_t i) {
  if (partitionable) {
    const U2 b = threefry2x32(k0, k1, 0u, i >> 1);
    return (i & 1) ? b.y : b.x;
  }
  BitGen g;
  g.k0 = k0; g.k1 = k1;
  g.nwords = 2u * num; g.half = num;
  g.partitionable = 0; g.width = 32;
  return g.word_original(i);
}

// word i of the keys of split(split(key, num)[p], inner), p = 0 .. num - 1; inner 0: of split(key, num)
AQTX_HD uint32_t split2_word(uint32_t k0, uint32_t k1, uint32_t num, uint32_t inner, int partitionable, uint32_t i) {
  if (inner == 0) return split_word(k0, k1, num, partitionable, i);
  const uint32_t p = i / (2 * inner);
  const uint32_t c0 = split_word(k0, k1, num, partitionable, 2 * p), c1 = split_word(k0, k1, num, partitionable, 2 * p + 1);
  return split_word(c0, c1, inner, partitionable, i % (2 * inner));
}

// Bound by its launch: the whole fan-out of a step's key (one split and a split of each part) in one instead of four,
// which spares a recorded step 4 us a launch.
__global__ __launch_bounds__(256) void prng_split_kernel(const uint32_t* __restrict__ key, int num, int inner, int partitionable,
                                                         uint32_t* __restrict__ out) {
  const int i = (int)(blockIdx.x * 256 + threadIdx.x);
  if (i >= 2 * num * (inner > 0 ? inner : 1)) return;
  out[i] = split2_word(key[0], key[1], (uint32_t)num, (uint32_t)inner, partitionable, (uint32_t)i);
}
}  // namespace
}  // namespace aqtx

extern "C" int aqtx_prng_split2(const uint32_t* key_device, int32_t num, int32_t inner, int32_t partitionable,
                                uint32_t* out_device, void* stream) {
  clear_error();
  AQTX_REQUIRE(num >= 0 && num <= (1 << 20) && inner >= 0 && (int64_t)num * inner <= (1 << 20),
               "aqtx_prng_split: num or num * inner outside 0..2^20");
  if (num == 0) return 0;
  AQTX_REQUIRE(key_device != nullptr && out_device != nullptr, "aqtx_prng_split: NULL argument");
  const int words = 2 * num * (inner > 0 ? inner : 1);
  prng_split_kernel<<<(unsigned)((words + 255) / 256), 256, 0, reinterpret_cast<hipStream_t>(stream)>>>(
      key_device, num, inner, partitionable, out_device);
  AQTX_HIP_CHECK_LAUNCH("prng_split_kernel");
  return 0;
}

extern "C" int aqtx_prng_split(const uint32_t* key_device, int32_t num, int32_t partitionable, uint32_t* out_device,
                               void* stream) {
  return aqtx_prng_split2(key_device, num, 0, partitionable, out_device, stream);
}

extern "C" int aqtx_prng_split2_host(const uint32_t key_host[2], int32_t num, int32_t inner, int32_t partitionable,
                                     uint32_t* out_host) {
  clear_error();
  AQTX_REQUIRE(key_host != nullptr && out_host != nullptr, "aqtx_prng_split_host: NULL argument");
  AQTX_REQUIRE(num >= 0 && inner >= 0, "aqtx_prng_split_host: negative num");
  const int64_t words = 2 * (int64_t)num * (inner > 0 ? inner : 1);
  AQTX_REQUIRE(words < (1ll << 31), "aqtx_prng_split_host: too many keys");
  for (int64_t i = 0; i < words; ++i)
    out_host[i] = split2_word(key_host[0], key_host[1], (uint32_t)num, (uint32_t)inner, partitionable, (uint32_t)i);
  return 0;
}

extern "C" int aqtx_prng_split_host(const uint32_t key_host[2], int32_t num, int32_t partitionable, uint32_t* out_host) {
  return aqtx_prng_split2_host(key_host, num, 0, partitionable, out_host);
}
