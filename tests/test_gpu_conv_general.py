"""Quantized conv_general_dilated: oracle pins (CPU) and GPU parity, after aqt_conv_general_test.py."""
import functools

import numpy as np
import pytest
import torch

from oracle import aqt_ref as R
from oracle import numerics as nm
from tests import gpu_util as U

BITS = [(1, 1), (1, 2), (2, 1), (2, 2), (8, 8), (None, 8), (8, None), (None, None)]  # aqt_conv_general_test.py:53-62


def _rand_unif(shape, maxval, seed, dt='f32'):
  """aqt_conv_general_test.py:26-30."""
  rng = np.random.default_rng(seed)
  return nm.cast(rng.uniform(-maxval, maxval, shape).astype(np.float32), dt)


def _qcfg(bits, po2=True):
  # dot_general_raw_make (aqt_dot_general.py:99-156): one bit cannot hold zero, so the value
  # stays in the float dtype
  if bits is None:
    return R.QuantizerCfg(bits=None)
  return R.QuantizerCfg(bits=bits, po2_scale=po2, preserve_zero=bits != 1, keep_float=bits == 1)


def test_oracle_conv_matches_scipy_correlate():
  """The float convolution behind the oracle against scipy's n-d correlation: SAME and VALID,
  strides and kernel dilation (a dilated kernel is the kernel with zeros inserted)."""
  from scipy.signal import correlate
  rng = np.random.default_rng(0)
  lhs = rng.standard_normal((2, 7, 6, 3))
  rhs = rng.standard_normal((3, 2, 3, 4))

  def full(x, w, pads):
    xp = np.pad(x, [(0, 0)] + pads + [(0, 0)])
    out = np.zeros((x.shape[0], xp.shape[1] - w.shape[0] + 1, xp.shape[2] - w.shape[1] + 1, w.shape[-1]))
    for n in range(x.shape[0]):
      for o in range(w.shape[-1]):
        out[n, :, :, o] = sum(correlate(xp[n, :, :, c], w[:, :, c, o], mode='valid') for c in range(x.shape[-1]))
    return out

  np.testing.assert_allclose(R.lax_conv_nhwc(lhs, rhs, (1, 1), 'VALID'), full(lhs, rhs, [(0, 0), (0, 0)]), atol=1e-12)
  # SAME with an even kernel extent pads the extra element at the high end
  np.testing.assert_allclose(R.lax_conv_nhwc(lhs, rhs, (1, 1), 'SAME'), full(lhs, rhs, [(1, 1), (0, 1)]), atol=1e-12)
  np.testing.assert_allclose(R.lax_conv_nhwc(lhs, rhs, (2, 3), 'VALID'), full(lhs, rhs, [(0, 0), (0, 0)])[:, ::2, ::3],
                             atol=1e-12)
  np.testing.assert_allclose(R.lax_conv_nhwc(lhs, rhs, (1, 1), [(2, 1), (0, 3)]), full(lhs, rhs, [(2, 1), (0, 3)]),
                             atol=1e-12)
  dil = np.zeros((5, 4, 3, 4))
  dil[::2, ::3] = rhs
  np.testing.assert_allclose(R.lax_conv_nhwc(lhs, rhs, (1, 1), 'VALID', (2, 3)), full(lhs, dil, [(0, 0), (0, 0)]),
                             atol=1e-12)
  # SAME with stride 2 on 7 rows: 4 output rows, total padding (4-1)*2+3-7 = 2
  got = R.lax_conv_nhwc(lhs, rhs, (2, 1), 'SAME')
  np.testing.assert_allclose(got, full(lhs, rhs, [(1, 1), (0, 1)])[:, ::2], atol=1e-12)


@pytest.mark.parametrize('lhs_bits,rhs_bits', BITS)
def test_oracle_conv_equals_conv_of_fake_quantized(lhs_bits, rhs_bits):
  """aqt_conv_general_test.py:63-103: with power-of-two scales the quantized convolution is
  exactly the float convolution of the fake-quantized operands."""
  lhs = _rand_unif((10, 4, 5, 20), 10.0, 0)
  rhs = _rand_unif((3, 3, 20, 30), 20.0, 1)
  raw = R.RawCfg(_qcfg(lhs_bits), _qcfg(rhs_bits))
  out, lqt, rqt = R.conv_general_dilated_fwd(lhs, rhs, 'f32', (1, 1), 'SAME', raw)
  if lhs_bits is not None:
    assert lqt.scale[0].shape == (10, 1, 1, 1)
  if rhs_bits is not None:
    assert rqt.scale[0].shape == (1, 1, 1, 30)
  fq = R.lax_conv_nhwc(R.dequant(lqt), R.dequant(rqt), (1, 1), 'SAME').astype(np.float32)
  if lhs_bits is None or rhs_bits is None:
    # the unquantized side makes the float sums inexact; only their order differs here
    np.testing.assert_allclose(out, fq, rtol=2e-6, atol=1e-3)
  else:
    np.testing.assert_array_equal(out, fq)


def _make(lhs_bits, rhs_bits, po2=True):
  """aqt_conv_general_test.py:33-84: conv_general_dilated_make with power-of-two scales."""
  from aqt_amd.v2 import aqt_conv_general as aqt_conv
  raw = aqt_conv.conv_general_dilated_make(2, lhs_bits, rhs_bits, initialize_calibration=False)
  for present, q in ((raw.lhs, raw.dg_quantizer.lhs), (raw.rhs, raw.dg_quantizer.rhs)):
    if present:
      if po2 and q.calibration is not None:
        q.calibration = functools.partial(q.calibration, po2_scale=True)
      q.init_calibration()
  return raw


@pytest.mark.gpu
@pytest.mark.parametrize('lhs_bits,rhs_bits', BITS)
def test_conv_general_dilated(gpu, lhs_bits, rhs_bits):
  """aqt_conv_general_test.py:63-103, and the same numbers as the oracle."""
  from aqt_amd.v2 import aqt_conv_general as aqt_conv
  from aqt_amd.v2 import aqt_quantizer
  raw = _make(lhs_bits, rhs_bits)
  lhs_np = _rand_unif((10, 4, 5, 20), 10.0, 0)
  rhs_np = _rand_unif((3, 3, 20, 30), 20.0, 1)
  lhs, rhs = U.to_dev(lhs_np, 'f32', gpu), U.to_dev(rhs_np, 'f32', gpu)
  kwargs = dict(window_strides=(1, 1), padding='SAME',
                dimension_numbers=aqt_conv.flax_conv_dimension_numbers(lhs.shape))
  lhs_fq = aqt_quantizer.make_fake_quant(raw.dg_quantizer.lhs)(lhs)
  rhs_fq = aqt_quantizer.make_fake_quant(raw.dg_quantizer.rhs)(rhs)
  prod_fq = aqt_conv.lax_conv_general_dilated(lhs_fq, rhs_fq, **kwargs)
  prod_aqt = aqt_conv.make_conv_general_dilated(raw)(lhs, rhs, **kwargs)
  assert prod_aqt.shape == (10, 4, 5, 30) and prod_aqt.dtype == torch.float32
  assert (prod_aqt == prod_fq).all()
  want, _, _ = R.conv_general_dilated_fwd(lhs_np, rhs_np, 'f32', (1, 1), 'SAME',
                                          R.RawCfg(_qcfg(lhs_bits), _qcfg(rhs_bits)))
  if lhs_bits is None or rhs_bits is None:
    np.testing.assert_allclose(prod_aqt.cpu().numpy(), want, rtol=2e-6, atol=1e-3)
  else:
    np.testing.assert_array_equal(prod_aqt.cpu().numpy(), want)


@pytest.mark.gpu
@pytest.mark.parametrize('lhs_bits,rhs_bits', BITS)
def test_conv_general_dilated_quantized(gpu, lhs_bits, rhs_bits):
  """aqt_conv_general_test.py:105-163: operands handed over as QTensors give the same result."""
  from aqt_amd.v2 import aqt_conv_general as aqt_conv
  raw = _make(lhs_bits, rhs_bits)
  lhs = U.to_dev(_rand_unif((10, 4, 5, 20), 10.0, 0), 'f32', gpu)
  rhs = U.to_dev(_rand_unif((3, 3, 20, 30), 20.0, 1), 'f32', gpu)
  fn = aqt_conv.make_conv_general_dilated_with_qt(raw)
  kwargs = dict(window_strides=(1, 1), padding='SAME',
                dimension_numbers=aqt_conv.flax_conv_dimension_numbers(lhs.shape))
  lhs_q, _ = raw.dg_quantizer.lhs.quant(lhs, calibration_axes=[0, 1, 2, 3])
  rhs_q, _ = raw.dg_quantizer.rhs.quant(rhs, calibration_axes=[0, 1, 2])
  out_no_quant, (lqt, rqt) = fn(lhs, rhs, lhs_qt=None, rhs_qt=None, **kwargs)
  out_lhs_quant, _ = fn(torch.zeros_like(lhs), rhs, lhs_qt=lhs_q, rhs_qt=None, **kwargs)
  out_rhs_quant, _ = fn(lhs, torch.zeros_like(rhs), lhs_qt=None, rhs_qt=rhs_q, **kwargs)
  out_both_quant, _ = fn(torch.zeros_like(lhs), torch.zeros_like(rhs), lhs_qt=lhs_q, rhs_qt=rhs_q, **kwargs)
  assert (out_no_quant == out_lhs_quant).all()
  assert (out_no_quant == out_rhs_quant).all()
  assert (out_no_quant == out_both_quant).all()
  if lhs_bits is not None:
    assert tuple(lqt.scale[0].shape) == (10, 1, 1, 1)
  if rhs_bits is not None:
    assert tuple(rqt.scale[0].shape) == (1, 1, 1, 30)


@pytest.mark.gpu
@pytest.mark.parametrize('dt', ['f32', 'bf16'])
@pytest.mark.parametrize('case', [
    dict(lhs=(3, 9, 8, 16), rhs=(3, 3, 16, 24), strides=(2, 1), padding='SAME'),
    dict(lhs=(2, 12, 11, 32), rhs=(2, 3, 32, 40), strides=(1, 2), padding='VALID', dil=(2, 1)),
    dict(lhs=(4, 33, 48), rhs=(5, 48, 64), strides=(3,), padding=[(2, 1)]),
    dict(lhs=(2, 5, 6, 4, 16), rhs=(2, 2, 2, 16, 8), strides=(1, 1, 2), padding='SAME'),
    dict(lhs=(1, 8, 8, 64), rhs=(1, 1, 64, 128), strides=(1, 1), padding='VALID'),
])
def test_conv_strides_padding_dilation_rank_match_oracle(gpu, case, dt):
  """int8 x int8 with ordinary (not power-of-two) abs-max scales: 1-d, 2-d and 3-d windows,
  strides, explicit padding, kernel dilation, in both float dtypes; bit-exact to the oracle."""
  from aqt_amd.v2 import aqt_conv_general as aqt_conv
  ns = len(case['lhs']) - 2
  raw = aqt_conv.conv_general_dilated_make(ns, 8, 8)
  lhs_np = _rand_unif(case['lhs'], 3.0, 5, dt)
  rhs_np = _rand_unif(case['rhs'], 0.5, 6, dt)
  lhs, rhs = U.to_dev(lhs_np, dt, gpu), U.to_dev(rhs_np, dt, gpu)
  out = aqt_conv.make_conv_general_dilated(raw)(
      lhs, rhs, window_strides=case['strides'], padding=case['padding'], rhs_dilation=case.get('dil'),
      dimension_numbers=aqt_conv.flax_conv_dimension_numbers(lhs.shape))
  want, _, _ = R.conv_general_dilated_fwd(lhs_np, rhs_np, dt, case['strides'], case['padding'],
                                          R.RawCfg(_qcfg(8, po2=False), _qcfg(8, po2=False)), case.get('dil'))
  assert out.dtype == U.TORCH_DT[dt] and tuple(out.shape) == want.shape
  np.testing.assert_array_equal(out.float().cpu().numpy(), want)


@pytest.mark.gpu
def test_conv_layout_and_axis_assertions(gpu):
  """aqt_conv_general.py:57-86: only the Flax layout, and the quantizers must share scales over
  the axes that layout implies."""
  from aqt_amd.v2 import aqt_conv_general as aqt_conv
  lhs = torch.zeros((2, 4, 4, 8), device=gpu)
  rhs = torch.zeros((3, 3, 8, 8), device=gpu)
  fn = aqt_conv.make_conv_general_dilated(aqt_conv.conv_general_dilated_make(2, 8, 8))
  dn = aqt_conv.flax_conv_dimension_numbers(lhs.shape)
  with pytest.raises(AssertionError, match='Flax-particular layout'):
    fn(lhs, rhs, (1, 1), 'SAME', dimension_numbers=None)
  with pytest.raises(AssertionError, match='Flax-particular layout'):
    fn(lhs, rhs, (1, 1), 'SAME', dimension_numbers=aqt_conv.ConvDimensionNumbers((0, 1, 2, 3), dn.rhs_spec, dn.out_spec))
  wrong = aqt_conv.make_conv_general_dilated(aqt_conv.conv_general_dilated_make(1, 8, 8))
  with pytest.raises(AssertionError, match='spatial'):
    wrong(lhs, rhs, (1, 1), 'SAME', dimension_numbers=dn)
  with pytest.raises(NotImplementedError):
    fn(lhs, rhs, (1, 1), 'SAME', dimension_numbers=dn, feature_group_count=2)
  # all-zero input: scales fall back to one, the output is zero
  assert (fn(lhs, rhs, (1, 1), 'SAME', dimension_numbers=dn) == 0).all()


@pytest.mark.gpu
@pytest.mark.parametrize('bits', [8, 4])
def test_conv_layer_train_convert_serve(gpu, bits):
  """AqtConvGeneralDilated as the reference's CNN example wires it (examples/flax_e2e_model.py:66-77,
  flax/aqt_flax.py:735-935): the kernel is frozen with its values, the input with its
  calibration only; serving reproduces the training-mode output without the float kernel."""
  from aqt_amd.v2 import aqt_conv_general as aqt_conv
  from aqt_amd.v2 import config, utils
  from aqt_amd.v2.flax import aqt_flax
  QM, FM = utils.QuantMode, aqt_flax.FreezerMode
  raw = config.conv_general_dilated_make(2, lhs_bits=bits, rhs_bits=bits, initialize_calibration=False)
  raw.dg_quantizer.lhs.init_calibration()
  raw.dg_quantizer.rhs.init_calibration()
  cfg = config.default_unquantized_config()
  cfg.fwd = raw
  x_np, k_np = _rand_unif((4, 14, 14, 32), 2.0, 3), _rand_unif((3, 3, 32, 64), 0.2, 4)
  x, k = U.to_dev(x_np, 'f32', gpu), U.to_dev(k_np, 'f32', gpu)
  dn = aqt_conv.flax_conv_dimension_numbers(x.shape)
  mk = lambda mode: aqt_flax.AqtConvGeneralDilated(
      cfg, lhs_quant_mode=QM.TRAIN, rhs_quant_mode=mode, lhs_freeze_mode=FM.CALIBRATION,
      rhs_freeze_mode=FM.CALIBRATION_AND_VALUE, rngs={'params': utils.prng_key(0)})
  out_train = mk(QM.TRAIN)(x, k, (1, 1), 'SAME', dimension_numbers=dn)
  want, _, _ = R.conv_general_dilated_fwd(x_np, k_np, 'f32', (1, 1), 'SAME',
                                          R.RawCfg(_qcfg(bits, po2=False), _qcfg(bits, po2=False)))
  np.testing.assert_array_equal(out_train.cpu().numpy(), want)
  conv = mk(QM.CONVERT)
  out_conv = conv(x, k, (1, 1), 'SAME', dimension_numbers=dn)
  v = conv.variables()
  assert set(v) == {'aqt'} and set(v['aqt']) == {'qrhs'}
  frozen = v['aqt']['qrhs']['frozen']
  assert tuple(frozen.qvalue.shape) == (3, 3, 32, 64) and frozen.qvalue.dtype == torch.int8
  assert [tuple(s.shape) for s in frozen.scale] == [(1, 1, 1, 64)]
  serve = mk(QM.SERVE)
  serve.load_variables(v)
  out_serve = serve(x, torch.zeros_like(k), (1, 1), 'SAME', dimension_numbers=dn)
  assert torch.equal(out_train, out_conv) and torch.equal(out_train, out_serve)
  # an unconfigured layer is the plain convolution
  plain = aqt_flax.AqtConvGeneralDilated(None)(x, k, (1, 1), 'SAME', dimension_numbers=dn)
  np.testing.assert_allclose(plain.cpu().numpy(), R.lax_conv_nhwc(x_np, k_np, (1, 1), 'SAME'), rtol=1e-4, atol=1e-4)


@pytest.mark.gpu
@pytest.mark.parametrize('case', [
    dict(x=(2, 7, 6, 16), ker=(3, 2), strides=(1, 1), pads=[(1, 1), (0, 1)], dil=(1, 1)),
    dict(x=(3, 9, 8, 32), ker=(3, 3), strides=(2, 1), pads=[(1, 1), (1, 1)], dil=(1, 1)),
    dict(x=(2, 12, 11, 16), ker=(2, 3), strides=(1, 2), pads=[(0, 0), (0, 0)], dil=(2, 1)),
    dict(x=(4, 33, 48), ker=(5,), strides=(3,), pads=[(2, 1)], dil=(1,)),
    dict(x=(2, 5, 6, 4, 16), ker=(2, 2, 2), strides=(1, 1, 2), pads=[(0, 1), (1, 0), (0, 1)], dil=(1, 1, 1)),
    dict(x=(2, 6, 5, 3), ker=(3, 3), strides=(1, 1), pads=[(1, 1), (1, 1)], dil=(1, 1)),   # features not a multiple of 16
    dict(x=(1, 4, 4, 16), ker=(5, 5), strides=(1, 1), pads=[(0, 0), (0, 0)], dil=(1, 1)),   # window larger than the input
    dict(x=(0, 4, 4, 16), ker=(3, 3), strides=(1, 1), pads=[(1, 1), (1, 1)], dil=(1, 1)),   # no images
])
def test_window_gather_kernel(gpu, case):
  """aqtx_im2col_i8 against pad + unfold on the same int8 tensor."""
  from aqt_amd import ops
  from aqt_amd.v2 import aqt_conv_general as aqt_conv
  rng = np.random.default_rng(3)
  x = torch.from_numpy(rng.integers(-127, 128, case['x']).astype(np.int8)).to(gpu)
  got, out_sizes = ops.im2col_i8(x, case['ker'], case['strides'], case['pads'], case['dil'])
  if x.shape[0] == 0 or any(o == 0 for o in out_sizes):
    assert got.shape[0] == 0
    return
  want, want_sizes = aqt_conv._windows(x, list(case['ker']), list(case['strides']), case['pads'], list(case['dil']))
  assert list(out_sizes) == list(want_sizes) and got.shape == want.shape
  assert torch.equal(got, want.contiguous())


@pytest.mark.gpu
@pytest.mark.parametrize('out,rdt,cdt', [('bf16', 'bf16', 'bf16'), ('bf16', 'f32', 'f32'), ('f32', 'f32', 'f32')])
@pytest.mark.parametrize('case', [
    dict(x=(2, 9, 8, 128), ker=(3, 3), strides=(1, 1), pads=[(1, 1), (1, 1)], dil=(1, 1), n=64),
    dict(x=(3, 12, 11, 256), ker=(3, 2), strides=(2, 1), pads=[(1, 0), (0, 1)], dil=(1, 2), n=200),
    dict(x=(5, 37, 128), ker=(5,), strides=(3,), pads=[(2, 1)], dil=(1,), n=130),
    dict(x=(2, 5, 6, 4, 128), ker=(2, 2, 2), strides=(1, 1, 2), pads=[(0, 1), (1, 0), (0, 1)], dil=(1, 1, 1), n=48),
    dict(x=(1, 4, 4, 128), ker=(5, 5), strides=(1, 1), pads=[(0, 0), (0, 0)], dil=(1, 1), n=16),   # no position at all
    dict(x=(2, 30, 30, 128), ker=(1, 1), strides=(1, 1), pads=[(0, 0), (0, 0)], dil=(1, 1), n=256),  # one tap = one stage
])
def test_convolution_without_the_window_matrix(gpu, case, out, rdt, cdt):
  """aqtx_conv_i8 (the windows read in place by the contraction kernel) against aqtx_im2col_i8 + aqtx_gemm_i8:
  the same bits, for strides, dilations, uneven padding, one to three spatial axes."""
  from aqt_amd import ops
  rng = np.random.default_rng(5)
  x = torch.from_numpy(rng.integers(-127, 128, case['x']).astype(np.int8)).to(gpu)
  taps = int(np.prod(case['ker']))
  k, n = taps * case['x'][-1], case['n']
  w = torch.from_numpy(rng.integers(-127, 128, (n, k)).astype(np.int8)).to(gpu)
  a, out_sizes = ops.im2col_i8(x, case['ker'], case['strides'], case['pads'], case['dil'])
  m = a.shape[0]
  if m == 0:
    return
  rs = torch.from_numpy(nm.cast(np.abs(rng.standard_normal(m).astype(np.float32)) * np.float32(0.02) + np.float32(1e-3), rdt)).to(gpu)
  cs = torch.from_numpy(nm.cast(np.abs(rng.standard_normal(n).astype(np.float32)) * np.float32(3e-3) + np.float32(1e-4), cdt)).to(gpu)
  kw = dict(out_dtype=U.TORCH_DT[out], row_scale_dtype=U.TORCH_DT[rdt], col_scale_dtype=U.TORCH_DT[cdt])
  want = ops.gemm(a[None], w[None], row_scale=rs[None], col_scale=cs[None], **kw)[0]
  got, got_sizes = ops.conv_i8(x, w, case['ker'], case['strides'], case['pads'], case['dil'], row_scale=rs, col_scale=cs, **kw)
  assert list(got_sizes) == list(out_sizes)
  assert torch.equal(got, want)


@pytest.mark.gpu
def test_conv_layer_with_128_features_matches_oracle(gpu):
  """A quantized convolution whose input has 128 features takes the one-kernel path (strides, dilation and
  uneven padding included); bit-exact to the oracle."""
  from aqt_amd.v2 import aqt_conv_general as aqt_conv
  dt = 'bf16'
  for case in (dict(lhs=(2, 10, 9, 128), rhs=(3, 3, 128, 40), strides=(1, 1), padding='SAME'),
               dict(lhs=(2, 13, 12, 256), rhs=(3, 2, 256, 130), strides=(2, 1), padding=[(1, 0), (0, 2)], dil=(1, 2))):
    raw = aqt_conv.conv_general_dilated_make(2, 8, 8)
    lhs_np = _rand_unif(case['lhs'], 3.0, 5, dt)
    rhs_np = _rand_unif(case['rhs'], 0.5, 6, dt)
    lhs, rhs = U.to_dev(lhs_np, dt, gpu), U.to_dev(rhs_np, dt, gpu)
    out = aqt_conv.make_conv_general_dilated(raw)(
        lhs, rhs, window_strides=case['strides'], padding=case['padding'], rhs_dilation=case.get('dil'),
        dimension_numbers=aqt_conv.flax_conv_dimension_numbers(lhs.shape))
    want, _, _ = R.conv_general_dilated_fwd(lhs_np, rhs_np, dt, case['strides'], case['padding'],
                                            R.RawCfg(_qcfg(8, po2=False), _qcfg(8, po2=False)), case.get('dil'))
    assert tuple(out.shape) == want.shape
    np.testing.assert_array_equal(out.float().cpu().numpy(), want)


@pytest.mark.gpu
@pytest.mark.parametrize('cout', [128, 24])  # with and without a window matrix
def test_scales_written_past_autograd_are_the_ones_used(gpu, cout):
  """A scale of a quantized tensor changed through .data (which no version counts) before the tensor is used again."""
  from aqt_amd.v2 import aqt_conv_general
  conv = aqt_conv_general.make_conv_general_dilated_with_qt(aqt_conv_general.conv_general_dilated_make(2, 8, 8))
  x = U.to_dev(_rand_unif((2, 7, 7, 16), 1.0, 1, 'bf16'), 'bf16', gpu)
  w = U.to_dev(_rand_unif((3, 3, 16, cout), 1.0, 2, 'bf16'), 'bf16', gpu)
  kw = dict(window_strides=(1, 1), padding='SAME', dimension_numbers=aqt_conv_general.flax_conv_dimension_numbers(x.shape))
  out, (lq, rq) = conv(x, w, **kw)
  rq.scale[0].data.mul_(2)
  lq.scale[0].data = lq.scale[0] * 4
  assert torch.equal(conv(x, w, lhs_qt=lq, rhs_qt=rq, **kw)[0], out * 8)

  quantizer = aqt_conv_general.conv_general_dilated_make(2, 8, 8).dg_quantizer.rhs
  qt = quantizer.calibrate(w, calibration_axes=[0, 1, 2])
  qt.scale[0].data.mul_(2)
  got, _ = quantizer.calculate_qvalue(w, qt)
  want = torch.clamp(torch.round((w * (1 / qt.scale[0]))), -127, 127).to(torch.int8)
  assert torch.equal(got.qvalue, want)


@pytest.mark.gpu
@pytest.mark.parametrize('n,positions,features', [(1, 1, 1), (3, 49, 24), (32, 100, 128), (2, 1, 300), (5, 0, 7)])
@pytest.mark.parametrize('rdt,cdt', [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.bfloat16), (torch.bfloat16, torch.float32)])
def test_conv_scales(gpu, rdt, cdt, n, positions, features):
  from aqt_amd import ops
  row = torch.rand((n, 1, 1, 1), device=gpu).to(rdt)
  col = torch.rand((1, 1, 1, 2 * features), device=gpu).to(cdt)[..., ::2]  # not contiguous
  rows, cols = ops.conv_scales(row, col, positions)
  assert torch.equal(rows, row.float().reshape(n, 1).expand(n, positions).reshape(-1)) and torch.equal(cols, col.float().reshape(-1))
  assert rows.data_ptr() % 16 == 0 and cols.data_ptr() % 16 == 0
