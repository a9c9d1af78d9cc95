"""GPU parity: aqtx_quantize / aqtx_random_bits against the numpy oracle (bit-exact)."""
import numpy as np
import pytest
import torch

from aqt_amd import _lib as L
from aqt_amd import ops
from oracle import aqt_ref as R
from oracle import numerics as nm
from oracle import prng
from tests import gpu_util as U

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('partitionable', [False, True])
@pytest.mark.parametrize('width', [16, 32])
@pytest.mark.parametrize('n', [1, 2, 7, 4096, 100003])
def test_random_bits(gpu, n, width, partitionable):
  key = prng.prng_key(42)
  got = ops.random_bits(key, n, width, partitionable, device=gpu).cpu().numpy()
  got = got.view(np.uint16 if width == 16 else np.uint32)
  want = prng.random_bits(key, (n,), width, partitionable)
  np.testing.assert_array_equal(got, want)


def test_prng_split_host():
  for part in (False, True):
    for num in (1, 2, 3, 5):
      np.testing.assert_array_equal(ops.prng_split(prng.prng_key(7), num, part),
                                    prng.split(prng.prng_key(7), num, part))


def _oracle_quant(x, dt, q, axes, prescale=None, ps_axis=None):
  if prescale is not None:
    shape = [1] * x.ndim
    shape[ps_axis] = x.shape[ps_axis]
    x = nm.cast(x * nm.cast(prescale.reshape(shape), dt), dt)
  return R.quantize(x, dt, q, axes)


def _check(qt, q_got, s_got, cfg, transpose=False):
  want_q = qt.qvalue
  if cfg.is_fp8():
    got = U.fp8_bytes_to_float(q_got, cfg.bits)
  else:
    got = q_got.astype(np.float32)
    want_q = want_q.astype(np.float32)
  if transpose:
    got = np.swapaxes(got, -1, -2)
  np.testing.assert_array_equal(s_got.reshape(-1), qt.scale[0].reshape(-1))
  np.testing.assert_array_equal(got, want_q)


ROW_CASES = [
    # (rows, cols, group)
    (4, 64, 0), (33, 128, 0), (5, 512, 0), (3, 2048, 0), (7, 4096, 0), (2, 8192, 0),
    (2, 14336, 0), (3, 100, 0), (2, 20000, 0), (6, 1024, 128), (3, 96, 32),
    # few long rows: taken as one scale per batch entry of [batch * rows][cols / c][c]
    (3, 32768, 0), (5, 16448, 0), (2, 401408, 0), (1, 16384, 0),
]


@pytest.mark.parametrize('dt', ['bf16', 'f32'])
@pytest.mark.parametrize('rows,cols,group', ROW_CASES)
def test_rows_int8_rtn(gpu, rows, cols, group, dt):
  x = U.rand((2, rows, cols), dt, seed=rows * 131 + cols, outliers=True)
  x[0, 0, :] = 0.0  # an all-zero row: abs-max 0 -> scale 1/127.5 path (calibration.py:148)
  q = R.QuantizerCfg(bits=8)
  if group:
    xv = x.reshape(2, rows, cols // group, group)
    qt = R.quantize(xv, dt, q, [3])
  else:
    qt = R.quantize(x, dt, q, [2])
  qb, cb = U.bounds(q)
  qg, sg = ops.quantize(U.to_dev(x, dt, gpu), reduce=L.REDUCE_COLS, out_dtype=L.I8,
                        quant_bound=qb, clip_bound=cb, group=group)
  got = qg.cpu().numpy()
  if group:
    got = got.reshape(2, rows, cols // group, group)
  _check(qt, got, sg.cpu().numpy(), q)


@pytest.mark.parametrize('bits,noise,scale_dtype', [
    (8, 'jax.uniform', None), (8, 'custom-1', None), (4, None, None), (4, 'jax.uniform', 'f32'),
    ('e4m3', None, None), ('e5m2', None, None), ('e4m3', 'sr', None), ('e5m2', 'sr', None),
    ('e5m2', 'sr', 'f32'), (8, None, 'f32'),
])
@pytest.mark.parametrize('partitionable', [False, True])
@pytest.mark.parametrize('dt', ['bf16', 'f32'])
def test_rows_numerics(gpu, bits, noise, scale_dtype, partitionable, dt, monkeypatch):
  monkeypatch.setattr(R, 'PARTITIONABLE', partitionable)
  rows, cols = 9, 1000 if noise else 256
  x = U.rand((1, rows, cols), dt, seed=5, scale=0.02)
  key = prng.prng_key(1234)
  q = R.QuantizerCfg(bits=bits, scale_dtype=scale_dtype, key=key)
  knoise = L.NOISE_NONE
  if noise == 'sr':
    q.fp8_sr = True
    knoise = L.NOISE_FP8_MANTISSA
  elif noise:
    q.noise = noise
    knoise = U.NOISE[noise]
  qt = R.quantize(x, dt, q, [2])
  qb, cb = U.bounds(q)
  qg, sg = ops.quantize(U.to_dev(x, dt, gpu), reduce=L.REDUCE_COLS, out_dtype=U.OUT_DT[bits],
                        quant_bound=qb, clip_bound=cb, noise=knoise, key=key,
                        partitionable=partitionable,
                        scale_dtype=U.TORCH_DT[scale_dtype] if scale_dtype else None)
  _check(qt, qg.cpu().numpy(), sg.cpu().numpy(), q)


@pytest.mark.parametrize('dt', ['bf16', 'f32'])
@pytest.mark.parametrize('rows,cols,group,transpose', [
    (128, 64, 0, True), (300, 200, 0, True), (256, 520, 0, False), (77, 13, 0, True),
    (77, 13, 0, False), (512, 256, 128, True), (256, 64, 32, False), (1024, 1024, 0, True),
])
def test_cols_int8(gpu, rows, cols, group, transpose, dt):
  x = U.rand((2, rows, cols), dt, seed=rows + cols, outliers=True)
  x[:, :, 1] = 0.0
  key = prng.prng_key(99)
  q = R.QuantizerCfg(bits=8, noise='jax.uniform', key=key)
  if group:
    qt = R.quantize(x.reshape(2, rows // group, group, cols), dt, q, [2])
    want_q = qt.qvalue.reshape(2, rows, cols)
    # noise index is the row-major index of the [2, rows/group, group, cols] tensor = same memory order
  else:
    qt = R.quantize(x, dt, q, [1])
    want_q = qt.qvalue
  qb, cb = U.bounds(q)
  qg, sg = ops.quantize(U.to_dev(x, dt, gpu), reduce=L.REDUCE_ROWS, out_dtype=L.I8,
                        quant_bound=qb, clip_bound=cb, group=group, transpose_out=transpose,
                        noise=L.NOISE_JAX_UNIFORM, key=key)
  got = qg.cpu().numpy()
  if transpose:
    got = np.swapaxes(got, 1, 2)
  np.testing.assert_array_equal(sg.cpu().numpy().reshape(-1), qt.scale[0].reshape(-1))
  np.testing.assert_array_equal(got, want_q)


@pytest.mark.parametrize('bits', [8, 'e4m3', 'e5m2'])
@pytest.mark.parametrize('dt', ['bf16', 'f32'])
def test_per_tensor(gpu, bits, dt):
  x = U.rand((3, 130, 72), dt, seed=3)
  q = R.QuantizerCfg(bits=bits, calib_shared_axes=None)
  qb, cb = U.bounds(q)
  qg, sg = ops.quantize(U.to_dev(x, dt, gpu), reduce=L.REDUCE_ALL, out_dtype=U.OUT_DT[bits],
                        quant_bound=qb, clip_bound=cb)
  qt = R.quantize(x, dt, q, [1, 2])  # one scale per batch entry
  _check(qt, qg.cpu().numpy(), sg.cpu().numpy(), q)


@pytest.mark.parametrize('dt', ['bf16', 'f32'])
def test_prescale_and_requant(gpu, dt):
  """The two bwd-side uses: g * other-side scale, and re-quantizing int8 residuals."""
  m, n = 96, 256
  g = U.rand((1, m, n), dt, seed=11, scale=1e-3)
  col_ps = nm.cast(np.abs(U.rand((n,), 'f32', 12, 6e-4)) + np.float32(1e-5), dt)
  row_ps = nm.cast(np.abs(U.rand((m,), 'f32', 13, 0.03)) + np.float32(1e-3), dt)
  key = prng.prng_key(5)
  q = R.QuantizerCfg(bits=8, noise='jax.uniform', key=key)
  qb, cb = U.bounds(q)
  gd = U.to_dev(g, dt, gpu)
  # dlhs: per-column prescale, row-wise scales
  qt = _oracle_quant(g, dt, q, [2], col_ps, 2)
  qg, sg = ops.quantize(gd, reduce=L.REDUCE_COLS, out_dtype=L.I8, quant_bound=qb, clip_bound=cb,
                        noise=L.NOISE_JAX_UNIFORM, key=key,
                        prescale=torch.from_numpy(col_ps).to(gpu), prescale_mode=L.PRESCALE_PER_COL)
  _check(qt, qg.cpu().numpy(), sg.cpu().numpy(), q)
  # drhs: per-row prescale, column-wise scales, transposed write
  qt = _oracle_quant(g, dt, q, [1], row_ps, 1)
  qg, sg = ops.quantize(gd, reduce=L.REDUCE_ROWS, out_dtype=L.I8, quant_bound=qb, clip_bound=cb,
                        noise=L.NOISE_JAX_UNIFORM, key=key, transpose_out=True,
                        prescale=torch.from_numpy(row_ps).to(gpu), prescale_mode=L.PRESCALE_PER_ROW)
  _check(qt, qg.cpu().numpy(), sg.cpu().numpy(), q, transpose=True)
  # residual re-quantization: int8 input in a [n, k] buffer standing for a logical [k, n] tensor
  k = 128
  w_q = np.random.default_rng(3).integers(-127, 128, size=(k, n)).astype(np.int8)  # logical [k, n]
  qt = R.quantize(w_q.astype(np.float32)[None], dt, q, [2])  # per-k scale over n
  mem = torch.from_numpy(np.ascontiguousarray(w_q.T)[None]).to(gpu)  # memory [1, n, k]
  qg, sg = ops.quantize(mem, reduce=L.REDUCE_ROWS, out_dtype=L.I8, quant_bound=qb, clip_bound=cb,
                        compute_dtype=U.TORCH_DT[dt], noise=L.NOISE_JAX_UNIFORM, key=key,
                        transpose_out=True, noise_strides=(k * n, 1, n), noise_total=k * n)
  np.testing.assert_array_equal(sg.cpu().numpy().reshape(-1), qt.scale[0].reshape(-1))
  np.testing.assert_array_equal(qg.cpu().numpy(), qt.qvalue)  # transposed write -> [1, k, n]


@pytest.mark.parametrize('kind', ['e4m3', 'e5m2'])
def test_fp8_cast_exhaustive(gpu, kind):
  """Every finite bf16 value through clip + fp8 cast (scale fixed to 1)."""
  bits = np.arange(65536, dtype=np.uint32)
  x = (bits << np.uint32(16)).astype(np.uint32).view(np.float32).copy()
  x[~np.isfinite(x)] = 0.0
  x = x.reshape(1, 64, 1024)
  q = R.QuantizerCfg(bits=kind)
  b = np.float32(R.quant_bound(q))
  want = (nm.to_e4m3fn if kind == 'e4m3' else nm.to_e5m2)(np.clip(x, -b, b))
  ones = torch.ones((1, 64, 1), dtype=torch.float32, device=gpu)
  qg, _ = ops.quantize(U.to_dev(x, 'bf16', gpu), reduce=L.REDUCE_COLS, out_dtype=U.OUT_DT[kind],
                       quant_bound=float(b), clip_bound=float(b), scale=ones)
  got = U.fp8_bytes_to_float(qg.cpu().numpy(), kind)
  np.testing.assert_array_equal(got, want)
  # signed zero / sign of tiny values must survive as well
  np.testing.assert_array_equal(np.signbit(got), np.signbit(want))


def test_workspace_kept_across_calls(gpu):
  """The abs-max workspace is shared by successive calls and handed back zeroed: calls with
  many, few, and again many scales, column-wise and per tensor, give what a first call gives."""
  from aqt_amd import _lib as L
  rng = np.random.default_rng(5)
  xs = [torch.from_numpy(rng.standard_normal(s).astype(np.float32)).to(torch.bfloat16).to(gpu)
        for s in ((1, 96, 4096), (1, 64, 24), (2, 40, 1000), (1, 128, 8192))]
  kw = dict(out_dtype=L.I8, quant_bound=127.5, clip_bound=127.0)
  first = {}
  for rnd in range(3):
    for i, x in enumerate(xs):
      for reduce in (L.REDUCE_ROWS, L.REDUCE_ALL_BATCH):
        q, s = ops.quantize(x, reduce=reduce, **kw)
        if rnd == 0:
          amax = x.float().abs().amax(dim=1) if reduce == L.REDUCE_ROWS else x.float().abs().amax().reshape(1)
          want = (amax / 127.5).to(torch.bfloat16).float()
          assert torch.equal(s.reshape(-1), want.reshape(-1))
          first[(i, reduce)] = (q.clone(), s.clone())
        else:
          assert torch.equal(q, first[(i, reduce)][0]) and torch.equal(s, first[(i, reduce)][1])


@pytest.mark.parametrize('noise', ['jax.uniform', 'custom-1'])
@pytest.mark.parametrize('dt', ['bf16', 'f32'])
@pytest.mark.parametrize('batch,rows,cols', [(1, 4, 32768), (2, 3, 16448), (3, 1, 65536)])
def test_few_long_rows_stochastic_rounding(gpu, batch, rows, cols, noise, dt):
  """The few-long-rows form with noise: the counters of [batch, rows, cols] carry over to the
  per-batch-entry form, and a scale handed in is used the same way."""
  x = U.rand((batch, rows, cols), dt, seed=cols + rows, scale=0.3)
  key = prng.prng_key(77)
  q = R.QuantizerCfg(bits=8, key=key, noise=noise)
  qt = R.quantize(x, dt, q, [2])
  qb, cb = U.bounds(q)
  qg, sg = ops.quantize(U.to_dev(x, dt, gpu), reduce=L.REDUCE_COLS, out_dtype=L.I8, quant_bound=qb, clip_bound=cb,
                        noise=U.NOISE[noise], key=key)
  _check(qt, qg.cpu().numpy(), sg.cpu().numpy(), q)
  qg2, _ = ops.quantize(U.to_dev(x, dt, gpu), reduce=L.REDUCE_COLS, out_dtype=L.I8, quant_bound=qb, clip_bound=cb,
                        noise=U.NOISE[noise], key=key, scale=sg.clone())
  assert torch.equal(qg, qg2)


@pytest.mark.parametrize('reduce,transpose,shape', [
    (L.REDUCE_COLS, False, (1, 64, 1024)),   # rows kernel, rows paired over one threefry block
    (L.REDUCE_COLS, False, (2, 9, 1000)),    # rows kernel, plain
    (L.REDUCE_COLS, False, (1, 5, 1001)),    # generic rows kernel
    (L.REDUCE_ROWS, True, (1, 256, 192)),    # tile kernel, transposed write
    (L.REDUCE_ALL, False, (2, 130, 70)),     # tile kernel, one scale per batch entry
])
@pytest.mark.parametrize('noise,out', [(L.NOISE_JAX_UNIFORM, L.I8), (L.NOISE_FP8_MANTISSA, L.E5M2)])
def test_key_in_device_memory_equals_key_in_the_plan(gpu, reduce, transpose, shape, noise, out):
  """plan.key_device: the kernels read the two key words from device memory (the form a traced
  jax key arrives in under XLA); same bits as the key given by value."""
  x = U.to_dev(U.rand(shape, 'bf16', seed=7, scale=0.5), 'bf16', gpu)
  key = prng.prng_key(4321)
  qb, cb = (127.5, 127.0) if out == L.I8 else (57344.0, 57344.0)
  kw = dict(reduce=reduce, out_dtype=out, quant_bound=qb, clip_bound=cb, noise=noise, transpose_out=transpose)
  q0, s0 = ops.quantize(x, key=key, **kw)
  kd = torch.tensor([int(key[0]), int(key[1])], dtype=torch.int64).to(torch.int32).to(gpu) if max(key) < 2**31 else \
      torch.from_numpy(np.asarray(key, dtype=np.uint32).view(np.int32).copy()).to(gpu)
  q1, s1 = ops.quantize(x, key_device=kd, **kw)
  assert torch.equal(q0, q1) and torch.equal(s0, s1)
  # and a different key gives different bits (the device key is really what is read)
  kd2 = kd.clone()
  kd2[1] += 1
  q2, _ = ops.quantize(x, key_device=kd2, **kw)
  assert not torch.equal(q0, q2)


@pytest.mark.parametrize('dt', ['bf16', 'f32'])
@pytest.mark.parametrize('reduce,shape', [
    (L.REDUCE_COLS, (2, 9, 1024)), (L.REDUCE_COLS, (1, 3, 1001)), (L.REDUCE_ROWS, (1, 200, 96)),
    (L.REDUCE_ALL, (3, 40, 64)),
])
def test_nan_reaches_the_scale(gpu, dt, reduce, shape):
  """jnp.max(jnp.abs(x)) propagates a NaN into the scale (calibration.py:126-157), which is how a
  diverged step shows up in the outputs; the kernels' abs-max does the same, and the scales of
  segments without a NaN are untouched."""
  x = U.rand(shape, dt, seed=11)
  x[0, 1, 5] = np.nan
  q = R.QuantizerCfg(bits=8)
  axes = {L.REDUCE_COLS: [2], L.REDUCE_ROWS: [1], L.REDUCE_ALL: [1, 2]}[reduce]
  with np.errstate(invalid='ignore'):
    want = R.quantize(x, dt, q, axes).scale[0].reshape(-1)
  _, sg = ops.quantize(U.to_dev(x, dt, gpu), reduce=reduce, out_dtype=L.I8, quant_bound=127.5, clip_bound=127.0)
  got = sg.cpu().numpy().reshape(-1)
  assert np.isnan(want).sum() == 1
  np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
  np.testing.assert_array_equal(got[~np.isnan(want)], want[~np.isnan(want)])


def test_nan_row_gives_nan_outputs(gpu):
  """End to end: one NaN activation makes exactly that token's outputs NaN (its scale is NaN), in
  the training-shape path and in the serving kernels."""
  from aqt_amd.v2 import aqt_dot_general as aqt
  from aqt_amd.v2 import config
  lhs = torch.randn(48, 256, device=gpu).to(torch.bfloat16)
  rhs = (torch.randn(256, 64, device=gpu) * 0.05).to(torch.bfloat16)
  lhs[7, 100] = float('nan')
  cfg = config.set_context(config.fully_quantized(fwd_bits=8, bwd_bits=8, use_stochastic_rounding=False), None, None)
  out, _ = cfg.dg_core(lhs, rhs, None, None, (((1,), (0,)), ((), ())))
  bad = torch.isnan(out).any(dim=1).cpu().numpy()
  assert bad[7] and bad.sum() == 1 and bool(torch.isnan(out[7]).all())
  wq = torch.randint(-127, 128, (64, 256), dtype=torch.int8, device=gpu)
  ws = torch.rand(64, device=gpu) * 1e-3
  for m in (2, 48):
    o, xs = ops.decode(lhs[6:6 + m].contiguous(), wq, ws, quant_bound=127.5, clip_bound=127.0)
    assert bool(torch.isnan(xs[1])) and bool(torch.isnan(o[1]).all()) and not bool(torch.isnan(o[0]).any())


@pytest.mark.parametrize('reduce,rows,cols', [
    # whole rows, two of them sharing the blocks of the generator: the smallest and largest of every launch shape
    (L.REDUCE_COLS, 2, 8), (L.REDUCE_COLS, 6, 128), (L.REDUCE_COLS, 4, 136), (L.REDUCE_COLS, 2, 2048),
    (L.REDUCE_COLS, 2, 2056), (L.REDUCE_COLS, 2, 8192), (L.REDUCE_COLS, 2, 8200), (L.REDUCE_COLS, 2, 16384),
    (L.REDUCE_COLS, 5, 1000),                           # an odd number of rows: one block an element
    # tiles: rows / 2 apart, with remainders in both directions; cols / 2 apart; an odd number of rows
    (L.REDUCE_ROWS, 256, 64), (L.REDUCE_ROWS, 258, 200), (L.REDUCE_ROWS, 130, 13), (L.REDUCE_ROWS, 77, 64),
])
@pytest.mark.parametrize('noise', [None, 'jax.uniform'])
def test_float32_pipelines_match_the_oracle(gpu, reduce, rows, cols, noise):
  """float32 values and scales: rows and tiles, and the re-quantization of int8 values in float32 arithmetic, with
  noise counters in memory order and in the order of the transposed tensor."""
  key = prng.prng_key(31)
  q = R.QuantizerCfg(bits=8, noise=noise, key=key)
  qb, cb = U.bounds(q)
  by_row = reduce == L.REDUCE_COLS
  kw = dict(reduce=reduce, out_dtype=L.I8, quant_bound=qb, clip_bound=cb, noise=U.NOISE[noise], key=key,
            transpose_out=not by_row)
  x = U.rand((1, rows, cols), 'f32', seed=rows + cols, outliers=True)
  qt = R.quantize(x, 'f32', q, [2 if by_row else 1])
  qg, sg = ops.quantize(U.to_dev(x, 'f32', gpu), **kw)
  _check(qt, qg.cpu().numpy(), sg.cpu().numpy(), q, transpose=not by_row)
  if by_row:
    return
  w = np.random.default_rng(rows).integers(-127, 128, size=(cols, rows)).astype(np.int8)  # logical [cols, rows]
  qt = R.quantize(w.astype(np.float32)[None], 'f32', q, [2])
  qg, sg = ops.quantize(torch.from_numpy(np.ascontiguousarray(w.T)[None]).to(gpu), compute_dtype=torch.float32,
                        noise_strides=(rows * cols, 1, rows), noise_total=rows * cols, **kw)
  _check(qt, qg.cpu().numpy(), sg.cpu().numpy(), q)


@pytest.mark.parametrize('dt,batch,rows,cols', [
    # around tiles of 32 x 64, halved where two tiles share the blocks of the generator; entries that do not pair
    *[(dt, *s) for dt in ('bf16', 'f32') for s in ((1, 31, 64), (1, 32, 128), (1, 62, 70), (1, 64, 126), (1, 66, 130), (1, 254, 58),
                                                   (2, 32, 64), (3, 33, 63), (2, 65, 57))],
    # the last and the first sizes on either side of the line to tall tiles
    ('f32', 1, 2 * 128 * 512, 9), ('f32', 1, 2 * 128 * 512 + 2, 9), ('bf16', 1, 2 * 128 * 2048, 9), ('bf16', 1, 2 * 128 * 2048 + 2, 9),
])
@pytest.mark.parametrize('bits', [8, 'e5m2'])
def test_tiles_with_noise_low_and_tall(gpu, bits, dt, batch, rows, cols):
  """Scales by column, with noise counters in memory order (both output orders) and, integers, in that of the transposed tensor."""
  key = prng.prng_key(rows + cols)
  q = R.QuantizerCfg(bits=bits, key=key, **({'noise': 'jax.uniform'} if bits == 8 else {'fp8_sr': True}))
  qb, cb = U.bounds(q)
  kw = dict(reduce=L.REDUCE_ROWS, out_dtype=U.OUT_DT[bits], quant_bound=qb, clip_bound=cb,
            noise=L.NOISE_JAX_UNIFORM if bits == 8 else L.NOISE_FP8_MANTISSA, key=key)
  x = U.rand((batch, rows, cols), dt, seed=rows + cols, outliers=True)
  qt = R.quantize(x, dt, q, [1])
  for transpose in (True, False):
    qg, sg = ops.quantize(U.to_dev(x, dt, gpu), transpose_out=transpose, **kw)
    _check(qt, qg.cpu().numpy(), sg.cpu().numpy(), q, transpose=transpose)
  if bits == 8 and batch == 1:
    w = np.random.default_rng(rows).integers(-127, 128, size=(cols, rows)).astype(np.int8)  # logical [cols, rows]
    qt = R.quantize(w.astype(np.float32)[None], dt, q, [2])
    qg, sg = ops.quantize(torch.from_numpy(np.ascontiguousarray(w.T)[None]).to(gpu), compute_dtype=U.TORCH_DT[dt],
                          noise_strides=(rows * cols, 1, rows), noise_total=rows * cols, transpose_out=True, **kw)
    _check(qt, qg.cpu().numpy(), sg.cpu().numpy(), q)


@pytest.mark.parametrize('rows,cols', [
    # around the pieces of 8, the launch shapes of the rows kernel and the 128 x 64 tiles (halved where two tiles share
    # the blocks of the generator); fewer than a piece or a tile
    (3, 7), (2, 9), (130, 63), (127, 65), (128, 129), (257, 130), (258, 67), (254, 126), (6, 511), (4, 2049), (2, 4099), (3, 8193),
    (2, 16383), (9, 1),
])
@pytest.mark.parametrize('bits,noise', [(8, None), (8, 'jax.uniform'), ('e5m2', 'sr'), ('e4m3', None)])
@pytest.mark.parametrize('dt', ['bf16', 'f32'])
def test_sizes_that_are_no_multiples_of_anything(gpu, dt, bits, noise, rows, cols):
  """Scales by row, by column and by tensor, written in the input's order and transposed, two batch entries where the
  noise does not pair tiles, and a prescale along the other axis."""
  key = prng.prng_key(rows * 7 + cols)
  q = R.QuantizerCfg(bits=bits, key=key)
  if noise == 'sr':
    q.fp8_sr = True
  elif noise:
    q.noise = noise
  kn = {None: L.NOISE_NONE, 'sr': L.NOISE_FP8_MANTISSA}.get(noise, U.NOISE.get(noise))
  qb, cb = U.bounds(q)
  kw = dict(out_dtype=U.OUT_DT[bits], quant_bound=qb, clip_bound=cb, noise=kn, key=key)
  for batch in (1, 2):
    x = U.rand((batch, rows, cols), dt, seed=rows + cols, outliers=True)
    xd = U.to_dev(x, dt, gpu)
    for reduce, axes, transpose in ((L.REDUCE_COLS, [2], False), (L.REDUCE_ROWS, [1], False), (L.REDUCE_ROWS, [1], True),
                                    (L.REDUCE_ALL, [1, 2], True)):
      qg, sg = ops.quantize(xd, reduce=reduce, transpose_out=transpose, **kw)
      _check(R.quantize(x, dt, q, axes), qg.cpu().numpy(), sg.cpu().numpy(), q, transpose=transpose)
  ps = nm.cast(np.abs(U.rand((cols,), 'f32', 3, 0.03)) + np.float32(1e-3), dt)
  x = x[:1]
  qg, sg = ops.quantize(xd[:1].contiguous(), reduce=L.REDUCE_COLS, prescale=torch.from_numpy(ps).to(gpu),
                        prescale_mode=L.PRESCALE_PER_COL, **kw)
  _check(_oracle_quant(x, dt, q, [2], ps, 2), qg.cpu().numpy(), sg.cpu().numpy(), q)
  ps = nm.cast(np.abs(U.rand((rows,), 'f32', 4, 0.03)) + np.float32(1e-3), dt)
  qg, sg = ops.quantize(xd[:1].contiguous(), reduce=L.REDUCE_ROWS, transpose_out=True, prescale=torch.from_numpy(ps).to(gpu),
                        prescale_mode=L.PRESCALE_PER_ROW, **kw)
  _check(_oracle_quant(x, dt, q, [1], ps, 1), qg.cpu().numpy(), sg.cpu().numpy(), q, transpose=True)


@pytest.mark.parametrize('rows,cols,dt,bits,noise', [
    # even row counts share the generator's blocks between rows, odd ones do not; either side of a line where it matters
    (20478, 9, 'bf16', 8, 'jax.uniform'), (20480, 9, 'bf16', 8, 'jax.uniform'), (6142, 31, 'f32', 8, 'jax.uniform'),
    (6144, 31, 'f32', 8, 'jax.uniform'), (2046, 129, 'bf16', 8, 'jax.uniform'), (2048, 129, 'bf16', 8, 'jax.uniform'),
    (4096, 570, 'bf16', 8, 'jax.uniform'), (32769, 10, 'bf16', 8, 'jax.uniform'), (4097, 100, 'f32', 8, 'jax.uniform'),
    (2049, 399, 'bf16', 8, 'jax.uniform'), (2049, 401, 'bf16', 8, 'jax.uniform'), (2049, 1023, 'f32', 'e5m2', 'sr'),
    (4096, 639, 'bf16', 8, None), (4096, 641, 'bf16', 8, None), (4095, 20, 'f32', 'e4m3', None), (4096, 20, 'f32', 'e4m3', None),
    (2048, 799, 'f32', 'e4m3', None),
])
def test_row_kernels_on_both_sides_of_their_lines(gpu, rows, cols, dt, bits, noise):
  q = R.QuantizerCfg(bits=bits, key=prng.prng_key(rows + cols))
  if noise == 'sr':
    q.fp8_sr = True
  elif noise:
    q.noise = noise
  qb, cb = U.bounds(q)
  x = U.rand((1, rows, cols), dt, seed=rows + cols, outliers=True)
  qg, sg = ops.quantize(U.to_dev(x, dt, gpu), reduce=L.REDUCE_COLS, out_dtype=U.OUT_DT[bits], quant_bound=qb, clip_bound=cb,
                        noise={None: L.NOISE_NONE, 'sr': L.NOISE_FP8_MANTISSA}.get(noise, U.NOISE.get(noise)), key=q.key)
  _check(R.quantize(x, dt, q, [2]), qg.cpu().numpy(), sg.cpu().numpy(), q)


@pytest.mark.parametrize('reduce,shape,group', [
    (L.REDUCE_ROWS, (1, 4096, 600), 0), (L.REDUCE_ROWS, (2, 130, 1025), 0), (L.REDUCE_ROWS, (1, 16, 5), 0),
    (L.REDUCE_ROWS, (2, 256, 513), 64), (L.REDUCE_ALL, (3, 1000, 257), 0), (L.REDUCE_ALL_BATCH, (3, 1000, 257), 0),
    (L.REDUCE_ALL_BATCH, (1, 3, 2), 0),
])
def test_scales_from_the_last_block_equal_those_of_their_own_launch(gpu, reduce, shape, group):
  """A kept workspace with room for the arrival counts and one without; calls of other sizes in between leave both as
  they have to be found (zero); and the same scales given instead of computed."""
  kw = dict(reduce=reduce, out_dtype=L.I8, quant_bound=127.5, clip_bound=127.0, group=group)
  x = U.to_dev(U.rand(shape, 'bf16', seed=sum(shape), outliers=True), 'bf16', gpu)
  y = U.to_dev(U.rand((2, 700, 1300), 'bf16', seed=1), 'bf16', gpu)
  results = []
  for room in (True, False):
    if room:
      with ops.private_workspaces({}) as store:
        for _ in range(3):
          results.append(ops.quantize(x, **kw))
          ops.quantize(y, reduce=L.REDUCE_ROWS, out_dtype=L.I8, quant_bound=127.5, clip_bound=127.0)
        words = [t for t in store.values()]
      assert len(words) == 1 and not bool(words[0][:words[0].numel() // 2].any())
    else:
      n = results[0][1].numel()
      ws = torch.zeros(8 * n, dtype=torch.uint8, device=gpu)
      with pytest.MonkeyPatch.context() as mp:
        mp.setattr(ops, '_quantize_workspace', lambda nbytes, device: ws)
        results.append(ops.quantize(x, **kw))
      assert not bool(ws[:4 * n].any())
  results.append(ops.quantize(x, scale=results[0][1], **kw))
  for q, s in results[1:]:
    assert torch.equal(q, results[0][0]) and torch.equal(s, results[0][1])
  want = x.float().abs()
  want = {L.REDUCE_ROWS: lambda: want.reshape(shape[0], -1, group or shape[1], shape[2]).amax(2), L.REDUCE_ALL: lambda: want.amax((1, 2)),
          L.REDUCE_ALL_BATCH: lambda: want.amax().reshape(1)}[reduce]()
  assert torch.equal(results[0][1], (want / 127.5).to(torch.bfloat16).float())


@pytest.mark.parametrize('reduce,shape,group', [
    (L.REDUCE_COLS, (2, 5, 3000), 0), (L.REDUCE_COLS, (1, 9, 20), 4), (L.REDUCE_COLS, (1, 2, 20000), 0), (L.REDUCE_COLS, (1, 30, 96), 32),
    (L.REDUCE_ROWS, (1, 300, 72), 0), (L.REDUCE_ROWS, (2, 256, 130), 64), (L.REDUCE_ALL, (2, 100, 64), 0), (L.REDUCE_ALL_BATCH, (2, 7, 9), 0),
])
@pytest.mark.parametrize('dt', ['bf16', 'i8', 'f32'])
def test_scales_given_as_bf16_elements(gpu, dt, reduce, shape, group):
  """Read where they lie, in every kernel that takes given scales: the same bytes as from a float32 copy of them."""
  x = U.rand(shape, 'f32', seed=3, outliers=True)
  x = torch.from_numpy(x * 20).to({'bf16': torch.bfloat16, 'i8': torch.int8, 'f32': torch.float32}[dt]).to(gpu)
  kw = dict(reduce=reduce, group=group, out_dtype=L.I8, quant_bound=127.5, clip_bound=127.0, scale_dtype=torch.bfloat16,
            compute_dtype=torch.float32 if dt == 'f32' else torch.bfloat16)
  _, s = ops.quantize(x, **kw)
  s = s * 0.5  # clipping, and no maximum of its own to fall back on
  want, _ = ops.quantize(x, scale=s, **kw)
  got, same = ops.quantize(x, scale=s.to(torch.bfloat16), **kw)
  assert torch.equal(got, want) and same.dtype == torch.bfloat16


@pytest.mark.parametrize('reduce,shape,scales', [(L.REDUCE_ALL_BATCH, (3, 300, 70), 1), (L.REDUCE_ALL, (3, 300, 70), 3),
                                                 (L.REDUCE_ROWS, (2, 300, 70), 140), (L.REDUCE_ROWS, (2, 64, 9), 18)])
def test_a_workspace_of_twice_the_bytes_holds_the_counts(gpu, reduce, shape, scales):
  """The smallest workspace with room for the arrival counts: nothing beside it is touched, its first half stays zero."""
  x = U.to_dev(U.rand(shape, 'bf16', seed=5, outliers=True), 'bf16', gpu)
  kw = dict(reduce=reduce, out_dtype=L.I8, quant_bound=127.5, clip_bound=127.0)
  want = ops.quantize(x, **kw)
  buf = torch.full((16 * scales + 64,), 0x5A, dtype=torch.uint8, device=gpu)
  ws = buf[:16 * scales]
  ws[:8 * scales] = 0
  with pytest.MonkeyPatch.context() as mp:
    mp.setattr(ops, '_quantize_workspace', lambda nbytes, device: ws if nbytes == 8 * scales else None)
    for _ in range(3):
      got = ops.quantize(x, **kw)
      assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
      assert not bool(ws[:8 * scales].any()) and bool((buf[16 * scales:] == 0x5A).all())


@pytest.mark.parametrize('reduce', [L.REDUCE_ROWS, L.REDUCE_ALL, L.REDUCE_ALL_BATCH])
@pytest.mark.parametrize('shape', [(511, 7, 24), (512, 7, 24), (513, 64, 9), (600, 65, 16), (520, 130, 127), (3, 64, 1000), (1, 9, 5),
                                   (2, 40, 3000)])
@pytest.mark.parametrize('dt', ['bf16', 'f32'])
def test_scales_of_many_small_entries(gpu, dt, shape, reduce):
  """Entries and groups whose maximum one block finds, in blocks of 4 and of 16 waves, next to ones of several blocks; an
  entry of zeros, one of the largest finite values, a NaN in another."""
  x = torch.randn(shape, generator=torch.Generator().manual_seed(sum(shape)))
  x[0] = 0.0
  x[-1, -1, -1] = torch.finfo(torch.bfloat16).max
  dtype = torch.bfloat16 if dt == 'bf16' else torch.float32
  x = x.to(dtype).to(gpu)
  axes = {L.REDUCE_ROWS: (1,), L.REDUCE_ALL: (1, 2), L.REDUCE_ALL_BATCH: (0, 1, 2)}[reduce]
  for nan in (False, True):
    if nan:
      x[shape[0] // 2, 0, 1] = float('nan')
    want = x.float().abs().amax(axes)
    want = torch.where(want == 0, torch.ones_like(want), want) / 128.0
    kw = dict(reduce=reduce, out_dtype=L.I8, quant_bound=128.0, clip_bound=127.0)
    for _ in range(2):  # (the second call finds the workspace as the first has left it)
      q, s = ops.quantize(x, **kw)
      assert torch.equal(s.reshape(-1).nan_to_num(-1.0), want.to(dtype).float().reshape(-1).nan_to_num(-1.0))
    if not nan:
      given, _ = ops.quantize(x, scale=s, **kw)
      assert torch.equal(q, given)


@pytest.mark.parametrize('rows,cols', [(8128, 512), (8192, 512), (8193, 1024), (16384, 1024), (16385, 1024)])
@pytest.mark.parametrize('dt,prescaled', [('bf16', False), ('bf16', True), ('f32', False), ('i8', False)])
def test_column_scales_on_both_sides_of_the_fold(gpu, dt, prescaled, rows, cols):
  """Blocks of 64 rows x 512 columns: 127 to 514, with the launch for the scales and without it."""
  x = torch.randn((1, rows, cols), generator=torch.Generator().manual_seed(rows)) * 20
  x = {'bf16': x.to(torch.bfloat16), 'f32': x, 'i8': x.to(torch.int8)}[dt].to(gpu)
  compute = torch.float32 if dt == 'f32' else torch.bfloat16
  kw, want = {}, x.to(compute).float()
  if prescaled:
    ps = torch.exp2(torch.arange(rows, device=gpu) % 5 - 2.0)  # powers of two: the products are exact
    kw, want = dict(prescale=ps, prescale_mode=L.PRESCALE_PER_ROW), want * ps[None, :, None]
  q, s = ops.quantize(x, reduce=L.REDUCE_ROWS, compute_dtype=compute, out_dtype=L.I8, quant_bound=128.0, clip_bound=127.0, **kw)
  assert torch.equal(s, (want.abs().amax(1, keepdim=True) / 128.0).to(compute).float())
  assert torch.equal(ops.quantize(x, reduce=L.REDUCE_ROWS, compute_dtype=compute, out_dtype=L.I8, quant_bound=128.0, clip_bound=127.0,
                                  scale=s, **kw)[0], q)


@pytest.mark.parametrize('batch,rows,cols', [(1, 8, 8), (1, 15, 40), (2, 16, 9), (3, 17, 130), (1, 129, 1024), (1, 2048, 200),
                                             (2, 2049, 72), (1, 4096, 24), (1, 4097, 24), (17, 100, 8200), (1, 128, 64)])
@pytest.mark.parametrize('dt,bits', [('bf16', 8), ('bf16', 4), ('f32', 8)])
def test_columns_in_one_pass(gpu, dt, bits, batch, rows, cols):
  """Fewest and most rows of the kernel that reads a column once, edges of its blocks, special values; the scales alone
  and the quantization with given scales come from other kernels."""
  x = U.rand((batch, rows, cols), dt, seed=rows + cols, outliers=True)
  x[:, :, 1] = 0.0
  x[:, rows - 1, 2], x[:, 0, cols - 1] = np.inf, -np.inf
  q = R.QuantizerCfg(bits=bits)
  qb, cb = U.bounds(q)
  kw = dict(reduce=L.REDUCE_ROWS, out_dtype=U.OUT_DT[bits], quant_bound=qb, clip_bound=cb, transpose_out=True)
  finite = np.isfinite(x).all((0, 1))
  with np.errstate(all='ignore'):
    qt = R.quantize(x, dt, q, [1])
  xt = U.to_dev(x, dt, gpu)
  qg, sg = ops.quantize(xt, **kw)
  np.testing.assert_array_equal(sg.cpu().numpy().reshape(-1), qt.scale[0].reshape(-1))
  np.testing.assert_array_equal(np.swapaxes(qg.cpu().numpy(), -1, -2)[..., finite], qt.qvalue.astype(np.int8)[..., finite])
  assert torch.equal(ops.quantize(xt, scale_only=True, **kw)[1], sg)
  assert torch.equal(ops.quantize(xt, scale=sg, **kw)[0], qg)  # infinite columns too
  if rows % 128 == 0 and cols % 64 == 0 and batch == 1:
    with_maxima, _ = ops.quantize(xt, want_other_axis_absmax=True, **kw)
    assert torch.equal(with_maxima, qg)
  x[0, rows // 2, 0] = np.nan
  assert torch.isnan(ops.quantize(U.to_dev(x, dt, gpu), **kw)[1].reshape(batch, cols)[0, 0])


@pytest.mark.parametrize('reduce,shape', [(L.REDUCE_COLS, (1, 5, 3000)), (L.REDUCE_COLS, (1, 3, 5)), (L.REDUCE_COLS, (2, 2, 20000)),
                                          (L.REDUCE_ROWS, (1, 300, 72)), (L.REDUCE_ALL, (2, 100, 64))])
def test_calibration_alone_gives_the_scales_of_the_quantization(gpu, reduce, shape):
  x = U.to_dev(U.rand(shape, 'bf16', seed=9, outliers=True), 'bf16', gpu)
  kw = dict(reduce=reduce, out_dtype=L.I8, quant_bound=127.5, clip_bound=127.0, want_typed_scale=True)
  _, s, t = ops.quantize(x, **kw)
  q, s1, t1 = ops.quantize(x, scale_only=True, **kw)
  assert q is None and torch.equal(s, s1) and torch.equal(t, t1)
  with pytest.raises(L.AqtxError, match='scale_only'):
    ops.quantize(x, reduce=reduce, out_dtype=L.I8, quant_bound=127.5, clip_bound=127.0, scale_only=True, scale=s)


@pytest.mark.parametrize('partitionable', [False, True])
@pytest.mark.parametrize('num,inner', [(1, 1), (3, 2), (2, 5)])
def test_two_levels_of_key_splits_in_one_call(gpu, num, inner, partitionable):
  key = prng.prng_key(77)
  want = np.stack([prng.split(k, inner, partitionable) for k in prng.split(key, num, partitionable)])
  np.testing.assert_array_equal(ops.prng_split(key, num, partitionable, inner=inner), want)
  dev = torch.from_numpy(key.view(np.int32).copy()).to(gpu)
  got = ops.prng_split(dev, num, partitionable, inner=inner).cpu().numpy().view(np.uint32)
  np.testing.assert_array_equal(got, want)
