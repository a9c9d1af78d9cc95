"""GPU parity: aqtx_gemm_i8 against exact integer arithmetic and the oracle's dequant."""
import numpy as np
import pytest
import torch

from aqt_amd import _lib as L
from aqt_amd import ops
from oracle import aqt_ref as R
from oracle import numerics as nm
from tests import gpu_util as U

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[4, 8, 16, 128, 129, 130, 131, 132, 133, 134, 0],
                ids=['waves4', 'waves8', 'persistent', 'tiles128', 'ring128', 'ring64x128', 'ring64', 'ring128x256', 'ring64pair', 'ring64x128pair', 'auto'])
def waves(request, monkeypatch):
  """Both workgroup shapes of the 256 x 256 int8 MFMA kernel, the kernel for few output tiles on each of its
  tile shapes and schedules, and the library's own choice (these shapes have few output tiles: the smaller
  tiles, with k in slices where it is long)."""
  monkeypatch.setattr(ops, 'GEMM_TUNING', request.param)
  return request.param


@pytest.fixture(params=[(8, L.ACC_FAST), (0, L.ACC_FAST), (0, L.ACC_F32)], ids=['tiles256', 'auto', 'f32sums'])
def tiles(request, monkeypatch):
  """fp8 operands: the 256 x 256 kernel, the library's own choice (the 128 x 128 kernel for these shapes), and
  the contraction through bf16 with float32-like sums (aqtx_gemm_plan.accumulate = AQTX_ACC_F32)."""
  monkeypatch.setattr(ops, 'GEMM_TUNING', request.param[0])
  monkeypatch.setattr(ops, 'FP8_ACCUMULATE', request.param[1])
  return request.param


def _ints(shape, seed):
  return np.random.default_rng(seed).integers(-127, 128, size=shape).astype(np.int8)


def _ref_acc(a, b):
  return np.einsum('bmk,bnk->bmn', a.astype(np.float64), b.astype(np.float64)).astype(np.int64)


SHAPES = [
    (1, 256, 256, 128), (1, 512, 768, 384), (1, 300, 520, 144), (1, 64, 64, 16), (3, 130, 70, 48),
    (1, 17, 9, 50), (2, 5, 3, 7), (1, 1, 4096, 4096), (1, 1024, 512, 1040),
]


@pytest.mark.parametrize('batch,m,n,k', SHAPES)
def test_raw_accumulators(gpu, waves, batch, m, n, k):
  a, b = _ints((batch, m, k), 1), _ints((batch, n, k), 2)
  c = ops.gemm(torch.from_numpy(a).to(gpu), torch.from_numpy(b).to(gpu), row_scale=None,
               col_scale=None, out_dtype=torch.int32)
  np.testing.assert_array_equal(c.cpu().numpy().astype(np.int64), _ref_acc(a, b))


@pytest.mark.parametrize('out', ['bf16', 'f32'])
@pytest.mark.parametrize('sdt', ['bf16', 'f32'])
@pytest.mark.parametrize('order', [L.SCALE_ROW_THEN_COL, L.SCALE_COL_THEN_ROW])
@pytest.mark.parametrize('batch,m,n,k', [(1, 256, 512, 4096), (2, 100, 72, 160), (1, 33, 20, 23)])
def test_dequant_epilogue(gpu, waves, batch, m, n, k, order, sdt, out):
  if out == 'f32' and sdt == 'bf16':
    pytest.skip('scale dtype never narrower than the dequant dtype in the reference')
  a, b = _ints((batch, m, k), 3), _ints((batch, n, k), 4)
  rs = nm.cast(np.abs(U.rand((batch, m), 'f32', 5, 0.03)) + np.float32(1e-3), sdt)
  cs = nm.cast(np.abs(U.rand((batch, n), 'f32', 6, 6e-4)) + np.float32(1e-5), sdt)
  acc = _ref_acc(a, b).astype(np.int32)
  s1, s2 = (rs[:, :, None], cs[:, None, :])
  if order == L.SCALE_COL_THEN_ROW:
    s1, s2 = s2, s1
  want = R.dequant(R.QTensor(acc, 'i32', [s1, s2], sdt, out))
  c, acc_got = ops.gemm(torch.from_numpy(a).to(gpu), torch.from_numpy(b).to(gpu),
                        row_scale=torch.from_numpy(rs).to(gpu), col_scale=torch.from_numpy(cs).to(gpu),
                        out_dtype=U.TORCH_DT[out], scale_dtype=U.TORCH_DT[sdt], scale_order=order,
                        want_acc=True)
  np.testing.assert_array_equal(acc_got.cpu().numpy(), acc)
  np.testing.assert_array_equal(c.float().cpu().numpy(), want)


@pytest.mark.parametrize('rdt,cdt', [('bf16', 'f32'), ('f32', 'bf16')])
@pytest.mark.parametrize('order', [L.SCALE_ROW_THEN_COL, L.SCALE_COL_THEN_ROW])
@pytest.mark.parametrize('batch,m,n,k', [(1, 256, 512, 512), (2, 100, 72, 160)])
def test_dequant_epilogue_mixed_scale_dtypes(gpu, tiles, batch, m, n, k, order, rdt, cdt):
  """A bf16 and an f32 scale: only a first product of two bf16 values is rounded to bf16."""
  a, b = _ints((batch, m, k), 3), _ints((batch, n, k), 4)
  rs = nm.cast(np.abs(U.rand((batch, m), 'f32', 5, 0.03)) + np.float32(1e-3), rdt)
  cs = nm.cast(np.abs(U.rand((batch, n), 'f32', 6, 6e-4)) + np.float32(1e-5), cdt)
  acc = _ref_acc(a, b).astype(np.int32)
  scales, sdts = [rs[:, :, None], cs[:, None, :]], [rdt, cdt]
  if order == L.SCALE_COL_THEN_ROW:
    scales, sdts = scales[::-1], sdts[::-1]
  want = R.dequant(R.QTensor(acc, 'i32', scales, None, 'bf16', scale_dtypes=sdts))
  c = ops.gemm(torch.from_numpy(a).to(gpu), torch.from_numpy(b).to(gpu),
               row_scale=torch.from_numpy(rs).to(gpu), col_scale=torch.from_numpy(cs).to(gpu),
               out_dtype=torch.bfloat16, row_scale_dtype=U.TORCH_DT[rdt], col_scale_dtype=U.TORCH_DT[cdt],
               scale_order=order)
  np.testing.assert_array_equal(c.float().cpu().numpy(), want)


def test_large_accumulators_round_like_xla(gpu, waves):
  """|acc| > 2**24: int32 -> f32 -> bf16 double rounding is part of the contract."""
  k = 4096
  a = np.full((1, 256, k), 127, np.int8)
  b = np.full((1, 256, k), 127, np.int8)
  b[0, ::2, : k // 3] = -126
  a[0, 1::3, 5:900] = 113
  acc = _ref_acc(a, b).astype(np.int32)
  assert np.abs(acc).max() > 2 ** 24
  want = nm.int32_to_float(acc, 'bf16')
  c = ops.gemm(torch.from_numpy(a).to(gpu), torch.from_numpy(b).to(gpu), row_scale=None,
               col_scale=None, out_dtype=torch.bfloat16)
  np.testing.assert_array_equal(c.float().cpu().numpy(), want)


# ---- k in slices (the 128 x 128 kernel writes int32 slabs, a second kernel adds and dequantizes) ----
@pytest.mark.parametrize('slices', [2, 3, 7])
@pytest.mark.parametrize('out,sdt,order', [('bf16', 'bf16', L.SCALE_ROW_THEN_COL), ('bf16', 'f32', L.SCALE_COL_THEN_ROW),
                                           ('f32', 'f32', L.SCALE_ROW_THEN_COL), ('i32', None, None)])
@pytest.mark.parametrize('batch,m,n,k', [(1, 128, 256, 4096), (2, 100, 72, 1200), (1, 33, 21, 528), (1, 300, 130, 2064)])
def test_k_slices_give_the_same_bits(gpu, batch, m, n, k, out, sdt, order, slices):
  a, b = _ints((batch, m, k), 31), _ints((batch, n, k), 32)
  at, bt = torch.from_numpy(a).to(gpu), torch.from_numpy(b).to(gpu)
  acc = _ref_acc(a, b).astype(np.int32)
  if out == 'i32':
    c = ops.gemm(at, bt, row_scale=None, col_scale=None, out_dtype=torch.int32, k_split=slices)
    np.testing.assert_array_equal(c.cpu().numpy(), acc)
    return
  rs = nm.cast(np.abs(U.rand((batch, m), 'f32', 5, 0.03)) + np.float32(1e-3), sdt)
  cs = nm.cast(np.abs(U.rand((batch, n), 'f32', 6, 6e-4)) + np.float32(1e-5), sdt)
  s1, s2 = (rs[:, :, None], cs[:, None, :])
  if order == L.SCALE_COL_THEN_ROW:
    s1, s2 = s2, s1
  want = R.dequant(R.QTensor(acc, 'i32', [s1, s2], sdt, out))
  kw = dict(row_scale=torch.from_numpy(rs).to(gpu), col_scale=torch.from_numpy(cs).to(gpu),
            out_dtype=U.TORCH_DT[out], scale_dtype=U.TORCH_DT[sdt], scale_order=order)
  c, acc_got = ops.gemm(at, bt, want_acc=True, k_split=slices, **kw)
  np.testing.assert_array_equal(acc_got.cpu().numpy(), acc)
  np.testing.assert_array_equal(c.float().cpu().numpy(), want)
  assert torch.equal(c, ops.gemm(at, bt, k_split=1, **kw))


def test_k_slices_chosen_by_the_library(gpu):
  """A long k over few output tiles is cut by default; the plan's answer and the result agree with k_split = 1."""
  import ctypes
  m, n, k = 128, 512, 14336
  a, b = _ints((1, m, k), 33), _ints((1, n, k), 34)
  at, bt = torch.from_numpy(a).to(gpu), torch.from_numpy(b).to(gpu)
  plan = L.GemmPlan()
  plan.batch, plan.m, plan.n, plan.k, plan.lda, plan.ldb, plan.ldc = 1, m, n, k, k, k, n
  plan.a_dtype = plan.b_dtype = L.I8
  assert L.lib().aqtx_gemm_i8_k_slices(ctypes.byref(plan)) == 8
  plan.k_split = 1
  assert L.lib().aqtx_gemm_i8_k_slices(ctypes.byref(plan)) == 1
  plan.k_split, plan.m, plan.n = 0, 8192, 14336  # many tiles: never
  assert L.lib().aqtx_gemm_i8_k_slices(ctypes.byref(plan)) == 1
  rs = torch.rand(1, m, device=gpu) * 0.01 + 1e-3
  cs = torch.rand(1, n, device=gpu) * 1e-3 + 1e-5
  kw = dict(row_scale=rs, col_scale=cs, out_dtype=torch.bfloat16)
  got, want = ops.gemm(at, bt, **kw), ops.gemm(at, bt, k_split=1, **kw)
  assert torch.equal(got, want)
  np.testing.assert_array_equal(ops.gemm(at, bt, row_scale=None, col_scale=None, out_dtype=torch.int32).cpu().numpy(),
                                _ref_acc(a, b))


def test_k_slices_packed_int4_b(gpu):
  a = _ints((1, 96, 2048), 35)
  b = np.random.default_rng(36).integers(-8, 8, size=(1, 200, 2048)).astype(np.int8)
  at, bt = torch.from_numpy(a).to(gpu), torch.from_numpy(b).to(gpu)
  bp = ops.pack_i4(bt.reshape(200, 2048)).reshape(1, 200, 1024)
  rs = torch.rand(1, 96, device=gpu) * 0.01 + 1e-3
  cs = torch.rand(1, 200, device=gpu) * 1e-3 + 1e-5
  kw = dict(row_scale=rs, col_scale=cs, out_dtype=torch.bfloat16, want_acc=True)
  c0, acc0 = ops.gemm(at, bt, b_dtype=L.I4, k_split=1, **kw)
  for a_in, order in ((at, L.K_NATURAL), (torch.from_numpy(_even_odd8(a)).to(gpu), L.K_EVEN_ODD8)):
    c1, acc1 = ops.gemm(a_in, bp, b_dtype=L.I4P, a_k_order=order, k_split=4, **kw)
    assert torch.equal(c0, c1) and torch.equal(acc0, acc1)
  np.testing.assert_array_equal(acc0.cpu().numpy(), _ref_acc(a, b))


def test_k_slices_rejected_where_unsupported(gpu):
  a = torch.zeros((1, 64, 512), dtype=torch.int8, device=gpu)
  b = torch.zeros((1, 64, 512), dtype=torch.int8, device=gpu)
  with pytest.raises(RuntimeError, match='k_split must be in 0..64'):
    ops.gemm(a, b, row_scale=None, col_scale=None, out_dtype=torch.int32, k_split=65)
  offs = torch.tensor([0, 64], dtype=torch.int32, device=gpu)
  with pytest.raises(RuntimeError, match='k_split > 1 with ragged batches'):
    ops.gemm(a, b, row_scale=None, col_scale=None, out_dtype=torch.int32, group_offsets=offs, k_split=2)


# ---- every tile shape and schedule of the kernel for few output tiles gives the bits of the large tiles ----
@pytest.mark.parametrize('b_kind', ['rows', 'fragments', 'packed', 'packed_fragments'])
@pytest.mark.parametrize('batch,m,n,k,out,sdt', [
    (1, 200, 328, 4160, 'bf16', 'bf16'),   # ragged m and n, a k tail of 64
    (1, 130, 201, 1056, 'bf16', 'f32'),    # rows of C not 16-byte aligned: the stores straight from the accumulators
    (2, 129, 136, 384, 'f32', 'f32'),      # batches, three stages: as many as the ring has buffers
    (1, 64, 72, 128, 'bf16', 'bf16'),      # one stage
    (1, 512, 1024, 256, 'i32', None),      # raw sums, two stages
    (1, 96, 4096, 2048, 'f32', 'f32'),
])
def test_few_tiles_kernel_shapes_give_the_same_bits(gpu, monkeypatch, batch, m, n, k, out, sdt, b_kind):
  """plan->tuning 128 (128 x 128 tiles, plain schedule) and 129 .. 134 (the ring schedule on 128 x 128,
  64 x 128, 64 x 64 and 128 x 256 tiles and, with a barrier per two stages, on 64 x 64 and 64 x 128) against the 256 x 256 kernel on the same operands: integer sums, the same
  epilogue arithmetic, so bit for bit, outputs and raw accumulators, for rows and the fragment order of b,
  int8 and packed int4."""
  packed, frag = b_kind.startswith('packed'), b_kind.endswith('fragments')
  if frag and (batch > 1 or out == 'i32'):
    pytest.skip('the fragment order holds one weight, whose column count the binding reads off the column scale')
  torch.manual_seed(11)
  lo, hi = (-8, 8) if packed else (-127, 128)
  a = torch.randint(-127, 128, (batch, m, k), dtype=torch.int8, device=gpu)
  b = torch.randint(lo, hi, (batch, n, k), dtype=torch.int8, device=gpu)
  b_arg, b_dtype = b, L.I8
  if packed:
    b_arg, b_dtype = ops.pack_i4(b.reshape(batch * n, k)).reshape(batch, n, k // 2), L.I4P
  kw = dict(b_dtype=b_dtype, want_acc=True, k_split=1)
  if out == 'i32':
    kw.update(row_scale=None, col_scale=None, out_dtype=torch.int32)
  else:
    kw.update(row_scale=torch.rand(batch, m, device=gpu) + 0.5, col_scale=torch.rand(batch, n, device=gpu) * 0.01 + 1e-4,
              out_dtype=U.TORCH_DT[out], scale_dtype=U.TORCH_DT[sdt])
  monkeypatch.setattr(ops, 'GEMM_TUNING', 8)
  want, want_acc = ops.gemm(a, b_arg, **kw)
  ref = torch.einsum('bmk,bnk->bmn', a.cpu().to(torch.int64), b.cpu().to(torch.int64)).to(torch.int32)
  assert torch.equal(want_acc.cpu(), ref)
  if frag:
    b_arg, kw['b_layout'] = ops.tile_weight(b_arg[0].contiguous(), b_dtype), L.W_FRAGMENTS
  for tuning in (128, 129, 130, 131, 132, 133, 134, 0):
    monkeypatch.setattr(ops, 'GEMM_TUNING', tuning)
    got, got_acc = ops.gemm(a, b_arg, **kw)
    alone = ops.gemm(a, b_arg, **dict(kw, want_acc=False))  # without the copy of the sums the tile leaves through LDS
    bits = torch.int16 if out == 'bf16' else torch.int32
    assert torch.equal(got_acc, want_acc), tuning
    assert torch.equal(got.view(bits), want.view(bits)), tuning
    assert torch.equal(alone.view(bits), want.view(bits)), tuning
  # k in slices on request: on the plain schedule and on the ring shapes that take slices (unpacked operands)
  for tuning in (0, 128, 129, 133, 134):
    monkeypatch.setattr(ops, 'GEMM_TUNING', tuning)
    got, got_acc = ops.gemm(a, b_arg, **dict(kw, k_split=3))
    assert torch.equal(got_acc, want_acc), ('slices', tuning)
    assert torch.equal(got.view(bits), want.view(bits)), ('slices', tuning)


@pytest.mark.gpu
def test_library_choice_on_random_shapes_gives_the_bits_of_the_large_tiles(gpu, monkeypatch):
  """Forty seeded shapes with m up to 700, n up to 4500 and k up to 16500 (ragged in all three, so that the tile
  shape, the slices of k and the tails the library picks vary), b as rows and in fragment order: outputs and raw
  sums equal those of the 256 x 256 kernel bit for bit."""
  rng = np.random.default_rng(20250607)
  for case in range(40):
    m = int(rng.integers(65, 700))
    n = int(rng.choice([rng.integers(16, 600), rng.integers(600, 4500)]))
    k = int(rng.choice([rng.integers(1, 40) * 16, rng.integers(40, 520) * 32]))
    torch.manual_seed(case)
    a = torch.randint(-127, 128, (1, m, k), dtype=torch.int8, device=gpu)
    b = torch.randint(-127, 128, (1, n, k), dtype=torch.int8, device=gpu)
    kw = dict(row_scale=torch.rand(1, m, device=gpu) + 0.5, col_scale=torch.rand(1, n, device=gpu) * 0.01 + 1e-4,
              out_dtype=torch.bfloat16, want_acc=True)
    monkeypatch.setattr(ops, 'GEMM_TUNING', 8)
    want, want_acc = ops.gemm(a, b, **kw)
    monkeypatch.setattr(ops, 'GEMM_TUNING', 0)
    got, got_acc = ops.gemm(a, b, **kw)
    assert torch.equal(got_acc, want_acc) and torch.equal(got.view(torch.int16), want.view(torch.int16)), (case, m, n, k, 'rows')
    frags = ops.tile_weight(b[0].contiguous(), L.I8)
    got, got_acc = ops.gemm(a, frags, b_layout=L.W_FRAGMENTS, **kw)
    assert torch.equal(got_acc, want_acc) and torch.equal(got.view(torch.int16), want.view(torch.int16)), (case, m, n, k, 'fragments')


# ---- packed int4 B (two values per byte, unpacked in registers) ---------------------------------
def _even_odd8(a):
  g = a.reshape(a.shape[:-1] + (a.shape[-1] // 8, 8))
  return np.ascontiguousarray(g[..., [0, 2, 4, 6, 1, 3, 5, 7]].reshape(a.shape))


@pytest.mark.parametrize('k_order', [L.K_NATURAL, L.K_EVEN_ODD8])
@pytest.mark.parametrize('batch,m,n,k', [(1, 256, 256, 256), (1, 512, 768, 384), (1, 300, 520, 160), (1, 64, 64, 32),
                                           (3, 130, 70, 96), (1, 17, 9, 64), (1, 1024, 512, 1056), (1, 100, 4096, 4096)])
def test_packed_int4_b_raw_accumulators(gpu, tiles, batch, m, n, k, k_order):
  """int32 output and the copy of the accumulators: exact, whatever the byte order of A."""
  a = _ints((batch, m, k), 11)
  b = np.random.default_rng(12).integers(-8, 8, size=(batch, n, k)).astype(np.int8)
  bp = ops.pack_i4(torch.from_numpy(b).to(gpu).reshape(batch * n, k)).reshape(batch, n, k // 2)
  at = torch.from_numpy(_even_odd8(a) if k_order == L.K_EVEN_ODD8 else a).to(gpu)
  c = ops.gemm(at, bp, row_scale=None, col_scale=None, out_dtype=torch.int32, b_dtype=L.I4P, a_k_order=k_order)
  np.testing.assert_array_equal(c.cpu().numpy().astype(np.int64), _ref_acc(a, b))


@pytest.mark.parametrize('out,rdt,cdt', [('bf16', 'bf16', 'bf16'), ('bf16', 'bf16', 'f32'), ('bf16', 'f32', 'f32'), ('f32', 'f32', 'f32')])
@pytest.mark.parametrize('batch,m,n,k', [(1, 256, 512, 4096), (2, 100, 72, 160), (1, 33, 20, 32)])
def test_packed_int4_b_dequant_epilogue(gpu, tiles, batch, m, n, k, out, rdt, cdt):
  """Same bits as the same contraction with the int4 values in int8 bytes, and as the oracle's dequant."""
  a = _ints((batch, m, k), 13)
  b = np.random.default_rng(14).integers(-8, 8, size=(batch, n, k)).astype(np.int8)
  rs = nm.cast(np.abs(U.rand((batch, m), 'f32', 5, 0.03)) + np.float32(1e-3), rdt)
  cs = nm.cast(np.abs(U.rand((batch, n), 'f32', 6, 6e-4)) + np.float32(1e-5), cdt)
  acc = _ref_acc(a, b).astype(np.int32)
  want = R.dequant(R.QTensor(acc, 'i32', [rs[:, :, None], cs[:, None, :]], None, out, scale_dtypes=[rdt, cdt]))
  kw = dict(row_scale=torch.from_numpy(rs).to(gpu), col_scale=torch.from_numpy(cs).to(gpu), out_dtype=U.TORCH_DT[out],
            row_scale_dtype=U.TORCH_DT[rdt], col_scale_dtype=U.TORCH_DT[cdt], want_acc=True)
  bt = torch.from_numpy(b).to(gpu)
  bp = ops.pack_i4(bt.reshape(batch * n, k)).reshape(batch, n, k // 2)
  c0, acc0 = ops.gemm(torch.from_numpy(a).to(gpu), bt, b_dtype=L.I4, **kw)
  c1, acc1 = ops.gemm(torch.from_numpy(a).to(gpu), bp, b_dtype=L.I4P, **kw)
  c2, acc2 = ops.gemm(torch.from_numpy(_even_odd8(a)).to(gpu), bp, b_dtype=L.I4P, a_k_order=L.K_EVEN_ODD8, **kw)
  np.testing.assert_array_equal(acc1.cpu().numpy(), acc)
  np.testing.assert_array_equal(acc2.cpu().numpy(), acc)
  np.testing.assert_array_equal(c1.float().cpu().numpy(), want)
  assert torch.equal(c0, c1) and torch.equal(c1, c2)


def test_packed_int4_b_rejected_where_unsupported(gpu):
  a = torch.zeros((1, 64, 64), dtype=torch.int8, device=gpu)
  bp = torch.zeros((1, 64, 32), dtype=torch.uint8, device=gpu)
  ones = torch.ones((1, 64), device=gpu)
  with pytest.raises(RuntimeError, match='ROW_THEN_COL'):
    ops.gemm(a, bp, row_scale=ones, col_scale=ones, out_dtype=torch.bfloat16, b_dtype=L.I4P, scale_order=L.SCALE_COL_THEN_ROW)
  with pytest.raises(RuntimeError, match='a_k_order'):
    ops.gemm(a, a, row_scale=ones, col_scale=ones, out_dtype=torch.bfloat16, a_k_order=L.K_EVEN_ODD8)
  with pytest.raises(RuntimeError, match='multiple of 32'):
    ops.gemm(a[:, :, :48].contiguous(), bp[:, :, :24].contiguous(), row_scale=ones, col_scale=ones,
             out_dtype=torch.bfloat16, b_dtype=L.I4P)


# ---- fp8 ---------------------------------------------------------------------------------
_FP8_TORCH = {'e4m3': torch.float8_e4m3fn, 'e5m2': torch.float8_e5m2}
_FP8_AQTX = {'e4m3': L.E4M3, 'e5m2': L.E5M2}


def _fp8_small_ints(shape, seed, kind):
  """Bytes of small integers (exact in both fp8 formats) and their float values."""
  v = np.random.default_rng(seed).integers(-4, 5, size=shape).astype(np.float32)
  b = torch.from_numpy(v).to(_FP8_TORCH[kind]).view(torch.uint8)
  return b, v


def _fp8_random_bytes(shape, seed, kind):
  """Random finite fp8 bit patterns (|x| <= 16 so that sums stay far from overflow)."""
  rng = np.random.default_rng(seed)
  allb = np.arange(256, dtype=np.uint8)
  vals = U.fp8_bytes_to_float(allb, kind)
  ok = allb[np.isfinite(vals) & (np.abs(vals) <= 16.0)]
  b = ok[rng.integers(0, len(ok), size=shape)]
  return torch.from_numpy(b), U.fp8_bytes_to_float(b, kind)


FP8_SHAPES = [(1, 256, 256, 256), (1, 300, 520, 144), (2, 130, 70, 48), (1, 17, 9, 50), (1, 512, 256, 4096)]
