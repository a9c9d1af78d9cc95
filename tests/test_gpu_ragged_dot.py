"""Quantized ragged_dot: oracle pins (CPU) and GPU parity, after aqt_ragged_dot_test.py."""
import numpy as np
import pytest
import torch

from oracle import aqt_ref as R
from oracle import numerics as nm
from tests import gpu_util as U


def _args(m, k, n, num_groups, dt, balanced, seed=1234):
  """aqt_ragged_dot_test.py:88-112: uniform [0, 1) operands representable in bf16; random
  group ends drawn with replacement so that empty groups occur."""
  rng = np.random.default_rng(seed)
  lhs = nm.cast(nm.cast(rng.uniform(0, 1, (m, k)).astype(np.float32), 'bf16'), dt)
  rhs = nm.cast(nm.cast(rng.uniform(0, 1, (num_groups, k, n)).astype(np.float32), 'bf16'), dt)
  if balanced:
    sizes = [m // num_groups] * num_groups
  else:
    ends = np.concatenate([np.sort(rng.choice(m, num_groups - 1)), [m]])
    sizes = list(np.diff(np.concatenate([[0], ends])))
  assert sum(sizes) == m
  return lhs, rhs, [int(s) for s in sizes]


@pytest.mark.parametrize('dt', ['bf16', 'f32'])
@pytest.mark.parametrize('balanced', [True, False])
def test_oracle_ragged_dot_close_to_float_and_to_batched_dot_general(dt, balanced):
  """aqt_ragged_dot_test.py:114-153: within rtol 1e-2 (bf16) / 5e-3 (f32) of the float ragged
  dot, and, with equal groups, of the quantized batched dot_general on the reshaped lhs."""
  m, k, n, g = 32, 128, 16, 8
  lhs, rhs, sizes = _args(m, k, n, g, dt, balanced)
  rtol = 1e-2 if dt == 'bf16' else 5e-3
  out, lqt, rqt = R.ragged_dot_fwd(lhs, rhs, dt, sizes, R.config_v4().fwd)
  assert lqt.scale[0].shape == (m, 1) and rqt.scale[0].shape == (1, 1, n)
  want = nm.cast(R.lax_ragged_dot(lhs, rhs, sizes, np.float32), dt)
  np.testing.assert_allclose(out, want, rtol=rtol, atol=1e-5)
  if balanced:
    f = R.dg_fwd(lhs.reshape(g, m // g, k), rhs, dt, (((2,), (1,)), ((0,), (0,))), R.config_v4())
    np.testing.assert_allclose(out, f.out.reshape(m, n), rtol=rtol, atol=1e-5)


def test_oracle_ragged_dot_integer_exact():
  """Small integers quantize without loss when the abs-max is 127: the quantized ragged dot
  is then the exact integer result."""
  rng = np.random.default_rng(0)
  lhs = rng.integers(-127, 128, (12, 16)).astype(np.float32)
  lhs[:, 0] = 127.0
  rhs = rng.integers(-127, 128, (3, 16, 5)).astype(np.float32)
  rhs[0, 0, :] = 127.0
  raw = R.config_v4().fwd
  raw.lhs.preserve_max_val = raw.rhs.preserve_max_val = True  # scale = absmax / 127 = 1
  out, _, _ = R.ragged_dot_fwd(lhs, rhs, 'f32', [5, 0, 7], raw)
  want = np.concatenate([lhs[:5] @ rhs[0], lhs[5:] @ rhs[2]])
  np.testing.assert_array_equal(out, want)


@pytest.mark.gpu
@pytest.mark.parametrize('dt', ['bf16', 'f32'])
@pytest.mark.parametrize('balanced', [True, False])
@pytest.mark.parametrize('shape', [(32, 128, 16, 8), (300, 96, 200, 5), (3000, 256, 520, 6), (66, 72, 40, 3)])
def test_ragged_dot_matches_oracle(gpu, dt, balanced, shape):
  from aqt_amd.v2 import aqt_ragged_dot
  m, k, n, g = shape
  lhs, rhs, sizes = _args(m, k, n, g, dt, balanced)
  want, _, _ = R.ragged_dot_fwd(lhs, rhs, dt, sizes, R.config_v4().fwd)
  L, Rr = U.to_dev(lhs, dt, gpu), U.to_dev(rhs, dt, gpu)
  out = aqt_ragged_dot.ragged_dot(L, Rr, torch.tensor(sizes, dtype=torch.int32, device=gpu))
  assert out.dtype == U.TORCH_DT[dt]
  np.testing.assert_array_equal(out.float().cpu().numpy(), want)
  # group sizes given on the host, rows past the last group stay zero
  short = sizes[:-1] + [max(sizes[-1] - 3, 0)]
  out2 = aqt_ragged_dot.ragged_dot(L, Rr, short)
  covered = sum(short)
  np.testing.assert_array_equal(out2[:covered].float().cpu().numpy(), want[:covered])
  assert (out2[covered:] == 0).all()


@pytest.mark.gpu
def test_ragged_dot_unquantized_and_precision(gpu):
  from aqt_amd.v2 import aqt_ragged_dot
  from aqt_amd.v2 import config
  lhs, rhs, sizes = _args(32, 128, 16, 8, 'f32', False)
  L, Rr = U.to_dev(lhs, 'f32', gpu), U.to_dev(rhs, 'f32', gpu)
  out = aqt_ragged_dot.ragged_dot(L, Rr, sizes, cfg=config.default_unquantized_config())
  np.testing.assert_allclose(out.cpu().numpy(), R.lax_ragged_dot(lhs, rhs, sizes, np.float32), rtol=1e-5)
  with pytest.raises(AssertionError):  # aqt_ragged_dot_test.py:155-166
    aqt_ragged_dot.ragged_dot(L, Rr, sizes, precision='highest')


@pytest.mark.gpu
def test_ragged_gemm_one_launch_against_integer_reference(gpu):
  """The grouped launch itself: groups that span several 256-row tiles, start in the middle of
  a tile, are empty, or leave the last rows uncovered; raw int32 accumulators."""
  from aqt_amd import ops
  rng = np.random.default_rng(3)
  m, k, n = 2000, 320, 300
  sizes = [700, 0, 257, 1, 511, 300]  # sums to 1769 < m
  a = rng.integers(-127, 128, (m, k)).astype(np.int8)
  b = rng.integers(-127, 128, (len(sizes), n, k)).astype(np.int8)
  offs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
  out = ops.gemm(torch.from_numpy(a).to(gpu)[None], torch.from_numpy(b).to(gpu), row_scale=None, col_scale=None,
                 out_dtype=torch.int32, group_offsets=torch.from_numpy(offs).to(gpu))[0].cpu().numpy()
  want = np.zeros((m, n), np.int64)
  for g, (lo, hi) in enumerate(zip(offs[:-1], offs[1:])):
    want[lo:hi] = a[lo:hi].astype(np.int64) @ b[g].astype(np.int64).T
  np.testing.assert_array_equal(out, want)


@pytest.mark.gpu
@pytest.mark.parametrize('groups', [1, 3, 64, 65, 200])
@pytest.mark.parametrize('left', [0, 1, 300, 4000])
def test_ragged_gemm_prepares_offsets_and_zeros_from_the_sizes(gpu, groups, left):
  """Sizes with empty groups, `left` rows behind the last group (negative room: sizes that overrun the rows are cut at
  m), int32 and bf16 outputs, one row of column scales for all groups: as the offsets made on the host give it."""
  from aqt_amd import ops
  rng = np.random.default_rng(groups + left)
  sizes = rng.integers(0, 40, groups) * rng.integers(0, 2, groups)
  sizes[-1] += 1
  total = int(sizes.sum())
  k, n = 64, 33
  for m in (total + left, max(1, total - 5)):
    a = torch.from_numpy(rng.integers(-127, 128, (1, m, k)).astype(np.int8)).to(gpu)
    b = torch.from_numpy(rng.integers(-127, 128, (groups, n, k)).astype(np.int8)).to(gpu)
    offs = torch.from_numpy(np.minimum(np.concatenate([[0], np.cumsum(sizes)]), m).astype(np.int32)).to(gpu)
    ones, cs = torch.ones((1, m), device=gpu), torch.rand((1, n), device=gpu)
    dev_sizes = ops.ragged_sizes(torch.from_numpy(sizes), gpu)
    junk = torch.full((2 * m * n * 4,), 0x7F, dtype=torch.uint8, device=gpu)  # what a freed block would leave behind
    del junk
    got = ops.gemm(a, b, row_scale=None, col_scale=None, out_dtype=torch.int32, group_sizes=dev_sizes)
    want = ops.gemm(a, b, row_scale=None, col_scale=None, out_dtype=torch.int32, group_offsets=offs)
    assert torch.equal(got, want) and not bool(got[0, min(total, m):].any())
    got = ops.gemm(a, b, row_scale=ones, col_scale=cs, out_dtype=torch.bfloat16, group_sizes=dev_sizes)
    want = ops.gemm(a, b, row_scale=ones, col_scale=cs.expand(groups, n).contiguous(), out_dtype=torch.bfloat16, group_offsets=offs)
    assert torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize('groups', [63, 64, 65, 128, 129, 200, 513, 1500, 2049])
def test_ragged_gemm_of_many_groups_against_integer_reference(gpu, groups):
  """Groups on both sides of the 64, 512 and 2048 looked up or summed at a time, some of several 256-row tiles, some empty, n
  of two tiles: every group meets its own B.  Sizes and offsets made on the host, on the device and by the contraction itself."""
  from aqt_amd import ops
  rng = np.random.default_rng(groups)
  sizes = rng.integers(0, max(2, 3000 // groups), groups) * rng.integers(0, 2, groups)
  for g, rows in ((2, 600), (61, 257), (62, 512), (64, 300), (65, 1), (511, 257), (512, 300), (groups - 1, 513)):
    if g < groups:
      sizes[g] = rows
  m, k, n = int(sizes.sum()) + 7, 32, 300
  a = rng.integers(-127, 128, (m, k)).astype(np.int8)
  b = rng.integers(-127, 128, (groups, n, k)).astype(np.int8)
  want, at = np.zeros((m, n)), 0
  for g, rows in enumerate(sizes):
    want[at:at + rows] = a[at:at + rows].astype(np.float64) @ b[g].astype(np.float64).T
    at += rows
  ta, tb = torch.from_numpy(a).to(gpu)[None], torch.from_numpy(b).to(gpu)
  on_device = torch.from_numpy(sizes.astype(np.int32)).to(gpu)
  for kw in (dict(group_sizes=ops.ragged_sizes(sizes.tolist(), gpu)), dict(group_offsets=ops.ragged_offsets(sizes.tolist(), m, gpu)),
             dict(group_offsets=ops.ragged_offsets(on_device, m, gpu))):
    out = ops.gemm(ta, tb, row_scale=None, col_scale=None, out_dtype=torch.int32, **kw)[0]
    np.testing.assert_array_equal(out.cpu().numpy(), want)


@pytest.mark.gpu
@pytest.mark.parametrize('m,groups', [(5, 2100), (1, 129), (300, 1000)])
def test_ragged_gemm_of_more_groups_than_rows(gpu, m, groups):
  from aqt_amd import ops
  rng = np.random.default_rng(m)
  sizes = np.zeros(groups, np.int64)
  np.add.at(sizes, rng.integers(0, groups, m), 1)
  a = rng.integers(-127, 128, (m, 16)).astype(np.int8)
  b = rng.integers(-127, 128, (groups, 24, 16)).astype(np.int8)
  owner = np.repeat(np.arange(groups), sizes)
  want = np.einsum('mk,mnk->mn', a.astype(np.int64), b[owner].astype(np.int64))
  ta, tb = torch.from_numpy(a).to(gpu)[None], torch.from_numpy(b).to(gpu)
  out = ops.gemm(ta, tb, row_scale=None, col_scale=None, out_dtype=torch.int32, group_sizes=ops.ragged_sizes(sizes.tolist(), gpu))[0]
  np.testing.assert_array_equal(out.cpu().numpy(), want)
  empty = ops.gemm(ta, tb, row_scale=None, col_scale=None, out_dtype=torch.int32, group_sizes=ops.ragged_sizes([0] * groups, gpu))[0]
  assert not bool(empty.any())
