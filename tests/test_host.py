"""CPU tests of the product's host logic and of the C ABI library itself
(loads, exports every declared symbol, host-only entry points).  No GPU
compute is called here."""
import ctypes
import os
import re

import numpy as np
import pytest
import torch

from conftest import ROOT
from oracle import grid as ogrid
from oracle import heston as oheston
from oracle import sobol as osobol
from tqf import _native
from tqf.math.random import sobol as tsobol
from tqf.models import utils
from tqf.models.heston import qe_step_coefficients


def _header_symbols():
  text = open(os.path.join(ROOT, 'include', 'tqf.h')).read()
  return sorted(set(re.findall(r'\b(tqf_[a-z0-9_]+)\s*\(', text)))


def test_library_exports_every_declared_symbol():
  lib = _native.lib()
  syms = _header_symbols()
  assert len(syms) >= 8
  for s in syms:
    assert hasattr(lib, s), s
  # the ctypes table binds exactly the declared entry points
  assert sorted(_native.exported_symbols()) == syms
  assert lib.tqf_version() >= 1


def test_error_path_maps_to_value_error():
  m = np.zeros((2, 32), np.uint32)
  poly = np.zeros(1, np.int64)
  with pytest.raises(ValueError, match='Dimension must be greater'):
    _native.call('tqf_sobol_direction_numbers',
                 poly.ctypes.data_as(ctypes.c_void_p),
                 poly.ctypes.data_as(ctypes.c_void_p), ctypes.c_int32(1),
                 ctypes.c_int32(0), m.ctypes.data_as(ctypes.c_void_p))


@pytest.mark.parametrize('nd', [0, -1, 33])
def test_exact_gbm_refuses_sobol_digits_out_of_range(nd):
  # the float32 transform shifts by 32 - nd; checked before any launch, so
  # also without a GPU (the addresses are not read)
  host = np.zeros(64, np.float64)
  addr = host.ctypes.data
  g = _native.Gbm(dim=1, drift=addr, vol=addr, s0=addr)
  grid = _native.Grid(dt=addr, sqrt_dt=addr, t_next=addr, slot=addr,
                      n_steps=1, n_slots=1, init_slot=-1, n_rng_steps=1)
  r = _native.Rng(kind=_native.RNG_SOBOL, sobol_v=addr, sobol_lo=addr,
                  sobol_nd=nd, sobol_ndims=1)
  with pytest.raises(ValueError, match='bad Sobol digits'):
    _native.call('tqf_gbm_exact', ctypes.byref(g), ctypes.byref(grid),
                 ctypes.byref(r), ctypes.c_int32(1), ctypes.c_void_p(addr),
                 ctypes.c_int64(1), ctypes.c_int32(_native.TQF_F32), None)


@pytest.mark.parametrize('items,blocks,steps', [(1, 1, 1), (3, 7, 16),
                                                (128, 2, 17), (255, 64, 500)])
def test_batch_workspace_is_what_the_kernel_carves(items, blocks, steps):
  # item sums up to the next 256 bytes, the counter's 256, and one float per
  # checkpoint, thread and block: the sweep keeps the variance only
  sums = (items * 16 * 8 + 255) // 256 * 256
  need = sums + 256 + blocks * 256 * ((steps + 15) // 16) * 4
  got = _native.lib().tqf_batch_workspace_size(items, blocks, steps)
  assert need <= got < need + 256


def test_native_direction_numbers_match_oracle():
  dim = 1200
  got = tsobol.direction_numbers(dim)
  want = osobol.direction_numbers(dim)
  want = np.array(want, dtype=object)
  want = np.vectorize(lambda v: v & 0xFFFFFFFF)(want).astype(np.uint64)
  np.testing.assert_array_equal(got.astype(np.uint64), want)


def test_generating_columns_match_qmc_matrices():
  g = osobol.sobol_generating_matrices(7, 500, 9)
  v = tsobol.generating_columns(7, 9, g.shape[1])
  np.testing.assert_array_equal(v[:, :g.shape[1]].astype(np.int64), g)


@pytest.mark.parametrize('kw', [
    dict(times=[1.0], num_time_steps=100),
    dict(times=[0.25, 0.5, 0.75, 1.0], num_time_steps=365),
    dict(times=[0.1, 0.5, 1.0], time_step=0.1),
    dict(times=[0.3, 0.7], time_step=0.05),
    dict(times=[0.33, 0.5], times_grid=np.linspace(0, 0.5, 11)),
])
@pytest.mark.parametrize('dtype', [np.float32, np.float64])
def test_prepare_grid_matches_oracle(kw, dtype):
  kw = dict(kw)
  times = kw.pop('times')
  ts = kw.get('time_step')
  if ts is None and kw.get('num_time_steps'):
    ts = np.asarray(times, dtype)[-1] / dtype(kw['num_time_steps'])
  a = utils.prepare_grid(times=times, time_step=ts, dtype=dtype,
                         num_time_steps=kw.get('num_time_steps'),
                         times_grid=kw.get('times_grid'))
  b = ogrid.prepare_grid(times, dtype, time_step=kw.get('time_step'),
                         num_time_steps=kw.get('num_time_steps'),
                         times_grid=kw.get('times_grid'))
  np.testing.assert_array_equal(a[0], b[0])
  np.testing.assert_array_equal(a[1], b[1])
  np.testing.assert_array_equal(a[2], b[2])


def test_heston_grid_matches_oracle():
  a = utils.heston_grid([0.5, 1.0], 0.1, None, [], np.float64)
  b = ogrid.heston_prepare_grid([0.5, 1.0], np.float64, time_step=0.1)
  np.testing.assert_array_equal(a[0], b[0])
  np.testing.assert_array_equal(a[1], b[1])
  a = utils.heston_grid([0.25, 1.0], 0.1, 10, [], np.float64)
  b = ogrid.heston_prepare_grid([0.25, 1.0], np.float64, num_time_steps=10)
  np.testing.assert_array_equal(a[0], b[0])


def _simulate_records(keep_mask, k, initial_written=None):
  """Replays the reference loop with state = step counter."""
  steps = len(keep_mask) - 1
  out = [None] * k
  record = k != 1
  written = int(keep_mask[0]) if initial_written is None else initial_written
  out[0] = -1  # TensorArray slot 0 / the plain result start as the state
  i = 0
  while i < steps and written < k:
    if record:
      out[written] = i
    else:
      out[0] = i
    written += int(keep_mask[i + 1])
    i += 1
  return out, i


@pytest.mark.parametrize('mask,k', [
    ([False, False, True, False, True], 2),
    ([True, False, True, True], 3),
    ([False, True, False, False], 1),
    ([False, False, False, True, False, True, False], 2),
    ([True, False, False], 1),
])
def test_record_plan_replays_reference_loop(mask, k):
  slots, init_slot, executed, filled = utils.record_plan(np.array(mask), k)
  want, n_exec = _simulate_records(mask, k)
  assert executed == n_exec
  got = [None] * k
  if init_slot >= 0:
    got[init_slot] = -1
  for i, s in enumerate(slots):
    if s >= 0:
      got[s] = i
  assert got == want


def test_record_plan_random_masks_replay_reference_loop():
  # the plan is computed from prefix sums of the mask: random masks, counts
  # (including none and more than the grid reaches) and starting counts
  # against the replayed loop, slot by slot, and the steps it executes
  rs = np.random.RandomState(11)
  for _ in range(3000):
    steps = rs.randint(0, 30)
    mask = rs.rand(steps + 1) < rs.rand()
    k = rs.randint(1, steps + 4)
    iw = None if rs.rand() < 0.5 else int(rs.randint(0, 3))
    slots, init_slot, executed, filled = utils.record_plan(mask, k, iw)
    want, n_exec = _simulate_records(mask, k, iw)
    assert executed == n_exec
    got = [None] * k
    if init_slot >= 0:
      got[init_slot] = -1
    for i, s in enumerate(slots):
      if s >= 0:
        got[s] = i
    assert got == want, (mask, k, iw)
    assert filled == sorted(j for j in range(k) if want[j] is not None)


def test_qe_step_coefficients_reproduce_oracle_moments():
  t = np.array([0.0, 0.1, 0.25, 0.25, 0.6])
  c = qe_step_coefficients(t, 1.5, 0.05, 0.6, -0.4, 1e-6, torch.float64)
  v = 0.07
  for i, dt in enumerate(np.diff(t)):
    e = np.exp(-1.5 * dt)
    m = 0.05 + (v - 0.05) * e
    s2 = v * 0.36 * e / 1.5 * (1 - e) + 0.05 * 0.36 / 2 / 1.5 * (1 - e)**2
    np.testing.assert_allclose(c[i, 8] + (v - c[i, 8]) * c[i, 0], m)
    np.testing.assert_allclose(v * c[i, 1] + c[i, 2], s2, atol=1e-18)
    assert c[i, 9] == (1.0 if dt > 1e-6 else 0.0)
  # log-spot update agrees with the oracle's for a pair of variances
  z = 0.3
  for i, dt in enumerate(np.diff(t)):
    if dt == 0:
      continue
    want = oheston.update_log_spot(1.5, 0.05, 0.6, -0.4, v, 0.06, 4.6, dt, z)
    got = (4.6 + c[i, 3] + c[i, 4] * v + c[i, 5] * 0.06 +
           np.sqrt(c[i, 6] * v + c[i, 7] * 0.06) * z)
    np.testing.assert_allclose(got, want, rtol=1e-14)


def test_product_fails_loudly_without_gpu():
  if torch.cuda.is_available():
    pytest.skip('a GPU is present')
  with pytest.raises(RuntimeError, match='ROCm GPU'):
    tsobol.sample(2, 5)


def _icdf_table():
  path = os.path.join(ROOT, 'tf-quant-finance_amd', 'csrc', 'icdf_table.h')
  text = open(path).read()
  zero = float.fromhex(re.search(r'kIcdfZero = (-?0x[0-9a-fA-F.]+p[+-]?\d+)f',
                                 text).group(1))
  body = text[text.index('kIcdfCoef'):]
  vals = [float.fromhex(h) for h in
          re.findall(r'(-?0x[0-9a-fA-F.]+p[+-]?\d+)f', body)]
  return np.asarray(vals, np.float32).reshape(-1, 4), np.float32(zero)


def test_icdf_table_matches_inverse_normal_exhaustively():
  """The float32 shifted-Sobol transform's table, evaluated as the kernels
  do (fold, float bit-pattern addressing, float32 Horner), against the
  oracle's float64 inverse CDF over all 2^25 values of the top 25 bits."""
  from oracle import normal as onormal
  coef, zero = _icdf_table()
  assert coef.shape == (192, 4)
  # LDS image: slot 0 = m = 0, slots 48..239 = segments, negated half
  img = np.zeros((2, 256, 4), np.float64)
  img[0, 0, 0] = zero
  img[0, 48:240] = coef
  img[1] = -img[0]
  n = np.arange(2**25, dtype=np.uint64)
  v = (n << np.uint64(7)).astype(np.uint32)
  s = (v.view(np.int32) >> 31).view(np.uint32)
  w = (v ^ s) & np.uint32(0xFFFFFF80)
  fi = w.astype(np.float32).view(np.uint32)
  assert np.all(w.astype(np.float32).astype(np.uint64) == w)  # exact
  slot = (fi >> np.uint32(20)) & np.uint32(0xFF)
  assert np.all((slot == 0) == (w == 0))
  assert slot[w != 0].min() >= 48 and slot.max() < 240
  g = (fi | np.uint32(0xFFF00000)).view(np.int32).astype(np.float32)
  c = img[(s & 1).astype(np.int64), slot.astype(np.int64)]
  p = c[:, 3]
  for k in (2, 1, 0):  # one rounding per FMA
    p = (p * g + c[:, k]).astype(np.float32).astype(np.float64)
  want = onormal.shifted_sobol_normals(v)
  err = np.abs(p - want)
  big = np.abs(want) >= 1e-3
  assert err.max() <= 5.5e-7, err.max()
  assert (err[big] / np.abs(want[big])).max() <= 3.5e-7
  assert err[~big].max() <= 2e-10
  # symmetry z(n) = -z(2^25 - 1 - n) holds exactly
  np.testing.assert_array_equal(p, -p[::-1])


def test_sobol_scrambling_host_matches_oracle_and_keeps_the_net():
  from tqf.math import qmc
  nd, n = 10, 1024
  g = qmc.sobol_generating_matrices(6, n, nd)
  sm = qmc.random_scrambling_matrices(6, nd, seed=(2, 3))
  assert sm.shape == (6, nd)
  assert np.all(sm >= 2**(nd - 1)) and np.all(sm < 2**nd)
  got = qmc.scramble_generating_matrices(g, sm, nd)
  np.testing.assert_array_equal(got,
                                osobol.scramble_generating_matrices(g, sm, nd))
  # minimum scrambling matrices are the identity (digital_net_test.py:274)
  ident = np.full_like(sm, 2**(nd - 1))
  np.testing.assert_array_equal(qmc.scramble_generating_matrices(g, ident, nd),
                                g)
  # the scrambled net is still a (0, m, 1)-net in every dimension: each
  # aligned block of 2^m points takes every value j / 2^m once
  pts = osobol.digital_net_sample_int(got, n, nd)
  for d in range(6):
    for m in (1, 4, 10):
      blk = (pts[:2**m, d] >> (nd - m)).astype(np.int64)
      assert sorted(blk) == list(range(2**m))


@pytest.mark.parametrize('shape', [(), (4,), (3, 4), (5, 1, 4), (5, 7, 4)])
def test_padded_discounts_tensor_and_array_agree(shape):
  """Discount factors given as a tensor are padded and transposed on their
  device exactly as the array form is (the reference's layout,
  lsm.py:239-256): [n_ex + 1, *, B] with a leading row of ones."""
  from tqf.models import longstaff_schwartz as lsm
  rs = np.random.RandomState(4)
  df = rs.uniform(0.8, 1.0, shape)
  want = lsm._padded_discounts(df, 4, torch.float64)
  got = lsm._padded_discounts(torch.as_tensor(df), 4, torch.float64)
  assert torch.is_tensor(got)
  assert tuple(got.shape) == want.shape
  np.testing.assert_array_equal(got.numpy(), want)
  np.testing.assert_array_equal(want[0], np.ones_like(want[0]))
