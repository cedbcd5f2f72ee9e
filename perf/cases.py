"""Workloads of the engine: what a program that uses it calls, at the sizes
it calls it with.

Every case goes through the public entry points.  `prepare` makes a case's
inputs from a seed (market data, contract tables, simulated market paths) and
the plan or handle a program keeps between calls; `run` is one call;
`exact` is the same result restated in float64 with torch alone (its own
Philox, Sobol and step loops), for the error of a result.

Kinds:
  calls      European calls over strikes x dates, simulation and payoff fused
  paths      euler_sampling.sample of Heston paths
  qe         HestonModel.sample_paths (Andersen QE)
  gbm        GeometricBrownianMotion / MultivariateGeometricBrownianMotion
             .sample_paths (exact scheme)
  grad       euler_sampling.sample and the gradient of its paths
  batch      a heterogeneous contract table with Greeks (engine.batch)
  basket     a basket call with adjoint Greeks (engine.greeks)
  american   bs_lsm_price, one shared set of Brownian paths per call
  lsm        least_square_mc on given multi-asset paths
  mlp        one exercise date of the learned continuation value
  swaption   bermudan_swaption_price under Hull-White
"""
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, 'tf-quant-finance_amd'))

import tqf  # noqa: E402
from tqf.engine import batch as batch_lib  # noqa: E402
from tqf.engine import euler as engine  # noqa: E402
from tqf.engine import greeks as greeks_lib  # noqa: E402
from tqf.engine import mlp_lsm  # noqa: E402
from tqf.engine import pricing  # noqa: E402
from tqf.experimental import american_option  # noqa: E402
from tqf.math.random.multivariate_normal import RandomType  # noqa: E402
from tqf.models import longstaff_schwartz as lsm_lib  # noqa: E402
from tqf.models.hull_white import bermudan_swaption_price  # noqa: E402

F64 = torch.float64


def listed():
  return [
      # the smallest pricing call: one textbook Black-Scholes check
      # (1e5 paths, 100 steps, 8 strikes, float64): launches and latency
      dict(name='calls_gbm_small', kind='calls', model='gbm', paths=100000,
           steps=100, strikes=8, dates=1, draws='philox', type='f64'),
      # a volatility surface in one call: a year of daily Heston steps,
      # 64 strikes x 4 maturities, quasi-random paths
      dict(name='calls_heston_sobol', kind='calls', model='heston',
           paths=2**20, steps=365, strikes=64, dates=4, draws='sobol',
           type='f32'),
      # every daily state of a path set, kept for the caller's own payoffs:
      # bound by the memory it fills
      dict(name='paths_heston_daily', kind='paths', paths=2**19, steps=365,
           dates=365, draws='sobol', type='f32'),
      # QE paths at quarterly dates of a year of daily steps
      dict(name='qe_quarterly', kind='qe', paths=2**20, steps=365, dates=4,
           draws='philox', type='f32'),
      # four correlated assets at 63 exact dates, an odd number of paths
      dict(name='gbm_four_assets', kind='gbm', assets=4, paths=200001,
           dates=63, draws='philox', type='f32'),
      # sampling and its gradient in the model's parameters (calibration)
      dict(name='grad_heston', kind='grad', paths=2**17, steps=100, dates=4,
           draws='philox', type='f32'),
      # an intraday revaluation of a mixed book with Greeks
      dict(name='batch_book', kind='batch', contracts=256, greeks='tangent'),
      # a 16-name basket with its 33 Greeks
      dict(name='basket_16', kind='basket', assets=16, paths=262144,
           steps=64),
      # four American options, a hundred exercise dates
      dict(name='american_four', kind='american', options=4, paths=2**20,
           dates=100),
      # the five-asset Bermudan max-call, independent pricing paths
      dict(name='lsm_max_call_5', kind='lsm', assets=5, paths=2**20,
           dates=9, payoff='max_call', split=True),
      # one exercise date of the learned continuation value: training steps
      # on the calibration paths, then a forward pass over every path
      dict(name='mlp_date', kind='mlp', rows=2**18, batch=65536, steps=40),
      # two Bermudan swaptions on one set of short-rate paths
      dict(name='swaption_pair', kind='swaption', swaptions=2, paths=2**19,
           maturity=5),
  ]


def _log_int(rng, lo, hi):
  """An integer spread over the logarithm of [lo, hi], any remainder."""
  return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
  kind = rng.choice(['calls', 'paths', 'qe', 'gbm', 'grad', 'batch',
                     'basket', 'american', 'lsm', 'mlp', 'swaption'])
  f = rng.choice(['f32', 'f32', 'f64'])
  if kind == 'calls':
    dates = rng.randint(1, 6)
    return dict(kind=kind, model=rng.choice(['gbm', 'heston', 'heston']),
                paths=_log_int(rng, 10000, 2**19),
                steps=rng.randint(max(12, 2 * dates), 365),
                strikes=rng.randint(1, 100), dates=dates,
                draws=rng.choice(['philox', 'sobol']), type=f)
  if kind == 'paths':
    steps = rng.randint(12, 365)
    return dict(kind=kind, paths=2 * _log_int(rng, 5000, 2**17), steps=steps,
                dates=rng.choice([steps, rng.randint(1, 6)]),
                draws=rng.choice(['philox', 'antithetic', 'sobol']), type=f)
  if kind == 'qe':
    return dict(kind=kind, paths=2 * _log_int(rng, 5000, 2**17),
                steps=rng.randint(24, 365), dates=rng.randint(1, 6),
                draws=rng.choice(['philox', 'antithetic', 'sobol']), type=f)
  if kind == 'gbm':
    assets = rng.choice([1, 1, 2, 3, 5, 8, 12])
    return dict(kind=kind, assets=assets,
                paths=2 * _log_int(rng, 5000, 2**18 // assets),
                dates=rng.randint(1, 100),
                draws=rng.choice(['philox', 'antithetic', 'sobol']), type=f)
  if kind == 'grad':
    return dict(kind=kind, paths=2 * _log_int(rng, 2000, 50000),
                steps=rng.randint(20, 120), dates=rng.randint(1, 6),
                draws=rng.choice(['philox', 'antithetic']), type=f)
  if kind == 'batch':
    return dict(kind=kind, contracts=rng.randint(16, 160),
                greeks=rng.choice(['tangent', 'tangent', 'adjoint']))
  if kind == 'basket':
    return dict(kind=kind, assets=rng.randint(2, 16),
                paths=_log_int(rng, 20000, 2**18), steps=rng.randint(12, 64))
  if kind == 'american':
    return dict(kind=kind, options=rng.randint(1, 6),
                paths=2 * _log_int(rng, 10000, 2**18),
                dates=rng.randint(10, 60))
  if kind == 'lsm':
    return dict(kind=kind, assets=rng.randint(1, 4),
                paths=_log_int(rng, 20000, 2**19), dates=rng.randint(4, 24),
                payoff=rng.choice(['max_call', 'basket_put']),
                split=rng.choice([True, False]))
  if kind == 'mlp':
    rows = _log_int(rng, 30000, 2**18)
    return dict(kind=kind, rows=rows, batch=min(rows // 2, 65536),
                steps=rng.randint(10, 40))
  return dict(kind='swaption', swaptions=rng.randint(1, 3),
              paths=2 * _log_int(rng, 10000, 2**18),
              maturity=rng.randint(3, 6))


# ------------------------------------------------------------- inputs -----

_TYPES = {'f32': torch.float32, 'f64': torch.float64}


def _dtype(case):
  return _TYPES[case['type']]


def _heston(rng):
  """Heston market parameters with 2 kappa theta > xi^2."""
  kappa, theta = rng.uniform(1.5, 3.0), rng.uniform(0.03, 0.06)
  xi = rng.uniform(0.5, 0.9) * math.sqrt(2 * kappa * theta)
  return dict(s0=rng.uniform(90, 110), v0=rng.uniform(0.03, 0.06),
              kappa=kappa, theta=theta, xi=xi, rho=rng.uniform(-0.8, -0.3),
              r=rng.uniform(0.01, 0.04))


def _times(n, t):
  return np.linspace(t / n, t, n)


def _calls_inputs(case, seed):
  rng = random.Random(seed)
  m = _heston(rng)
  m['sigma'] = rng.uniform(0.15, 0.3)
  m['strikes'] = np.linspace(0.6, 1.4, case['strikes']) * m['s0']
  m['maturities'] = _times(case['dates'], 1.0)
  m['seed'] = rng.getrandbits(30)
  return m


def _paths_inputs(case, seed):
  rng = random.Random(seed)
  m = _heston(rng)
  m['seed'] = rng.getrandbits(30)
  m['skip'] = rng.randrange(0, 5000)
  m['times'] = _times(case['dates'], 1.0)
  return m


def _random_type(case):
  return {'philox': RandomType.PSEUDO,
          'antithetic': RandomType.PSEUDO_ANTITHETIC,
          'sobol': RandomType.SOBOL}[case['draws']]


def _gbm_inputs(case, seed):
  rng = random.Random(seed)
  d = case['assets']
  rs = np.random.RandomState(seed % 2**31)
  a = rs.standard_normal((d, d + 2))
  c = a @ a.T
  return dict(mu=rs.uniform(0.0, 0.06, d), sigma=rs.uniform(0.1, 0.4, d),
              corr=c / np.sqrt(np.outer(np.diag(c), np.diag(c))),
              s0=rs.uniform(80, 120, d), seed=rng.getrandbits(30),
              skip=rng.randrange(0, 5000), times=_times(case['dates'], 1.0))


def _contracts(n, seed):
  """A mixed book: GBM and Heston calls, 2^12 .. 2^18 paths, 50 .. 500
  steps (the distribution of engine.batch.random_contracts), the volatility
  of variance held to 2 kappa theta >= xi^2 so every Greek has a finite
  variance."""
  rs = np.random.RandomState(seed % 2**31)
  out = []
  for i in range(n):
    vol = rs.uniform(0.1, 0.5)
    kappa, theta = rs.uniform(0.5, 5.0), rs.uniform(0.01, 0.09)
    xi = min(rs.uniform(0.1, 0.8), math.sqrt(2 * kappa * theta))
    s0 = rs.uniform(50, 150)
    out.append(dict(
        # half of the book is GBM, whatever the seed: the work is the case's
        kind=batch_lib.KIND_GBM if i % 2 else batch_lib.KIND_HESTON,
        n_steps=int(rs.randint(50, 501)),
        n_paths=int(round(2.0**(12 + 6 * (i // 2 + 0.5) * 2 / (n + 1)))),
        s0=s0, strike=rs.uniform(0.7, 1.3) * s0, maturity=rs.uniform(0.1, 3.0),
        rate=0.03, sigma=vol, v0=max(vol * vol, theta), kappa=kappa,
        theta=theta, xi=xi, rho=rs.uniform(-0.9, 0.0)))
  return out


def _basket_inputs(case, seed):
  d = case['assets']
  rs = np.random.RandomState(seed % 2**31)
  a = rs.standard_normal((d, d))
  c = a @ a.T + np.eye(d)
  return dict(s0=rs.uniform(80, 120, d), sigma=rs.uniform(0.15, 0.45, d),
              corr=c / np.sqrt(np.outer(np.diag(c), np.diag(c))), rate=0.02,
              maturity=1.0, strike=100.0, seed=int(rs.randint(1 << 30)))


def _american_inputs(case, seed):
  rs = np.random.RandomState(seed % 2**31)
  n = case['options']
  expiry = rs.uniform(0.5, 2.0, n)
  return dict(spots=rs.uniform(90, 110, n), expiry=expiry,
              strikes=np.full(n, 100.0), vol=rs.uniform(0.15, 0.35, n),
              df=np.exp(-rs.uniform(0.02, 0.06, n) * expiry),
              seed=(int(rs.randint(1 << 30)), 2))


def _lsm_inputs(case, seed):
  """Correlated GBM market paths, float64, in the engine's step-major
  memory ([N, T, d] view of [T][d][N])."""
  g = torch.Generator(device='cuda').manual_seed(seed)
  n, d, dates = case['paths'], case['assets'], case['dates']
  dt, r, q, sigma, corr = 3.0 / dates, 0.05, 0.1, 0.2, 0.3
  c = torch.full((d, d), corr, dtype=F64, device='cuda')
  c.fill_diagonal_(1.0)
  chol = torch.linalg.cholesky(c)
  x = torch.empty((dates + 1, d, n), dtype=F64, device='cuda')
  x[0] = 100.0
  for i in range(dates):
    z = chol @ torch.randn((d, n), dtype=F64, device='cuda', generator=g)
    x[i + 1] = x[i] * torch.exp((r - q - 0.5 * sigma**2) * dt +
                                sigma * math.sqrt(dt) * z)
  df = np.exp(-r * dt * np.arange(1, dates + 1))
  return x.permute(2, 0, 1), df


def _mlp_inputs(case, seed):
  """Standardised asset prices and exercise value, noisy continuation
  targets, in-the-money weights, as mlp_lsm_price feeds the network."""
  g = torch.Generator(device='cuda').manual_seed(seed)
  n = case['rows']
  x = torch.zeros((n, 8), dtype=torch.float32, device='cuda')
  x[:, :5] = torch.randn((n, 5), device='cuda', generator=g)
  top = x[:, :5].max(1).values
  x[:, 5] = torch.relu(0.25 * (top - 0.5))
  noise = torch.randn(n, device='cuda', generator=g)
  t = torch.relu(0.05 + 0.2 * top + 0.1 * noise)
  w = (x[:, 5] > 0).float()
  return x, t, w


def _mlp_params(seed):
  rs = np.random.RandomState(seed % 2**31)
  w1 = rs.standard_normal((6, 64)) * math.sqrt(2.0 / 6)
  w2 = rs.standard_normal((64, 64)) * math.sqrt(2.0 / 64)
  w3 = rs.standard_normal(64) * math.sqrt(1.0 / 64)
  return np.concatenate([w1.ravel(), np.zeros(64), w2.ravel(), np.zeros(64),
                         w3, [0.0]]).astype(np.float32)


def _swaption_inputs(case, seed):
  """Semiannual payer swaptions to `maturity`, first exercise after one
  year and half a year later for each further one."""
  rng = random.Random(seed)
  end_t, b = float(case['maturity']), case['swaptions']
  n = 2 * case['maturity'] - 2
  base = 1.0 + 0.5 * np.arange(n + 1)
  at = lambda i: base[min(i, n)]
  ex = np.array([[at(k + i) for i in range(n)] for k in range(b)])
  start = np.array([[[at(k + i + j) for j in range(n)] for i in range(n)]
                    for k in range(b)])
  end = np.clip(start + 0.5, 0.0, end_t)
  rate = rng.uniform(0.008, 0.015)
  return dict(ex=ex, start=start, end=end, dcf=end - start, rate=rate,
              coupon=rate + 0.001, a=rng.uniform(0.02, 0.05),
              sigma=rng.uniform(0.008, 0.012),
              seed=[rng.getrandbits(30), 0])


def prepare(case, seed):
  kind = case['kind']
  if kind == 'calls':
    # a program prices one product again and again: it keeps the launch
    m = _calls_inputs(case, seed)
    dtype = _dtype(case)
    grid, keep = pricing.heston_grid_for(m['maturities'], case['steps'],
                                         'reference', dtype)
    dims = (grid.shape[0] - 1) * (2 if case['model'] == 'heston' else 1)
    if case['draws'] == 'sobol':
      rng = engine.RngSpec('sobol_shifted', first_index=0,
                           shift=pricing.sobol_digital_shift(dims, m['seed']))
    else:
      rng = engine.RngSpec('philox', seed=m['seed'])
    if case['model'] == 'heston':
      spec = ('heston', m['r'], m['kappa'], m['theta'], m['xi'], m['rho'],
              0.0)
      x0 = np.array([np.log(m['s0']), m['v0']])
    else:
      spec, x0 = ('gbm', m['r'], m['sigma']), [m['s0']]
    return dict(case=case, launch=pricing.european_calls(
        spec, x0, m['strikes'], grid, keep, case['paths'], rng,
        discount_rate=m['r'], dtype=dtype, prepare=True))
  if kind in ('paths', 'qe', 'grad'):
    m = _paths_inputs(case, seed)
    state = dict(case=case, m=m)
    if kind == 'grad':
      t = lambda v: torch.tensor(v, dtype=_dtype(case), device='cuda',
                                 requires_grad=True)
      state['inputs'] = [t([math.log(m['s0']), m['v0']])] + [
          t(m[k]) for k in ('r', 'kappa', 'theta', 'xi', 'rho')]
      g = torch.Generator(device='cuda').manual_seed(seed)
      state['weights'] = torch.rand(
          (case['paths'], case['dates'], 2), dtype=_dtype(case),
          device='cuda', generator=g)
    return state
  if kind == 'gbm':
    return dict(case=case, m=_gbm_inputs(case, seed))
  if kind == 'batch':
    plan = batch_lib.BatchPlan(_contracts(case['contracts'], seed),
                               tile=2048, greeks=case['greeks'],
                               seed=seed % 2**31)
    return dict(case=case, plan=plan)
  if kind == 'basket':
    return dict(case=case, m=_basket_inputs(case, seed))
  if kind == 'american':
    return dict(case=case, m=_american_inputs(case, seed))
  if kind == 'lsm':
    x, df = _lsm_inputs(case, seed)
    return dict(case=case, paths=x, df=df)
  if kind == 'mlp':
    x, t, w = _mlp_inputs(case, seed)
    params = _mlp_params(seed)
    return dict(case=case, x=x, t=t, w=w, params=params,
                model=mlp_lsm.MlpModel(params=params),
                out=torch.empty(case['rows'], device='cuda'))
  return dict(case=case, m=_swaption_inputs(case, seed))


# ---------------------------------------------------------------- run -----

def run(state):
  return _RUN[state['case']['kind']](state)


def _run_calls(st):
  r = st['launch'].launch()
  return {k: r[k] for k in ('prices', 'stderrs', 'sums')}


def _sample_heston(case, m, kappa, theta, xi, rho, r, x0):
  drift, vol = tqf.models.HestonModel(
      kappa, theta, xi, rho, dtype=_dtype(case)).euler_ft_fns(r)
  return tqf.models.euler_sampling.sample(
      2, drift, vol, m['times'], num_time_steps=case['steps'],
      num_samples=case['paths'], initial_state=x0,
      random_type=_random_type(case), seed=m['seed'], skip=m['skip'],
      dtype=_dtype(case))


def _run_paths(st):
  m = st['m']
  return _sample_heston(st['case'], m, m['kappa'], m['theta'], m['xi'],
                        m['rho'], m['r'],
                        np.array([math.log(m['s0']), m['v0']]))


def _run_grad(st):
  x0, r, kappa, theta, xi, rho = st['inputs']
  paths = _sample_heston(st['case'], st['m'], kappa, theta, xi, rho, r, x0)
  grads = torch.autograd.grad(paths, st['inputs'], st['weights'])
  return dict(paths=paths.detach(), grads=list(grads))


def _run_qe(st):
  case, m = st['case'], st['m']
  return tqf.models.HestonModel(
      m['kappa'], m['theta'], m['xi'], m['rho'],
      dtype=_dtype(case)).sample_paths(
          m['times'], [math.log(m['s0']), m['v0']],
          num_samples=case['paths'], num_time_steps=case['steps'],
          random_type=_random_type(case), seed=m['seed'], skip=m['skip'])


def _run_gbm(st):
  case, m = st['case'], st['m']
  kw = dict(num_samples=case['paths'], random_type=_random_type(case),
            seed=m['seed'], skip=m['skip'])
  if case['assets'] == 1:
    return tqf.models.GeometricBrownianMotion(
        float(m['mu'][0]), float(m['sigma'][0]),
        dtype=_dtype(case)).sample_paths(
            m['times'], initial_state=float(m['s0'][0]), **kw)
  return tqf.models.MultivariateGeometricBrownianMotion(
      case['assets'], m['mu'], m['sigma'], m['corr'],
      dtype=_dtype(case)).sample_paths(m['times'], initial_state=m['s0'],
                                       **kw)


def _run_batch(st):
  return st['plan'].launch()


def _run_basket(st):
  m, case = st['m'], st['case']
  return greeks_lib.basket_call_greeks(
      m['s0'], m['sigma'], m['corr'], m['rate'], m['maturity'], m['strike'],
      case['steps'], case['paths'], seed=m['seed'])


def _run_american(st):
  m, case = st['m'], st['case']
  return american_option.bs_lsm_price(
      m['spots'], m['expiry'], m['strikes'], m['vol'], m['df'],
      num_samples=case['paths'], num_exercise_times=case['dates'],
      is_call_option=False, seed=m['seed'])


def _run_lsm(st):
  case = st['case']
  payoff = (lsm_lib.make_max_call_payoff([100.0])
            if case['payoff'] == 'max_call'
            else lsm_lib.make_basket_put_payoff([100.0]))
  return lsm_lib.least_square_mc(
      st['paths'], list(range(1, case['dates'] + 1)), payoff,
      lsm_lib.make_polynomial_basis(2), discount_factors=st['df'],
      num_calibration_samples=case['paths'] // 2 if case['split'] else None)


def _run_mlp(st):
  case, model = st['case'], st['model']
  model.reset(params=st['params'])
  model.train_date(st['x'], st['t'], st['w'], case['rows'], case['batch'],
                   case['steps'], 1e-3)
  model.forward(st['x'], st['out'])
  return dict(params=model.params, loss=model.loss, out=st['out'])


def _run_swaption(st):
  m, case = st['m'], st['case']
  return bermudan_swaption_price(
      exercise_times=m['ex'], floating_leg_start_times=m['start'],
      floating_leg_end_times=m['end'], fixed_leg_payment_times=m['end'],
      floating_leg_daycount_fractions=m['dcf'],
      fixed_leg_daycount_fractions=m['dcf'],
      fixed_leg_coupon=m['coupon'] * np.ones_like(m['end']),
      reference_rate_fn=lambda t: m['rate'] * torch.ones_like(
          torch.as_tensor(t)),
      notional=100.0, mean_reversion=m['a'], volatility=m['sigma'],
      num_samples=case['paths'], time_step=0.1,
      random_type=RandomType.STATELESS_ANTITHETIC, seed=m['seed'],
      dtype=F64)


_RUN = dict(calls=_run_calls, paths=_run_paths, qe=_run_qe, gbm=_run_gbm,
            grad=_run_grad, batch=_run_batch, basket=_run_basket,
            american=_run_american, lsm=_run_lsm, mlp=_run_mlp,
            swaption=_run_swaption)


# ----------------------------------------------------------- the work -----

def work(case):
  """Bytes a pass cannot avoid (inputs read and outputs written once) and
  its arithmetic, a transcendental or a generated normal's Box-Muller term
  one operation each, integer work none."""
  kind = case['kind']
  size = 8 if case.get('type') == 'f64' else 4
  n = case.get('paths', 0)
  if kind == 'calls':
    out = case['strikes'] * case['dates']
    step = 73 if case['model'] == 'heston' else 8.5
    return dict(bytes=40 * out, flops=n * (case['steps'] * step + 4 * out))
  if kind in ('paths', 'qe', 'grad'):
    out = n * case['dates'] * 2 * size
    step = {'paths': 73, 'qe': 60, 'grad': 73 + 95}[kind]
    return dict(bytes=out * (3 if kind == 'grad' else 1),
                flops=n * case['steps'] * step)
  if kind == 'gbm':
    d = case['assets']
    return dict(bytes=n * case['dates'] * d * size,
                flops=n * case['dates'] * d * (12 + d))
  if kind == 'batch':
    paths = [round(2.0**(12 + 6 * (i // 2 + 0.5) * 2 /
                         (case['contracts'] + 1)))
             for i in range(case['contracts'])]
    flops = sum(275 * p * (10 if i % 2 else 95) for i, p in enumerate(paths))
    return dict(bytes=case['contracts'] * 240, flops=flops)
  if kind == 'basket':
    d = case['assets']
    return dict(bytes=8 * d * (d + 3),
                flops=n * (case['steps'] * d * 6 + d * (d + 40)))
  if kind == 'american':
    return dict(bytes=64 * case['options'],
                flops=n * case['dates'] * (12 + 40 * case['options']))
  if kind == 'lsm':
    d = case['assets']
    k = 3**d
    calib = n // 2 if case['split'] else n
    moments = 2 * 5**d + 2 * k
    return dict(bytes=n * case['dates'] * d * 8,
                flops=(case['dates'] - 1) * (calib * moments + n * 2 * k))
  if kind == 'mlp':
    return dict(bytes=case['rows'] * 44,
                flops=27264 * case['batch'] * case['steps'] +
                9088 * case['rows'])
  n_ex = 2 * case['maturity'] - 2
  return dict(bytes=64 * case['swaptions'],
              flops=n * (10 * case['maturity'] * 10 + case['swaptions'] *
                         n_ex * (n_ex * 4 + 40)))


def tolerance(case):
  """About four times what a float32 (or float64) result differs from its
  float64 restatement at these sizes."""
  kind = case['kind']
  f64 = case.get('type') == 'f64'
  if kind in ('calls', 'paths', 'gbm'):
    return dict(rel=1e-11 if f64 else 4e-6)
  if kind == 'qe':
    # a path at the switch between the two branches takes the other one
    return dict(rel=1e-9 if f64 else 1e-4, max=0.5)
  if kind == 'grad':
    # the derivative of sqrt(v+) grows as a path nears v = 0
    return dict(rel=1e-8 if f64 else 1.5e-3)
  if kind == 'batch':
    return dict(rel=3e-3)
  if kind == 'basket':
    return dict(rel=4e-6)
  if kind == 'mlp':
    # bfloat16 products, then Adam's normalised steps
    return dict(rel=2e-2, max=0.5)
  # a path whose exercise and continuation values agree to rounding may take
  # either
  return dict(rel=1e-6)


# -------------------------------------------------------------- exact -----
# The same numbers in float64 with torch operations alone.

_CHUNK = 2**17


def _mulhilo(m, x):
  """High and low words of m x for 32-bit words held in int64."""
  low = m * (x & 0xffff)
  mid = m * (x >> 16) + (low >> 16)
  return mid >> 16, ((mid & 0xffff) << 16) | (low & 0xffff)


def _philox(c0, c1, c2, c3, key):
  k0, k1 = key & 0xffffffff, (key >> 32) & 0xffffffff
  for _ in range(10):
    h0, l0 = _mulhilo(0xD2511F53, c0)
    h1, l1 = _mulhilo(0xCD9E8D57, c2)
    c0, c1, c2, c3 = h1 ^ c1 ^ k0, l1, h0 ^ c3 ^ k1, l0
    k0, k1 = (k0 + 0x9E3779B9) & 0xffffffff, (k1 + 0xBB67AE85) & 0xffffffff
  return c0, c1, c2, c3


def _box_muller(a, b, single):
  if single:
    u, t = ((a >> 8) + 1).to(F64) * 2.0**-24, (b >> 8).to(F64) * 2.0**-24
  else:
    u, t = (a + 1).to(F64) * 2.0**-32, b.to(F64) * 2.0**-32
  r = torch.sqrt(-2.0 * torch.log(u))
  t = 2.0 * math.pi * t
  return r * torch.cos(t), r * torch.sin(t)


class _Philox:
  """Normal j of the paths p, four per counter block."""

  def __init__(self, p, key, single, stream=0):
    self.p, self.key, self.single, self.stream = p, key, single, stream
    self.block, self.z = -1, None

  def normal(self, j):
    if j // 4 != self.block:
      self.block = j // 4
      z = torch.zeros_like(self.p)
      w = _philox(self.p, z + self.block, z + self.stream, z, self.key)
      self.z = (_box_muller(w[0], w[1], self.single) +
                _box_muller(w[2], w[3], self.single))
    return self.z[j % 4]


def _direction_numbers(dim):
  """The first 32 direction integers of every dimension, from the Joe-Kuo
  table."""
  m = [[1] * 32]
  name = os.path.join(ROOT, 'tf-quant-finance_amd', 'tqf', 'data', 'sobol',
                      'new-joe-kuo-6.21201')
  with open(name) as f:
    next(f)
    for line in f:
      if len(m) == dim:
        break
      tok = [int(v) for v in line.split()]
      s, a, v = tok[1], tok[2], tok[3:]
      for k in range(s, 32):
        x = v[k - s] ^ (v[k - s] << s)
        for i in range(1, s):
          if (a >> (s - 1 - i)) & 1:
            x ^= v[k - i] << i
        v.append(x)
      m.append(v)
  return m


class _Sobol:
  """Normal j (dimension j) of the points of index `first` + p: the
  reference transform of 2^-digits points, or (shift given) the engine's of
  32-digit shifted points."""

  def __init__(self, p, first, digits, dim, shift, single):
    self.lo, self.hi = (first + p) & 1023, (first + p) >> 10
    self.digits, self.shift, self.single = digits, shift, single
    self.rows = int(self.hi.max()) + 1
    self.m = _direction_numbers(dim)

  def _word(self, j):
    def table(n, bit0):
      i = torch.arange(n, device='cuda')
      t = torch.zeros(n, dtype=torch.int64, device='cuda')
      b = 0
      while (n - 1) >> b:
        v = self.m[j][bit0 + b] << (self.digits - 1 - bit0 - b)
        t ^= ((i >> b) & 1) * v
        b += 1
      return t
    return table(1024, 0)[self.lo] ^ table(self.rows, 10)[self.hi]

  def normal(self, j):
    x = self._word(j)
    if self.shift is None:
      q = x.to(F64) * 2.0**(1 - self.digits) - 1.0
    else:
      x = x ^ self.shift[j]
      if self.single:
        q = ((x >> 7).to(F64) + 0.5) * 2.0**-24 - 1.0
      else:
        q = (x.to(F64) + 0.5) * 2.0**-31 - 1.0
    return torch.erfinv(q) * math.sqrt(2.0)


def _shift_words(n, key):
  i = torch.arange((n + 3) // 4, device='cuda')
  z = torch.zeros_like(i)
  w = torch.stack(_philox(z, i, z + 0x5348, z, key), 1)
  return [int(v) for v in w.reshape(-1)[:n].cpu()]


def _normals(case, m, p, dim):
  """The draws of the paths p, and their sign (antithetic halves)."""
  single = case.get('type') == 'f32'
  n = case['paths']
  if case['draws'] == 'sobol':
    digits = math.ceil(math.log2(m['skip'] + n + 1))
    return _Sobol(p, m['skip'] + 1, digits, dim, None, single), 1.0
  if case['draws'] == 'antithetic':
    half = n // 2
    return (_Philox(torch.where(p < half, p, p - half), m['seed'], single),
            torch.where(p < half, 1.0, -1.0).to(F64))
  return _Philox(p, m['seed'], single), 1.0


def _chunks(n):
  for p0 in range(0, n, _CHUNK):
    yield torch.arange(p0, min(p0 + _CHUNK, n), device='cuda')


def _np_type(case):
  return np.float64 if case['type'] == 'f64' else np.float32


def _grid(times, steps, npd):
  """The sampler's grid: a uniform one with `times` merged in."""
  times = np.asarray(times, npd)
  step = npd(times[-1] / npd(steps))
  uniform = np.linspace(step, times[-1] - step, max(steps - len(times), 0),
                        dtype=npd)
  grid = np.concatenate([np.zeros(1, npd),
                         np.sort(np.concatenate([uniform, times]).astype(npd),
                                 kind='stable')])
  return grid, np.searchsorted(grid, times, side='left')


def _exact_calls(case, seed):
  m = _calls_inputs(case, seed)
  npd = _np_type(case)
  times = np.asarray(m['maturities']).astype(npd)
  step = npd(np.asarray(m['maturities'])[-1] / case['steps'])
  uniform = np.linspace(step, times[-1] - step,
                        max(case['steps'] - len(times), 0), dtype=npd)
  grid = np.concatenate([np.zeros(1, npd), np.sort(
      np.concatenate([uniform, times]).astype(npd), kind='stable')])
  at = np.searchsorted(grid, times, side='left')
  d = 2 if case['model'] == 'heston' else 1
  dt = (grid[1:] - grid[:-1]).astype(np.float64)
  shift = None
  if case['draws'] == 'sobol':
    shift = _shift_words(d * len(dt), m['seed'])
  k = torch.as_tensor(m['strikes'], device='cuda')
  sums = torch.zeros((len(times), len(k), 2), dtype=F64, device='cuda')
  s1r = math.sqrt(1 - m['rho']**2)
  for p in _chunks(case['paths']):
    src = (_Sobol(p, 0, 32, d * len(dt), shift, case['type'] == 'f32')
           if shift else _Philox(p, m['seed'], case['type'] == 'f32'))
    x = torch.full(p.shape, math.log(m['s0']), dtype=F64, device='cuda')
    v = torch.full_like(x, m['v0'])
    for i, h in enumerate(dt):
      z0 = src.normal(i * d) * math.sqrt(h)
      if d == 2:
        z1 = src.normal(i * d + 1) * math.sqrt(h)
        vp = torch.clamp(v, min=0)
        sq = torch.sqrt(vp)
        x = x + (m['r'] - 0.5 * vp) * h + sq * z0
        v = (v + m['kappa'] * (m['theta'] - vp) * h +
             m['xi'] * sq * (m['rho'] * z0 + s1r * z1))
      else:
        x = x + torch.log1p(m['r'] * h + m['sigma'] * z0)
      for c in np.flatnonzero(at == i + 1):
        pay = torch.relu(torch.exp(x)[:, None] - k)
        sums[c, :, 0] += pay.sum(0)
        sums[c, :, 1] += (pay * pay).sum(0)
  n = case['paths']
  df = torch.as_tensor(np.exp(-m['r'] * grid[at].astype(np.float64)),
                       device='cuda')[:, None]
  mean = sums[..., 0] / n
  var = torch.clamp((sums[..., 1] - n * mean * mean) / (n - 1), min=0)
  return dict(prices=df * mean, stderrs=df * torch.sqrt(var / n), sums=sums)


def _exact_paths(case, seed):
  m = _paths_inputs(case, seed)
  grid, at = _grid(m['times'], case['steps'], _np_type(case))
  dt = (grid[1:] - grid[:-1]).astype(np.float64)
  out = torch.empty((len(at), 2, case['paths']), dtype=F64, device='cuda')
  s1r = math.sqrt(1 - m['rho']**2)
  for p in _chunks(case['paths']):
    src, sign = _normals(case, m, p, 2 * len(dt))
    x = torch.full(p.shape, math.log(m['s0']), dtype=F64, device='cuda')
    v = torch.full_like(x, m['v0'])
    for i, h in enumerate(dt):
      z0 = sign * src.normal(2 * i) * math.sqrt(h)
      z1 = sign * src.normal(2 * i + 1) * math.sqrt(h)
      vp = torch.clamp(v, min=0)
      sq = torch.sqrt(vp)
      x = x + (m['r'] - 0.5 * vp) * h + sq * z0
      v = (v + m['kappa'] * (m['theta'] - vp) * h +
           m['xi'] * sq * (m['rho'] * z0 + s1r * z1))
      for c in np.flatnonzero(at == i + 1):
        out[c, 0, p], out[c, 1, p] = x, v
  return out.permute(2, 0, 1)


def _exact_grad(case, seed):
  m = _paths_inputs(case, seed)
  grid, at = _grid(m['times'], case['steps'], _np_type(case))
  dt = (grid[1:] - grid[:-1]).astype(np.float64)
  g = torch.Generator(device='cuda').manual_seed(seed)
  weights = torch.rand((case['paths'], case['dates'], 2),
                       dtype=_dtype(case), device='cuda', generator=g).to(F64)
  npd = _np_type(case)
  t = lambda v: torch.tensor(np.asarray(v, npd).astype(np.float64),
                             dtype=F64, device='cuda', requires_grad=True)
  names = ('r', 'kappa', 'theta', 'xi', 'rho')
  inputs = [t([math.log(m['s0']), m['v0']])] + [t(m[k]) for k in names]
  x0, r, kappa, theta, xi, rho = inputs
  total = [torch.zeros_like(q) for q in inputs]
  paths = []
  for p in _chunks(case['paths']):
    src, sign = _normals(case, m, p, 2 * len(dt))
    x, v = x0[0].expand(p.shape), x0[1].expand(p.shape)
    recs = []
    for i, h in enumerate(dt):
      z0 = sign * src.normal(2 * i) * math.sqrt(h)
      z1 = sign * src.normal(2 * i + 1) * math.sqrt(h)
      pos = v > 0
      vp = torch.where(pos, v, torch.zeros_like(v))
      sq = torch.where(pos, torch.sqrt(torch.where(pos, v,
                                                   torch.ones_like(v))),
                       torch.zeros_like(v))
      x = x + (r - 0.5 * vp) * h + sq * z0
      v = (v + kappa * (theta - vp) * h +
           xi * sq * (rho * z0 + torch.sqrt(1 - rho**2) * z1))
      for _ in np.flatnonzero(at == i + 1):
        recs.append(torch.stack([x, v], -1))
    recs = torch.stack(recs, 1)
    for q, gq in zip(total, torch.autograd.grad(recs, inputs, weights[p])):
      q += gq
    paths.append(recs.detach())
  return dict(paths=torch.cat(paths), grads=total)


def _exact_qe(case, seed):
  m = _paths_inputs(case, seed)
  npd = _np_type(case)
  times = np.asarray(m['times'], npd)
  step = npd(times[-1] / npd(case['steps']))
  grid = np.concatenate([
      np.linspace(npd(0.0), times[-1] - step, case['steps'], dtype=npd),
      times])
  mask = np.arange(len(grid)) >= case['steps']
  order = np.argsort(grid, kind='stable')
  grid, mask = grid[order], mask[order]
  dt = (grid[1:] - grid[:-1]).astype(np.float64)
  skip = ~((grid[1:] - grid[:-1]).astype(npd) > npd(1e-6))
  k, th, xi, rho = m['kappa'], m['theta'], m['xi'], m['rho']
  out = torch.empty((len(times), 2, case['paths']), dtype=F64, device='cuda')
  for p in _chunks(case['paths']):
    src, sign = _normals(case, m, p, 2 * len(dt))
    x = torch.full(p.shape, math.log(m['s0']), dtype=F64, device='cuda')
    v = torch.full_like(x, m['v0'])
    c = 0
    for i, h in enumerate(dt):
      z0 = sign * src.normal(2 * i)
      z1 = sign * src.normal(2 * i + 1)
      if not skip[i]:
        e = math.exp(-k * h)
        mean = th + (v - th) * e
        s2 = (v * xi * xi * e / k * (1 - e) +
              th * xi * xi / 2 / k * (1 - e)**2)
        psi = s2 / mean**2
        pinv = 2.0 / torch.clamp(psi, max=2.0)
        b2 = pinv - 1 + torch.sqrt(pinv * (pinv - 1))
        quad = mean / (1 + b2) * (torch.sqrt(b2) + z0)**2
        pr = (psi - 1) / (psi + 1)
        beta = (1 - pr) / mean
        u = 0.5 * (1 + torch.erf(z0 / math.sqrt(2.0)))
        tail = torch.where(u > pr, torch.log((1 - pr) / (1 - u)) / beta,
                           torch.zeros_like(u))
        vn = torch.where(psi < 1.5, quad, tail)
        a = 0.5 * h * (k * rho / xi - 0.5)
        x = (x - rho * k * th / xi * h + (a - rho / xi) * v +
             (a + rho / xi) * vn +
             torch.sqrt(0.5 * h * (1 - rho**2) * (v + vn)) * z1)
        v = vn
      if mask[i + 1]:
        out[c, 0, p], out[c, 1, p] = x, v
        c += 1
  return out.permute(2, 0, 1)


def _exact_gbm(case, seed):
  m = _gbm_inputs(case, seed)
  d = case['assets']
  npd = _np_type(case)
  grid = np.concatenate([np.zeros(1, npd), np.asarray(m['times'], npd)])
  dt = (grid[1:] - grid[:-1]).astype(np.float64)
  chol = (np.eye(1) if d == 1 else np.linalg.cholesky(m['corr']))
  out = torch.empty((len(dt), d, case['paths']), dtype=F64, device='cuda')
  for p in _chunks(case['paths']):
    src, sign = _normals(case, m, p, d * len(dt))
    cum = torch.zeros((d, len(p)), dtype=F64, device='cuda')
    for i, h in enumerate(dt):
      z = torch.stack([sign * src.normal(i * d + c) for c in range(d)])
      w = torch.as_tensor(chol, device='cuda') @ z
      vol = torch.as_tensor(m['sigma'], device='cuda')[:, None]
      mu = torch.as_tensor(m['mu'], device='cuda')[:, None]
      cum = cum + (mu - 0.5 * vol * vol) * h + vol * math.sqrt(h) * w
      out[i, :, p] = torch.as_tensor(m['s0'], device='cuda')[:, None] * (
          torch.exp(cum))
  return out.permute(2, 0, 1)


def _exact_batch(case, seed):
  """Both halves of the book, every path of a half side by side, the
  contracts by falling step count so finished ones drop off the end."""
  cs = _contracts(case['contracts'], seed)
  key = seed % 2**31
  out = torch.zeros((len(cs), 16), dtype=F64, device='cuda')
  for heston in (False, True):
    ids = [i for i, c in enumerate(cs)
           if (c['kind'] == batch_lib.KIND_HESTON) == heston]
    ids.sort(key=lambda i: -cs[i]['n_steps'])
    groups = [ids[i:i + 16] for i in range(0, len(ids), 16)]
    for g in groups:
      stats = _batch_group(cs, g, key, heston)
      for i, s in zip(g, stats):
        out[i] = s
  return out


def _batch_group(cs, ids, key, heston):
  count = torch.tensor([cs[i]['n_paths'] for i in ids], device='cuda')
  own = torch.repeat_interleave(torch.arange(len(ids), device='cuda'), count)
  first = torch.cumsum(count, 0) - count
  p = torch.arange(len(own), device='cuda') - first[own]
  stream = torch.tensor(ids, device='cuda')[own]
  col = lambda f: torch.tensor([float(np.float32(cs[i][f])) for i in ids],
                               dtype=F64, device='cuda')[own]
  steps = [cs[i]['n_steps'] for i in ids]
  alive = lambda i: int(count[:sum(1 for s in steps if s > i)].sum())
  s0, strike, t, r = (col(f) for f in ('s0', 'strike', 'maturity', 'rate'))
  dt = t / torch.tensor(steps, dtype=F64, device='cuda')[own]
  sdt = torch.sqrt(dt)
  z = None
  zero = torch.zeros_like(s0)
  if heston:
    x, v = torch.log(s0), col('v0')
    kappa, theta, xi, rho = (col(f) for f in ('kappa', 'theta', 'xi', 'rho'))
    s1r = torch.sqrt(1 - rho * rho)
    tx = [zero.clone() for _ in range(5)]
    tv = [zero + 1] + [zero.clone() for _ in range(4)]
  else:
    x, w, sigma = zero.clone(), zero.clone(), col('sigma')
  per = 2 if heston else 4
  for i in range(max(steps)):
    a = alive(i)
    if i % per == 0:
      b = torch.zeros_like(p[:a])
      q = _philox(p[:a], b + i // per, stream[:a], b, key)
      z = (_box_muller(q[0], q[1], True) + _box_muller(q[2], q[3], True))
    if not heston:
      dw = z[i % 4][:a] * sdt[:a]
      x[:a] += (r[:a] - 0.5 * sigma[:a]**2) * dt[:a] + sigma[:a] * dw
      w[:a] += dw
      continue
    dw0 = z[2 * (i % 2)][:a] * sdt[:a]
    dw1 = z[2 * (i % 2) + 1][:a] * sdt[:a]
    h, va = dt[:a], v[:a]
    pos = va > 0
    vp = torch.where(pos, va, zero[:a])
    sq = torch.sqrt(vp)
    half = torch.where(pos, 0.5 / sq, zero[:a])
    noise = rho[:a] * dw0 + s1r[:a] * dw1
    for c in range(5):
      tvp = torch.where(pos, tv[c][:a], zero[:a])
      tsq = tvp * half
      tx[c][:a] += -0.5 * h * tvp + tsq * dw0
      tv[c][:a] += -h * kappa[:a] * tvp + tsq * xi[:a] * noise
    tv[1][:a] += h * (theta[:a] - vp)
    tv[2][:a] += h * kappa[:a]
    tv[3][:a] += sq * noise
    tv[4][:a] += xi[:a] * sq * (dw0 - rho[:a] / s1r[:a] * dw1)
    x[:a] += h * (r[:a] - 0.5 * vp) + sq * dw0
    v[:a] = va + h * kappa[:a] * (theta[:a] - vp) + xi[:a] * sq * noise
  disc = torch.exp(-r * t)
  s = torch.exp(x) if heston else s0 * torch.exp(x)
  sb = torch.where(s > strike, disc * s, zero)
  pay = disc * torch.relu(s - strike)
  if heston:
    g = [pay, sb / s0, sb * tx[0], -t * pay + sb * t, sb * tx[1], sb * tx[2],
         sb * tx[3], sb * tx[4]]
  else:
    g = [pay, sb / s0, sb * (w - sigma * t), -t * pay + sb * t,
         zero, zero, zero, zero]
  g = torch.stack(g)
  out = []
  for f, n in zip(first.tolist(), count.tolist()):
    part = g[:, f:f + n]
    out.append(torch.cat([part.mean(1), part.std(1) / math.sqrt(n)]))
  return out


def _exact_basket(case, seed):
  m = _basket_inputs(case, seed)
  d, n, steps, t = case['assets'], case['paths'], case['steps'], m['maturity']
  pad = (d + 3) // 4 * 4  # the engine draws whole blocks of four assets
  f = lambda a: torch.as_tensor(np.asarray(a, np.float64), device='cuda')
  chol = f(np.linalg.cholesky(m['corr']))
  s0, sig = f(m['s0'])[:, None], f(m['sigma'])[:, None]
  disc = math.exp(-m['rate'] * t)
  sums = torch.zeros((2, 2 + 2 * d), dtype=F64, device='cuda')
  for p in _chunks(n):
    src = _Philox(p, m['seed'], True)
    zs = torch.zeros((d, len(p)), dtype=F64, device='cuda')
    for i in range(steps):
      for c in range(d):
        zs[c] += src.normal(i * pad + c)
    w = chol @ zs * math.sqrt(t / steps)
    s = s0 * torch.exp((m['rate'] - 0.5 * sig * sig) * t + sig * w)
    a = s.mean(0)
    itm = (a > m['strike']).to(F64) * disc
    pay = itm * (a - m['strike'])
    g = torch.cat([pay[None], (-t * pay + itm * t * a)[None],
                   itm * s / d / s0, itm * s / d * (w - sig * t)])
    sums[0] += g.sum(1)
    sums[1] += (g * g).sum(1)
  mean = sums[0] / n
  se = torch.sqrt(torch.clamp(
      (sums[1] - n * mean * mean) / (n - 1), min=0) / n)
  mean, se = mean.cpu().numpy(), se.cpu().numpy()
  return {'price': (mean[0], se[0]), 'rho': (mean[1], se[1]),
          'delta': (mean[2:2 + d], se[2:2 + d]),
          'vega': (mean[2 + d:], se[2 + d:])}


def _exact_lsm(feature, payoff, ratio, n_ex, calib, degree=2):
  """Backward induction over n_ex dates: feature(e) [N, d] and payoff(e)
  [N] of date e, ratio(e) the discount factor of date e over date e - 1
  (date -1: today)."""
  value = payoff(n_ex - 1)
  for e in range(n_ex - 2, -1, -1):
    x, ev = feature(e), payoff(e)
    y = ratio(e + 1) * value
    sd = x.std(0, unbiased=False)
    c = (x - x.mean(0)) / torch.where(sd > 1e-12, sd, torch.ones_like(sd))

    def design(part):
      cols = torch.ones((len(part), 1), dtype=F64, device='cuda')
      for j in range(part.shape[1]):
        pw = torch.stack([part[:, j]**q for q in range(degree + 1)], 1)
        cols = (cols[:, :, None] * pw[:, None, :]).reshape(len(part), -1)
      return cols
    gram, rhs, size = 0.0, 0.0, 2**16
    for p0 in range(0, calib, size):
      p1 = min(p0 + size, calib)
      a = design(c[p0:p1]) * (ev[p0:p1, None] > 0)
      gram = gram + a.T.contiguous() @ a
      rhs = rhs + a.T.contiguous() @ y[p0:p1]
    sc = torch.sqrt(torch.diagonal(gram))
    sc = torch.where(sc > 0, 1 / sc, torch.zeros_like(sc))
    beta = sc * (torch.linalg.pinv(
        gram * sc[:, None] * sc, hermitian=True,
        rtol=10 * len(sc) * 2.0**-52) @ (rhs * sc))
    cont = torch.cat([design(c[p0:p0 + size]) @ beta
                      for p0 in range(0, len(c), size)])
    value = torch.where(ev > torch.relu(cont), ev, y)
  return ratio(0) * value


def _exact_american(case, seed):
  m = _american_inputs(case, seed)
  n, dates = case['paths'], case['dates']
  times = np.linspace(0.0, 1.0, dates)
  dt = np.diff(np.concatenate([[0.0], times]))
  key = m['seed'][0] | (m['seed'][1] << 32)
  w = torch.empty((dates, n), dtype=F64, device='cuda')
  for p in _chunks(n // 2):
    src = _Philox(p, key, False)
    b = torch.zeros(p.shape, dtype=F64, device='cuda')
    for i in range(dates):
      b = b + math.sqrt(dt[i]) * src.normal(i)
      w[i, p], w[i, p + n // 2] = b, -b
  out = []
  for k in range(case['options']):
    t, vol = m['expiry'][k], m['vol'][k]
    rate = -math.log(m['df'][k]) / t
    strike = m['strikes'][k] / m['spots'][k]
    log_s = lambda e: ((rate - 0.5 * vol**2) * times[e] * t +
                       vol * math.sqrt(t) * w[e])
    df = np.exp(-rate * times * t)
    pv = _exact_lsm(lambda e: log_s(e)[:, None],
                    lambda e: torch.relu(strike - torch.exp(log_s(e))),
                    lambda e: df[e] / (df[e - 1] if e else 1.0), dates, n)
    out.append(pv.mean() * m['spots'][k])
  return torch.stack(out)


def _exact_lsm_case(case, seed):
  x, df = _lsm_inputs(case, seed)
  n = case['paths']
  calib = n // 2 if case['split'] else n
  if case['payoff'] == 'max_call':
    pay = lambda e: torch.relu(x[:, e + 1].max(-1).values - 100.0)
  else:
    pay = lambda e: torch.relu(100.0 - x[:, e + 1].mean(-1))
  pv = _exact_lsm(lambda e: x[:, e + 1], pay,
                  lambda e: df[e] / (df[e - 1] if e else 1.0), case['dates'],
                  calib)
  return pv[calib if case['split'] else 0:].mean().reshape(1)


def _exact_mlp(case, seed):
  x, t, w = (a.to(F64) for a in _mlp_inputs(case, seed))
  x = x[:, :6]
  p = torch.as_tensor(_mlp_params(seed), dtype=F64, device='cuda')
  size = [384, 64, 4096, 64, 64, 1]

  def net(q, rows):
    w1, b1, w2, b2, w3, b3 = torch.split(q, size)
    h = torch.nn.functional.silu(rows @ w1.reshape(6, 64) + b1)
    h = torch.nn.functional.silu(h @ w2.reshape(64, 64) + b2)
    return h @ w3 + b3
  m, v = torch.zeros_like(p), torch.zeros_like(p)
  for k in range(case['steps']):
    i = (k * case['batch']) % max(case['rows'] - case['batch'] + 1, 1)
    sl = slice(i, i + case['batch'])
    q = p.clone().requires_grad_(True)
    loss = (w[sl] * (net(q, x[sl]) - t[sl])**2).sum() / case['batch']
    g = torch.autograd.grad(loss, q)[0]
    m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
    p = p - 1e-3 * (m / (1 - 0.9**(k + 1))) / (
        torch.sqrt(v / (1 - 0.999**(k + 1))) + 1e-8)
  return dict(params=p, loss=loss.detach().reshape(1), out=net(p, x))


def _exact_swaption(case, seed):
  m = _swaption_inputs(case, seed)
  n, a, sigma, r0 = case['paths'], m['a'], m['sigma'], m['rate']
  _, at = np.unique(m['ex'].reshape(-1), return_index=True)
  dates = m['ex'].reshape(-1)[np.sort(at)]  # in order of first appearance
  sim = np.unique(np.concatenate([dates, np.arange(0.1, dates[-1], 0.1)]))
  grid = np.sort(np.concatenate([[0.0], sim]))
  key = m['seed'][0] | (m['seed'][1] << 32)
  mean = lambda t: ((math.exp(a * t) + math.exp(-a * t) - 2) * sigma**2 /
                    (2 * a * a))
  rates = torch.empty((len(dates), n), dtype=F64, device='cuda')
  disc = torch.empty_like(rates)
  for p in _chunks(n // 2):
    src = _Philox(p, key, False)
    for sign, rows in ((1.0, p), (-1.0, p + n // 2)):
      src.block = -1
      x = torch.zeros(p.shape, dtype=F64, device='cuda')
      total = torch.zeros_like(x)
      for i in range(len(grid) - 1):
        t, u = grid[i], grid[i + 1]
        sd = math.sqrt(max(sigma**2 / (2 * a) * (
            math.exp(2 * a * u) - math.exp(2 * a * t)), 0.0)) * math.exp(
                -a * u)
        x = (x * math.exp(-a * (u - t)) +
             (mean(u) - mean(t)) * math.exp(-a * u) +
             sd * sign * src.normal(i))
        # the rate of the first simulated date carries no discounting
        total = total + (x + r0) * ((u - t) if i else 0.0)
        for c in np.flatnonzero(dates == u):
          rates[c, rows], disc[c, rows] = x + r0, torch.exp(-total)
  out = []
  for b in range(case['swaptions']):
    swap = torch.zeros_like(rates)
    for e, t in enumerate(m['ex'][b]):
      c = int(np.flatnonzero(dates == t)[0])
      y = sigma**2 / (2 * a) * (1 - math.exp(-2 * a * t))
      value = 1.0
      for j, u in enumerate(m['end'][b, e]):
        g = (1 - math.exp(-a * (u - t))) / a
        bond = math.exp(-r0 * (u - t)) * torch.exp(
            -(rates[c] - r0) * g - 0.5 * y * g * g)
        last = 1.0 if j == len(m['end'][b, e]) - 1 else 0.0
        value = value - (m['coupon'] * m['dcf'][b, e, j] + last) * bond
      swap[c] = torch.relu(value)
    pv = _exact_lsm(lambda e: rates[e][:, None], lambda e: swap[e],
                    lambda e: disc[e] / (disc[e - 1] if e else 1.0),
                    len(dates), n)
    out.append(100.0 * pv.mean())
  return torch.stack(out)


def exact(case, seed):
  return dict(calls=_exact_calls, paths=_exact_paths, qe=_exact_qe,
              gbm=_exact_gbm, grad=_exact_grad, batch=_exact_batch,
              basket=_exact_basket, american=_exact_american,
              lsm=_exact_lsm_case, mlp=_exact_mlp,
              swaption=_exact_swaption)[case['kind']](case, seed)
