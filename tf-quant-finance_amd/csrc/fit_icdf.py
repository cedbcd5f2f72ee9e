"""Derives the piecewise-cubic inverse normal CDF table (icdf_table.h) used
by the float32 shifted-Sobol transform of the fused kernels.

The transform maps the top 25 bits n of a 32-bit Sobol point to
z = Phi^-1((n + 1/2) 2^-25).  By the symmetry Phi^-1(1 - u) = -Phi^-1(u)
the kernels fold the point onto the lower half: with s the sign mask of
the point (all ones when the top bit is set), m = ((v ^ s) >> 7) is in
[0, 2^24) and z = -+Phi^-1((m + 1/2) 2^-25), negated for the upper half.

Segments follow the float32 representation of m * 128 (exact: m has at
most 24 significant bits, and the kernels form it by masking the low 7
bits of v ^ s): for m >= 1 its exponent gives the octave of m (24 octaves,
geometric towards the tail) and the top 3 mantissa bits the sub-segment,
segment = (bits >> 20) - (134 << 3), 192 segments; m = 0 is the float 0,
a slot of its own holding the constant.  Inside a segment the variable is
g = (low 20 mantissa bits) - 2^20, an exact integer in [-2^20, -1] (the
kernels form it as a signed integer with one OR), i.e. the expansion point
is the segment's right end; the segment that ends at u = 1/2 therefore has
a constant term near 0 and keeps relative accuracy as z -> 0.
z = ((c3 g + c2) g + c1) g + c0 in float32 FMAs.

Each cubic is a weighted least-squares fit (weight 1/max(|z|, 1e-3)),
sharpened towards minimax by Lawson's iteration, over every m of the
segment; segments of octaves with at most 4 points interpolate them.  The
whole table is then checked exhaustively over all 2^24 values of m with
the float32 Horner evaluation.

A second table (icdf_dyadic_table.h) serves the reference transform of
unshifted points, erfinv((u - 1/2) 2) sqrt 2 at u = v 2^-nd, nd <= 24: with y
= t 2^-24 the point folded onto (0, 1/2], z = Phi^-1(y) as a function of the
float32 value of t 2^8, 16 sub-segments to an octave, the constant of the
segment that ends at y = 1/2 held at zero.

The log of the normal tail (log2_normal_tail in common.h): a degree-13
polynomial for log2(Phi(-z) e^(z^2 / 2)) on [-0.9, 6.5], minimax in the error
of log2 Phi(-z) relative to max(1/2, its size).

Run: python fit_icdf.py  (writes icdf_table.h and icdf_dyadic_table.h next
to this file, prints the error bounds and the tail's coefficients).
"""
import os

import numpy as np
from scipy import special

SEG_BITS = 3
LOW_BITS = 23 - SEG_BITS
E_MIN = 127 + 7  # exponent of float(1 * 128)
N_SEG = 24 << SEG_BITS


def segments():
  """(m, seg, g, z) for every m in [1, 2^24)."""
  m = np.arange(1, 2**24, dtype=np.int64)
  fi = (m * 128).astype(np.float32).view(np.uint32).astype(np.int64)
  seg = (fi >> LOW_BITS) - (E_MIN << SEG_BITS)
  g = (fi & ((1 << LOW_BITS) - 1)) - (1 << LOW_BITS)
  z = special.ndtri((m + 0.5) * 2.0**-25)
  return m, seg, g, z


def fit_segment(g, z, iters=30, max_pts=20000):
  k = min(3, g.size - 1)
  c = np.zeros(4)
  if k == 0:
    c[0] = z[0]
    return c
  sc = -float(g.min())
  x = g / sc
  if x.size > max_pts:
    sel = np.linspace(0, x.size - 1, max_pts).astype(np.int64)
    x, z = x[sel], z[sel]
  v = np.vander(x, k + 1, increasing=True)
  if x.size == k + 1:  # interpolation
    cc = np.linalg.solve(v, z)
    c[:k + 1] = cc / sc**np.arange(k + 1)
    return c
  base = 1.0 / np.maximum(np.abs(z), 1e-3)
  wt = np.ones_like(x) / x.size
  for _ in range(iters):
    w = np.sqrt(wt) * base
    cc, *_ = np.linalg.lstsq(v * w[:, None], z * w, rcond=None)
    e = np.abs(v @ cc - z) * base
    if e.max() == 0:
      break
    wt = wt * (e + 1e-6 * e.max())
    wt /= wt.sum()
  c[:k + 1] = cc / sc**np.arange(k + 1)
  return c


def horner_f32(c32, seg, g):
  """float32 Horner with one rounding per FMA (float64 products of float32
  operands are exact, so rounding the float64 sum once emulates fmaf)."""
  gf = g.astype(np.float64)
  p = c32[seg, 3].astype(np.float64)
  for k in (2, 1, 0):
    p = (p * gf + c32[seg, k]).astype(np.float32).astype(np.float64)
  return p


DYADIC_BITS = 4
N_DYADIC = 23 << DYADIC_BITS


def fit_to_zero(g, z, iters=30):
  """fit_segment with c0 = 0 (the segment that ends at y = 1/2)."""
  sc = -float(g.min())
  x = g / sc
  v = np.stack([x, x * x, x**3], 1)
  base = 1.0 / np.maximum(np.abs(z), 1e-6)
  wt = np.ones_like(x) / x.size
  for _ in range(iters):
    w = np.sqrt(wt) * base
    cc, *_ = np.linalg.lstsq(v * w[:, None], z * w, rcond=None)
    e = np.abs(v @ cc - z) * base
    wt = wt * (e + 1e-6 * e.max())
    wt /= wt.sum()
  return np.concatenate([[0.0], cc / sc**np.arange(1, 4)])


def dyadic_main():
  low = 23 - DYADIC_BITS
  t = np.arange(1, 2**23, dtype=np.int64)
  fi = (t * 256).astype(np.float32).view(np.uint32).astype(np.int64)
  seg = (fi >> low) - ((127 + 8) << DYADIC_BITS)
  g = ((fi & ((1 << low) - 1)) - (1 << low)).astype(np.float64)
  z = special.ndtri(t * 2.0**-24)
  bounds = np.searchsorted(seg, np.arange(N_DYADIC + 1))
  coef = np.zeros((N_DYADIC, 4))
  for s in range(N_DYADIC):
    sl = slice(bounds[s], bounds[s + 1])
    if bounds[s + 1] > bounds[s]:
      fit = fit_to_zero if s == N_DYADIC - 1 else fit_segment
      coef[s] = fit(g[sl], z[sl])
  # the kernel's variable is 2^-23 g: exact powers of two
  c32 = coef.astype(np.float32)
  err = np.abs(horner_f32(c32, seg, g) - z)
  bound = ('max abs err %.2e, max rel err %.2e, rms rel err %.2e' % (
      err.max(), (err / np.abs(z)).max(), np.sqrt(np.mean((err / z)**2))))
  print('dyadic: ' + bound)
  out = os.path.join(os.path.dirname(os.path.abspath(__file__)),
                     'icdf_dyadic_table.h')
  with open(out, 'w') as f:
    f.write('// Generated by fit_icdf.py: piecewise-cubic Phi^-1(t 2^-24) on '
            't in [1, 2^23),\n// segment s = (bits(float(t * 256)) >> 19) - '
            '2160, variable h in [-2^-4, -2^-23],\n'
            '// z = ((c3 h + c2) h + c1) h + c0.  Exhaustive float32 check:\n'
            '// %s.\n' % bound)
    f.write('#pragma once\n\nnamespace tqf {\n\n')
    f.write('constexpr int kDyadicSegBits = %d;\n'
            'constexpr int kDyadicSegs = %d;\n\n' % (DYADIC_BITS, N_DYADIC))
    f.write('// {c0, c1, c2, c3} per segment\n')
    f.write('__device__ __constant__ const float '
            'kDyadicCoef[kDyadicSegs * 4] = {\n')
    for s in range(N_DYADIC):
      f.write('    ' + ', '.join(
          '%sf' % float(v * 2.0**(23 * k)).hex()
          for k, v in enumerate(c32[s].astype(np.float64))) + ',\n')
    f.write('};\n\n}  // namespace tqf\n')
  print('wrote', out)


def tail_main(lo=-0.9, hi=6.5, deg=13, iters=80):
  cheb, poly = np.polynomial.chebyshev, np.polynomial.polynomial
  def want(z):
    return np.log2(0.5 * special.erfcx(z / np.sqrt(2)))
  z = lo + (hi - lo) * (1 - np.cos(np.pi * np.arange(4001) / 4000)) / 2
  v = cheb.chebvander((2 * z - lo - hi) / (hi - lo), deg)
  full = want(z) - z * z * 0.5 * np.log2(np.e)
  w0 = 1 / np.maximum(0.5, np.abs(full))
  wt = np.ones_like(z) / z.size
  for _ in range(iters):
    w = np.sqrt(wt) * w0
    c, *_ = np.linalg.lstsq(v * w[:, None], want(z) * w, rcond=None)
    e = np.abs(v @ c - want(z)) * w0
    wt = wt * (e + 1e-3 * e.max())
    wt /= wt.sum()
  out = np.zeros(1)
  for k in cheb.cheb2poly(c)[::-1]:
    out = poly.polyadd(
        poly.polymul(out, [-(lo + hi) / (hi - lo), 2 / (hi - lo)]), [k])
  print('normal tail, fit %.1e:' % e.max(),
        [float(x).hex() for x in out[:deg + 1].astype(np.float32)])


def main():
  m, seg, g, z = segments()
  order = np.argsort(seg, kind='stable')
  bounds = np.searchsorted(seg[order], np.arange(N_SEG + 1))
  coef = np.zeros((N_SEG, 4))
  for s in range(N_SEG):
    idx = order[bounds[s]:bounds[s + 1]]
    if idx.size:
      coef[s] = fit_segment(g[idx].astype(np.float64), z[idx])
  c32 = coef.astype(np.float32)
  p = horner_f32(c32, seg, g)
  err = np.abs(p - z)
  big = np.abs(z) >= 1e-3
  zero = np.float32(special.ndtri(0.5 * 2.0**-25))
  max_abs = max(err.max(), abs(float(zero) - special.ndtri(0.5 * 2.0**-25)))
  max_rel = (err[big] / np.abs(z[big])).max()
  near0 = err[~big].max()
  print('max abs err %.3e, max rel err (|z| >= 1e-3) %.3e, max abs err '
        '(|z| < 1e-3) %.3e' % (max_abs, max_rel, near0))
  out = os.path.join(os.path.dirname(os.path.abspath(__file__)),
                     'icdf_table.h')
  with open(out, 'w') as f:
    f.write('// Generated by fit_icdf.py: piecewise-cubic Phi^-1((m + 1/2) '
            '2^-25) on the lower\n// half, segment s = (bits(float(m * 128)) '
            '>> 20) - 1072 for m >= 1, variable\n// g in [-2^20, -1], '
            'z = ((c3 g + c2) g + c1) g + c0; kIcdfZero is z at m = 0.\n'
            '// Exhaustive float32 check over all 2^24 values of m:\n'
            '// max abs err %.2e, max rel err %.2e for |z| >= 1e-3, max abs '
            'err %.2e for |z| < 1e-3.\n' % (max_abs, max_rel, near0))
    f.write('#pragma once\n\nnamespace tqf {\n\n')
    f.write('constexpr int kIcdfSegBits = %d;\nconstexpr int kIcdfSegs = %d;\n'
            % (SEG_BITS, N_SEG))
    f.write('constexpr float kIcdfZero = %sf;\n\n' % float(zero).hex())
    f.write('// {c0, c1, c2, c3} per segment\n')
    f.write('__device__ __constant__ const float kIcdfCoef[kIcdfSegs * 4] = {\n')
    for s in range(N_SEG):
      f.write('    ' + ', '.join('%sf' % float(v).hex() for v in c32[s]) +
              ',\n')
    f.write('};\n\n}  // namespace tqf\n')
  print('wrote', out)


if __name__ == '__main__':
  main()
  dyadic_main()
  tail_main()
