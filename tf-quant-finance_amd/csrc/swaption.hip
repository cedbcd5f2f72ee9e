// Regression inputs of Bermudan swaptions under one-factor Hull-White, from
// short-rate paths (payoff mapping of tff/models/hull_white/swaption.py:
// 591-724, 876-935; bond reconstitution vector_hull_white.py:783-814).
//
// One thread walks one path over the simulation dates: it sums the rate
// times the step length, and at an exercise date writes the rate, the path's
// discount factor exp(-sum r dt) and every swaption's exercise value
//   max(1 - sum_j w_j P(t, T_j), 0),  P(t, T_j) = exp(C_j - r G_j),
// with the host's constants C, G and weights w (coupon times day count, plus
// one at the last payment; payments on one date merged, zero weights left
// out).  Everything is read once and written once, in the regression's
// date-major layout.  As separate tensor operations (gathers, a matrix
// product for the discounts, an exponential over [N, batch, dates, payments]
// and a product with block-diagonal weights) the same took about 2 ms for
// two swaptions of 2^19 paths; bound by the exponentials here (22 float64
// instructions each).
#include "common.h"

using namespace tqf;

namespace {

struct SwaptionArgs {
  int64_t sp, st, n;
  int n_dates, n_ex, n_payoffs;
  const double* dt;       // [n_dates]
  const int32_t* slot;    // [n_dates] exercise index or -1
  const int32_t* first;   // [n_ex * n_payoffs + 1] entry ranges
  const double* entries;  // [.][3] C, G, w
  double* short_rate;     // [n_ex][n]
  double* payoff;         // [n_payoffs][n_ex][n]
  double* discounts;      // [n_ex + 1][n]
};

template <typename R>
__global__ void __launch_bounds__(256)
swaption_inputs_kernel(const R* __restrict__ rates, SwaptionArgs a) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= a.n) return;
  const R* rp = rates + p * a.sp;
  double total = 0.0;
  a.discounts[p] = 1.0;
#pragma unroll 4
  for (int i = 0; i < a.n_dates; ++i) {
    const double r = (double)rp[(int64_t)i * a.st];
    total = fma(r, ld_uniform(a.dt, i), total);
    const int u = ld_uniform(a.slot, i);
    if (u < 0) continue;
    a.short_rate[(int64_t)u * a.n + p] = r;
    a.discounts[(int64_t)(u + 1) * a.n + p] = exp_f64(-total);
    for (int b = 0; b < a.n_payoffs; ++b) {
      const int k0 = ld_uniform(a.first, u * a.n_payoffs + b);
      const int k1 = ld_uniform(a.first, u * a.n_payoffs + b + 1);
      double v = 1.0;
#pragma unroll 2
      for (int k = k0; k < k1; ++k)
        v = fma(-ld_uniform(a.entries, 3 * (int64_t)k + 2),
                exp_f64(fma(-r, ld_uniform(a.entries, 3 * (int64_t)k + 1),
                            ld_uniform(a.entries, 3 * (int64_t)k))), v);
      // a date without entries is not one of the swaption's own; NaN stays
      a.payoff[((int64_t)b * a.n_ex + u) * a.n + p] =
          k1 == k0 || v < 0 ? 0.0 : v;
    }
  }
  // a path whose rates are not finite has no price: its values at dates
  // before the first such rate may look sound, and its sums of the
  // regression are NaN, so its last factor, which every value is multiplied
  // by, says so
  if (!(total - total == 0.0)) a.discounts[a.n + p] = total - total;
}

}  // namespace

extern "C" int tqf_swaption_inputs(const void* rates, int64_t stride_path,
                                   int64_t stride_time, int64_t n_paths,
                                   int32_t dtype,
                                   const tqf_swaption_plan* plan,
                                   double* short_rate, double* payoff,
                                   double* discounts, void* stream) {
  clear_error();
  TQF_REQUIRE(rates && plan && short_rate && payoff && discounts,
              "null swaption argument");
  TQF_REQUIRE(dtype == TQF_F32 || dtype == TQF_F64, "bad dtype %d", dtype);
  TQF_REQUIRE(n_paths >= 1 && plan->n_dates >= 1 && plan->n_ex >= 1 &&
                  plan->n_payoffs >= 1,
              "empty swaption plan");
  TQF_REQUIRE(plan->dt && plan->slot && plan->first && plan->entries,
              "null swaption plan arrays");
  const SwaptionArgs a{stride_path,   stride_time,     n_paths,
                       plan->n_dates, plan->n_ex,      plan->n_payoffs,
                       plan->dt,      plan->slot,      plan->first,
                       plan->entries, short_rate,      payoff,
                       discounts};
  const unsigned blocks = (unsigned)((n_paths + 255) / 256);
  if (dtype == TQF_F32)
    hipLaunchKernelGGL(swaption_inputs_kernel<float>, blocks, 256, 0,
                       (hipStream_t)stream, (const float*)rates, a);
  else
    hipLaunchKernelGGL(swaption_inputs_kernel<double>, blocks, 256, 0,
                       (hipStream_t)stream, (const double*)rates, a);
  return check_launch("tqf_swaption_inputs");
}
