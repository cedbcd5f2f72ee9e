// One-asset Longstaff-Schwartz (tff/models/longstaff_schwartz/lsm.py:
// 128-436) for several payoffs on the same paths, two launches per exercise
// date for all of them.
//
// With one asset and a monomial basis the regression needs the power sums
// c^0 .. c^(2 deg) and y c^0 .. y c^deg of the in-the-money calibration rows,
// and each path's state is one float64 per payoff: the reference's pair
// (cashflow, discounted later values) always has one member zero after an
// update, so their sum is exact and is all the regression and the price
// read.  For date r = n_ex - 2 .. -1:
//   pass r, over the paths: the value of date r + 1 (the payoff at the last
//     date, else exercise against the continuation polynomial fitted
//     before), then the power sums of date r, one row per workgroup and
//     payoff (pass -1: the discounted values' sum and sum of squares);
//   solve r, one workgroup per payoff: the rows added in a fixed order, and
//     the regression solved in registers (column scaling, Cholesky with
//     pivot truncation, back substitution).
// The centring (mean and variance of the basis variable over all paths, per
// date) comes from one sweep over the paths before the first date.  It is
// the same for every affine image of the paths, so payoffs whose log price
// is a_t + b W(t) of shared Brownian paths W read W itself and form no paths
// of their own.
//
// The paths' columns are read once per date for all payoffs; the values
// (8 bytes per path and payoff, read and written per date) are the traffic:
// 80 MB a date for four payoffs of 2^20 paths, which the 256 MB last-level
// cache holds.
#include "lsm_chain.h"

namespace tqf {
namespace {

constexpr int kThreads = 256;
constexpr int kRows = 4;         // paths per thread and round
constexpr int kMaxBlocks = 512;  // workgroups per payoff
constexpr int kSolveThreads = 1024;
constexpr int kStatSlices = 64;

struct PassItem {
  double strike, log_strike;
  double shift_u, shift_m, scale;  // log price = shift + scale * stored
  double ratio_u, ratio_m;         // scalar discount ratios
  const double* tab_u;             // table payoff rows of the two dates
  const double* tab_m;
  int payoff, pad;
};

struct PassArgs {
  const double* col_u;   // stored values of date r + 1: col_u[p * sp]
  const double* col_m;   // of date r
  int64_t sp, n, n_calib;
  int64_t rows_per_block;
  const double* stat_u;  // (mean, variance) of the basis variable
  const double* stat_m;
  const double* dnum_u;  // per-path discount rows, or null
  const double* dden_u;
  const double* dnum_m;
  const double* dden_m;
  int terminal;          // date r + 1 is the last date: value = payoff
  int last;              // no regression: sums of the discounted values
  double* values;        // [items][n]
  double* zero;          // last: cleared [n], or null
  double* rows;          // [items][gridDim.x][NM]
  const double* coef;    // [items][kChainMaxDeg + 1]
  int64_t first;         // last: first pricing row
  int n_items;
  PassItem it[kChainMaxItems];
};

// LOGM is basis_log: 0 the basis variable and the price are the stored
// value; 1 the basis variable is its logarithm; 2 the basis variable is the
// stored value and the price exp(shift + scale * stored).
template <int LOGM>
__device__ __forceinline__ double basis_var(double x) {
  return LOGM == 1 ? log(x) : x;
}

template <int LOGM>
__device__ __forceinline__ bool in_money(const PassItem& it, double x,
                                         double shift, const double* tab,
                                         int64_t p) {
  if (it.payoff == TQF_PAYOFF_TABLE) return tab[p] > 0;
  if (LOGM == 2) {
    const double l = fma(it.scale, x, shift);
    return it.payoff == TQF_PAYOFF_BASKET_PUT ? l < it.log_strike
                                              : l > it.log_strike;
  }
  return it.payoff == TQF_PAYOFF_BASKET_PUT ? x < it.strike : x > it.strike;
}

// The payoff of a path in the money, else 0.  A table's value at the last
// date stays as it is, negative or NaN.  (Before it the sign makes no
// difference, since no continuation is below 0; but with tab[p] alone the
// compiler schedules the pass of the other payoffs 3 % slower.)
template <int LOGM>
__device__ __forceinline__ double payoff(const PassItem& it, double x,
                                         double shift, const double* tab,
                                         int64_t p, int terminal) {
  if (it.payoff == TQF_PAYOFF_TABLE)
    return terminal || tab[p] > 0 ? tab[p] : 0.0;
  if (!in_money<LOGM>(it, x, shift, tab, p)) return 0.0;
  const double s = LOGM == 2 ? exp_f64(fma(it.scale, x, shift)) : x;
  const double v = it.payoff == TQF_PAYOFF_BASKET_PUT ? it.strike - s
                                                      : s - it.strike;
  return v > 0 ? v : 0;
}

// Standardisation of the basis variable as (mean, factor): 1 / std, or the
// variable's own unit where its spread is zero (the log price's: scale).
struct Centre {
  double mean, fac;
};
__device__ __forceinline__ Centre centre(const double* stat, double shift,
                                         double scale) {
  const double m = stat[0], var = stat[1];
  const double vx = scale * scale * var, mx = shift + scale * m;
  const bool ok = vx > 1e-300 && sqrt(vx) > 1e-12 * fabs(mx);
  return {m, ok ? 1.0 / sqrt(var) : scale};
}

// Time indices of up to kStatDates exercise dates, by value (no copy of a
// host array whose lifetime a capture would have to share).
constexpr int kStatDates = 128;
struct StatDates {
  int32_t idx[kStatDates];
};

// Sum and sum of squares of the basis variable: slice blockIdx.x of date
// blockIdx.y.
template <int LOGM>
__global__ void __launch_bounds__(kThreads)
chain_stats_kernel(const double* __restrict__ paths, int64_t sp, int64_t st,
                   int64_t n, StatDates dates,
                   double* __restrict__ part) {
  __shared__ double red[4][2];
  const double* col = paths + (int64_t)dates.idx[blockIdx.y] * st;
  double s1 = 0, s2 = 0;
  const int64_t stride = (int64_t)gridDim.x * kThreads;
  int64_t p = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  for (; p + 3 * stride < n; p += 4 * stride) {
    double x[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = col[(p + i * stride) * sp];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const double b = basis_var<LOGM>(x[i]);
      s1 += b;
      s2 = fma(b, b, s2);
    }
  }
  for (; p < n; p += stride) {
    const double b = basis_var<LOGM>(col[p * sp]);
    s1 += b;
    s2 = fma(b, b, s2);
  }
  for (int o = 32; o > 0; o >>= 1) {
    s1 += __shfl_xor(s1, o, 64);
    s2 += __shfl_xor(s2, o, 64);
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    red[wave][0] = s1;
    red[wave][1] = s2;
  }
  __syncthreads();
  if (threadIdx.x < 2)
    part[((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * 2 + threadIdx.x] =
        ((red[0][threadIdx.x] + red[1][threadIdx.x]) + red[2][threadIdx.x]) +
        red[3][threadIdx.x];
}

// (mean, variance) per date from the slices, in slice order.
__global__ void __launch_bounds__(64)
chain_mean_kernel(const double* __restrict__ part, int n_dates, int64_t n,
                  double* __restrict__ stats) {
  const int d = blockIdx.x * 64 + threadIdx.x;
  if (d >= n_dates) return;
  double s1 = 0, s2 = 0;
#pragma unroll 8
  for (int i = 0; i < kStatSlices; ++i) {
    s1 += part[((int64_t)d * kStatSlices + i) * 2];
    s2 += part[((int64_t)d * kStatSlices + i) * 2 + 1];
  }
  const double m = s1 / (double)n;
  stats[2 * d] = m;
  stats[2 * d + 1] = s2 / (double)n - m * m;
}

// The regression from the power sums M[m] = sum c^m (m <= 2 deg) and
// M[NX + m] = sum y c^m: columns scaled by 1 / sqrt(G_kk), pivots at or
// below rcond * (largest scaled diagonal) dropped with their column, which
// leaves the fitted values of the pseudo-inverse solution unchanged.
// Monomials outside `mask` count as dropped.
template <int DEG>
__device__ void solve_chain(const double* M, int mask, double rcond,
                            double* coef, int32_t* rank_out) {
  constexpr int K = DEG + 1, NX = 2 * DEG + 1;
  double sc[K], A[K][K], z[K];
  double maxdiag = 0.0;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const double g = M[2 * k];
    sc[k] = ((mask >> k) & 1) && g > 0 ? 1.0 / sqrt(g) : 0.0;
    maxdiag = fmax(maxdiag, g * (sc[k] * sc[k]));
  }
#pragma unroll
  for (int i = 0; i < K; ++i) {
#pragma unroll
    for (int j = 0; j <= i; ++j) A[i][j] = M[i + j] * (sc[i] * sc[j]);
    z[i] = M[NX + i] * sc[i];
  }
  const double thr = rcond * maxdiag;
  int rank = 0;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const double d = A[k][k];
    const bool keep = d > thr && d > 0;
    rank += keep ? 1 : 0;
    const double root = keep ? sqrt(d) : 0.0;
    const double inv = keep ? 1.0 / root : 0.0;
    A[k][k] = inv;
    z[k] *= inv;
#pragma unroll
    for (int i = k + 1; i < K; ++i) A[i][k] *= inv;
#pragma unroll
    for (int i = k + 1; i < K; ++i) {
#pragma unroll
      for (int j = k + 1; j <= i; ++j) A[i][j] -= A[i][k] * A[j][k];
      z[i] -= A[i][k] * z[k];
    }
  }
#pragma unroll
  for (int i = K - 1; i >= 0; --i) {
    double w = z[i];
#pragma unroll
    for (int j = i + 1; j < K; ++j) w -= A[j][i] * z[j];
    z[i] = w * A[i][i];
    coef[i] = z[i] * sc[i];
  }
  if (rank_out) *rank_out = rank;
}

// Workgroup (b, q): payoff q on paths [b rows_per_block, ...), kRows per
// thread and round, the next round's loads in flight over this one.  Four
// waves per SIMD for every degree, although degrees 2 to 4 on log prices
// spill 2, 8 and 30 registers: at three waves four options of degree 3 took
// 541 us (504 at four; 2^18 paths, 20 dates), degree 4 553 (552).
template <int DEG, int LOGM>
__global__ void __launch_bounds__(kThreads, 4)
chain_pass_kernel(PassArgs a) {
  constexpr int K = DEG + 1, NX = 2 * DEG + 1, NM = NX + K;
  constexpr int kRound = kRows * kThreads;
  __shared__ Centre cen[2];
  __shared__ double sums[NM][kThreads];
  const int t = threadIdx.x, q = blockIdx.y;
  const PassItem& it = a.it[q];
  const int64_t p0 = (int64_t)blockIdx.x * a.rows_per_block;
  const int64_t left = a.n - p0;
  const int n_rows = (int)(left < a.rows_per_block ? left : a.rows_per_block);
  double* const values = a.values + (int64_t)q * a.n + p0;
  const double* const col_u = a.col_u + p0 * a.sp;
  const double* const col_m = a.col_m + p0 * a.sp;
  double xu[kRows], xm[kRows], v[kRows];
  double nu[kRows], nm[kRows], nv[kRows];
  // rows past the end load the last path and are not used
  auto load = [&](int base) {
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
      int p = base + i * kThreads + t;
      p = p < n_rows ? p : n_rows - 1;
      nu[i] = col_u[p * a.sp];
      if (!a.last) nm[i] = col_m[p * a.sp];
      if (!a.terminal) nv[i] = values[p];
    }
  };
  load(0);
  if (t < 2)
    cen[t] = centre(t ? a.stat_m : a.stat_u,
                    LOGM == 2 ? (t ? it.shift_m : it.shift_u) : 0.0,
                    LOGM == 2 ? it.scale : 1.0);
  __syncthreads();
  const Centre cu = cen[0], cm = cen[1];
  double dn[K];
#pragma unroll
  for (int m = 0; m < K; ++m)
    dn[m] = a.terminal ? 0.0 : ld_uniform(a.coef, q * (kChainMaxDeg + 1) + m);
  double acc[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) acc[m] = 0.0;
  for (int base = 0; base < n_rows; base += kRound) {
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
      xu[i] = nu[i];
      xm[i] = nm[i];
      v[i] = nv[i];
    }
    if (base + kRound < n_rows) load(base + kRound);
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
      const int pr = base + i * kThreads + t;
      if (pr >= n_rows) continue;
      const int64_t p = p0 + pr;
      const double ex = payoff<LOGM>(it, xu[i], it.shift_u, it.tab_u, p,
                                     a.terminal);
      if (a.terminal) {
        v[i] = ex;
      } else {
        const double c = (basis_var<LOGM>(xu[i]) - cu.mean) * cu.fac;
        double h = dn[DEG];
#pragma unroll
        for (int m = DEG - 1; m >= 0; --m) h = fma(h, c, dn[m]);
        const double cont = h > 0 ? h : 0;
        const double ratio = a.dnum_u ? a.dnum_u[p] / a.dden_u[p]
                                      : it.ratio_u;
        v[i] = ex > cont ? ex : ratio * v[i];
      }
      values[pr] = v[i];
      if (a.last) {
        if (a.zero) a.zero[p] = 0.0;
        if (p >= a.first) {
          const double y = (a.dnum_m ? a.dnum_m[p] / a.dden_m[p]
                                     : it.ratio_m) * v[i];
          acc[0] += y;
          acc[1] = fma(y, y, acc[1]);
        }
      } else if (p < a.n_calib &&
                 in_money<LOGM>(it, xm[i], it.shift_m, it.tab_m, p)) {
        // in-the-money calibration rows only
        const double c = (basis_var<LOGM>(xm[i]) - cm.mean) * cm.fac;
        double w = 1.0, u = (a.dnum_m ? a.dnum_m[p] / a.dden_m[p]
                                      : it.ratio_m) * v[i];
#pragma unroll
        for (int m = 0; m < NX; ++m) {
          acc[m] += w;
          w *= c;
        }
#pragma unroll
        for (int m = NX; m < NM; ++m) {
          acc[m] += u;
          u *= c;
        }
      }
    }
  }
  // the workgroup's sums through LDS, in a fixed order: 32 threads per sum
  // add eight threads' each, then each other's
#pragma unroll
  for (int m = 0; m < NM; ++m) sums[m][t] = acc[m];
  lds_barrier();
  double* out = a.rows + ((int64_t)q * gridDim.x + blockIdx.x) * NM;
  for (int m = t >> 5; m < NM; m += kThreads / 32) {
    double s = 0;
#pragma unroll
    for (int i = 0; i < kThreads / 32; ++i) s += sums[m][(t & 31) + 32 * i];
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) s += __shfl_xor(s, o, 32);
    if ((t & 31) == 0) out[m] = s;
  }
}

// Solve r: workgroup q adds payoff q's rows, column t % NM of rows t / NM,
// t / NM + S, ..., then the S slices in order, and solves the regression on
// one thread (last: the mean and standard error).
template <int DEG>
__global__ void __launch_bounds__(kSolveThreads)
chain_solve_kernel(const double* __restrict__ rows_all, int n_rows, int last,
                   int64_t count, int mask, double rcond,
                   double* __restrict__ coef, int32_t* __restrict__ ranks,
                   int rank_stride, double* __restrict__ results) {
  constexpr int NM = 3 * DEG + 2, S = kSolveThreads / NM;
  __shared__ double red[S * NM], M[NM];
  const int t = threadIdx.x, q = blockIdx.x;
  const double* rows = rows_all + (int64_t)q * n_rows * NM;
  if (t < S * NM) {
    double s = 0;
#pragma unroll 8
    for (int i = t / NM; i < n_rows; i += S)
      s += rows[(int64_t)i * NM + t % NM];
    red[t] = s;
  }
  __syncthreads();
  // 16 lanes per sum, each S / 16 slices, then a fixed-shape tree
  if (t < 16 * NM) {
    const int m = t >> 4;
    double s = 0;
    for (int i = t & 15; i < S; i += 16) s += red[i * NM + m];
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) s += __shfl_xor(s, o, 16);
    if ((t & 15) == 0) M[m] = s;
  }
  __syncthreads();
  if (t != 0) return;
  if (last) {
    const double n = (double)count, mean = M[0] / n;
    const double var = n > 1 ? (M[1] - n * mean * mean) / (n - 1) : 0.0;
    results[2 * q] = mean;
    results[2 * q + 1] = sqrt((var > 0 ? var : 0.0) / n);
  } else {
    solve_chain<DEG>(M, mask, rcond, coef + q * (kChainMaxDeg + 1),
                     ranks ? ranks + (int64_t)q * rank_stride : nullptr);
  }
}

// Paths per workgroup: one round, more once kMaxBlocks workgroups are there.
int64_t rows_per_block(int64_t n) {
  constexpr int64_t round = kRows * kThreads;
  const int64_t r = (n + kMaxBlocks - 1) / kMaxBlocks;
  return (r + round - 1) / round * round;
}

int64_t align256(int64_t b) { return (b + 255) & ~(int64_t)255; }

}  // namespace

int64_t chain_workspace(int64_t n_paths, int n_items, int n_ex) {
  const int64_t rpb = rows_per_block(n_paths);
  const int64_t blocks = (n_paths + rpb - 1) / rpb;
  const int64_t nm = 3 * kChainMaxDeg + 2;
  return align256(blocks * n_items * nm * 8) +
         align256((int64_t)n_items * (kChainMaxDeg + 1) * 8) +
         align256((int64_t)n_ex * kStatSlices * 16) +
         align256((int64_t)n_ex * 16);
}

int run_chain(const ChainProblem& pb, const ChainItem* items, int n_items,
              void* workspace, double* values, double* zero,
              double* results, int32_t* ranks, int rank_stride,
              hipStream_t s) {
  const int64_t n = pb.n_paths;
  const int64_t first = pb.num_calibration > 0 ? pb.num_calibration : 0;
  TQF_REQUIRE(n - first >= 1, "no pricing rows after the calibration samples");
  char* w = (char*)workspace;
  auto take = [&](int64_t bytes) {
    char* p = w;
    w += align256(bytes);
    return p;
  };
  PassArgs a{};
  a.rows_per_block = rows_per_block(n);
  const unsigned grid =
      (unsigned)((n + a.rows_per_block - 1) / a.rows_per_block);
  a.rows = (double*)take((int64_t)grid * n_items *
                         (3 * kChainMaxDeg + 2) * 8);
  double* coef = (double*)take((int64_t)n_items * (kChainMaxDeg + 1) * 8);
  a.coef = coef;
  double* part = (double*)take((int64_t)pb.n_ex * kStatSlices * 16);
  double* stats = (double*)take((int64_t)pb.n_ex * 16);
  for (int d0 = 0; d0 < pb.n_ex; d0 += kStatDates) {
    const int nd = pb.n_ex - d0 < kStatDates ? pb.n_ex - d0 : kStatDates;
    StatDates dates{};
    for (int d = 0; d < nd; ++d) dates.idx[d] = pb.ex_idx[d0 + d];
    hipLaunchKernelGGL(
        pb.basis_log == 1 ? chain_stats_kernel<1> : chain_stats_kernel<0>,
        dim3(kStatSlices, (unsigned)nd), dim3(kThreads), 0, s, pb.paths,
        pb.sp, pb.st, n, dates, part + (int64_t)d0 * kStatSlices * 2);
  }
  hipLaunchKernelGGL(chain_mean_kernel, dim3((unsigned)((pb.n_ex + 63) / 64)),
                     dim3(64), 0, s, part, pb.n_ex, n, stats);
  int rc = check_launch("one-asset chain statistics");
  if (rc) return rc;

  a.sp = pb.sp;
  a.n = n;
  a.n_calib = pb.num_calibration > 0 ? pb.num_calibration : n;
  a.values = values;
  a.zero = zero;
  a.first = first;
  a.n_items = n_items;
  void (*kern)(PassArgs) = nullptr;
  void (*solve)(const double*, int, int, int64_t, int, double, double*,
                int32_t*, int, double*) = nullptr;
#define TQF_CHAIN(DEG)                                              \
  case DEG:                                                         \
    kern = pb.basis_log == 0   ? chain_pass_kernel<DEG, 0>          \
           : pb.basis_log == 1 ? chain_pass_kernel<DEG, 1>          \
                               : chain_pass_kernel<DEG, 2>;         \
    solve = chain_solve_kernel<DEG>;                                \
    break;
  switch (pb.degree) {
    TQF_CHAIN(0)
    TQF_CHAIN(1)
    TQF_CHAIN(2)
    TQF_CHAIN(3)
    TQF_CHAIN(4)
  }
#undef TQF_CHAIN
  TQF_REQUIRE(kern != nullptr, "one-asset chain: degree %d", pb.degree);
  const double* pd = pb.path_discounts;
  for (int r = pb.n_ex - 2; r >= -1; --r) {
    const int u = r + 1;  // the date whose exercise is decided
    a.terminal = u == pb.n_ex - 1;
    a.last = r < 0;
    const int m = a.last ? u : r;
    a.col_u = pb.paths + (int64_t)pb.ex_idx[u] * pb.st;
    a.col_m = pb.paths + (int64_t)pb.ex_idx[m] * pb.st;
    a.stat_u = stats + 2 * u;
    a.stat_m = stats + 2 * m;
    // discount of the value held at date u back to date u (later dates'
    // value) and of date m's continuation: factors e + 1 over e
    if (pd) {
      const int eu = a.terminal ? u : u + 1, em = a.last ? 0 : m + 1;
      a.dnum_u = pd + (int64_t)(eu + 1 < pb.n_ex + 1 ? eu + 1 : eu) * n;
      a.dden_u = pd + (int64_t)eu * n;
      a.dnum_m = pd + (int64_t)(em + 1) * n;
      a.dden_m = pd + (int64_t)em * n;
    }
    for (int q = 0; q < n_items; ++q) {
      const ChainItem& it = items[q];
      PassItem& o = a.it[q];
      o.payoff = it.payoff;
      o.strike = it.strike;
      o.log_strike = it.strike > 0 ? log(it.strike) : -HUGE_VAL;
      o.scale = it.shift ? it.scale : 1.0;
      o.shift_u = it.shift ? it.shift[u] : 0.0;
      o.shift_m = it.shift ? it.shift[m] : 0.0;
      o.ratio_u = a.terminal ? 1.0 : it.df[u + 2] / it.df[u + 1];
      o.ratio_m = a.last ? it.df[1] / it.df[0] : it.df[m + 2] / it.df[m + 1];
      o.tab_u = it.table ? it.table + (int64_t)pb.ex_idx[u] * n : nullptr;
      o.tab_m = it.table ? it.table + (int64_t)pb.ex_idx[m] * n : nullptr;
    }
    hipLaunchKernelGGL(kern, dim3(grid, n_items), dim3(kThreads), 0, s, a);
    hipLaunchKernelGGL(solve, dim3(n_items), dim3(kSolveThreads), 0, s,
                       a.rows, (int)grid, a.last, n - first, pb.mask,
                       pb.rcond, coef, (ranks && !a.last) ? ranks + r : nullptr,
                       rank_stride, results);
    rc = check_launch("one-asset chain");
    if (rc) return rc;
  }
  return TQF_OK;
}

}  // namespace tqf
