// One-asset Longstaff-Schwartz date chain (lsm_chain.hip), shared by
// tqf_lsm_price and tqf_lsm_price_shared.
#pragma once

#include <stdint.h>

#include "common.h"

namespace tqf {

constexpr int kChainMaxDeg = 4;
constexpr int kChainMaxItems = 16;

// One payoff on the shared paths.
struct ChainItem {
  int payoff;             // TQF_PAYOFF_*
  double strike;
  const double* table;    // TQF_PAYOFF_TABLE: [n_times][n_paths]
  const double* df;       // host [n_ex + 1] padded discount factors
  const double* shift;    // host [n_ex] or null: with basis_log 2 the log
  double scale;           // price is shift[e] + scale * stored value
};

struct ChainProblem {
  const double* paths;    // element (p, t) at paths[p sp + t st]
  int64_t sp, st, n_paths;
  int degree;
  int mask;               // bit m: the monomial c^m is in the basis
  int basis_log;
  double rcond;
  int64_t num_calibration;       // 0: every row
  const double* path_discounts;  // [n_ex + 1][n_paths] or null
  const int32_t* ex_idx;  // host [n_ex]
  int n_ex;
};

// Bytes of device workspace for n_items payoffs and n_ex dates.
int64_t chain_workspace(int64_t n_paths, int n_items, int n_ex);

// values [n_items][n_paths]: each path's value at the first exercise date
// (before the final discount); zero (optional) [n_paths] is cleared; results
// [n_items][2] (price, standard error); ranks (optional)
// [n_items][rank_stride].
int run_chain(const ChainProblem& pb, const ChainItem* items, int n_items,
              void* workspace, double* values, double* zero, double* results,
              int32_t* ranks, int rank_stride, hipStream_t s);

}  // namespace tqf
