// Batched heterogeneous pricing with pathwise adjoint Greeks.
//
// A contract is a European call under GBM (log-Euler, exact in law) or
// Heston (full-truncation log-Euler), with its own parameters, path count,
// uniform step count and maturity.  The host splits every contract into
// work items of `tile` paths (one thread per path, several paths per thread
// when tile > block) and orders them longest first; a persistent grid pulls
// items from an atomic counter, so a 640x spread in work per contract does
// not leave CUs idle.  Each item writes its sums (price, Greeks and their
// squares) to its own row; a second kernel adds the rows of each contract
// in a fixed order.
//
// Greeks are pathwise.  GBM's adjoint does not depend on the path, so it is
// closed form at maturity.  Heston's does: in reverse mode (the default) the
// forward pass stores the state every kSeg steps (about sqrt(steps)), and
// the reverse sweep re-runs each segment from its checkpoint with the same
// Philox counters, keeps the segment's states and normals in registers, and
// walks it backwards; in tangent mode (a contract's greeks_mode) five
// tangents ride along the forward pass instead.  Truncation kinks use the
// subgradient 0 at v = 0.
//
// Forward step (euler_sampling.py:513-537 with the truncated Heston
// coefficients of heston_model.py:143-173, drift r):
//   x' = x + dt (r - v+/2) + sqrt(v+) dw0
//   v' = v + dt k (th - v+) + xi rho sqrt(v+) dw0 + xi sqrt(1-rho^2) sqrt(v+) dw1
#include "common.h"

using namespace tqf;

namespace {

constexpr int kBlockB = 256;
constexpr int kSeg = 16;  // steps per checkpoint segment

__device__ __forceinline__ void normals4(uint32_t p_lo, uint32_t p_hi,
                                         uint32_t blk, uint32_t stream,
                                         const PhiloxKeys<true>& keys, float* z) {
  const u32x4 w = philox4x32_10(u32x4{p_lo, blk, stream, p_hi}, keys);
  box_muller(w.x, w.y, z[0], z[1]);
  box_muller(w.z, w.w, z[2], z[3]);
}

struct Contract {
  int kind, n_steps, greeks_mode;
  uint32_t stream;
  float s0, strike, t, r;
  float sigma;                         // GBM
  float v0, kappa, theta, xi, rho;     // Heston
  int64_t n_paths;
};

__device__ __forceinline__ void load_contract(const tqf_contract* __restrict__ c,
                                              Contract& k) {
  k.kind = c->kind;
  k.n_steps = c->n_steps;
  k.greeks_mode = c->greeks_mode;
  k.stream = c->stream_id;
  k.n_paths = c->n_paths;
  k.s0 = (float)c->s0;
  k.strike = (float)c->strike;
  k.t = (float)c->maturity;
  k.r = (float)c->rate;
  k.sigma = (float)c->sigma;
  k.v0 = (float)c->v0;
  k.kappa = (float)c->kappa;
  k.theta = (float)c->theta;
  k.xi = (float)c->xi;
  k.rho = (float)c->rho;
}

// One GBM path: price and (delta, vega, rho).  Every step adds the same
// drift and scale, so the steps only sum their normals: w = sqrt(dt) sum z
// and x = n drift + sigma w, one addition per step (and one rounding of x
// instead of one per step).
__device__ __forceinline__ void gbm_path(const Contract& c, int64_t p,
                                         uint32_t stream,
                                         const PhiloxKeys<true>& keys,
                                         float* g) {
  const float dt = c.t / (float)c.n_steps;
  const float sdt = sqrtf(dt);
  float sum = 0.f;
  float z[4];
  // four steps per Philox block (block i / 4 serves steps i .. i + 3)
  int i = 0;
  for (; i + 4 <= c.n_steps; i += 4) {
    normals4((uint32_t)p, (uint32_t)(p >> 32), (uint32_t)(i >> 2), stream,
             keys, z);
#pragma unroll
    for (int u = 0; u < 4; ++u) sum += z[u];
  }
  if (i < c.n_steps) {
    normals4((uint32_t)p, (uint32_t)(p >> 32), (uint32_t)(i >> 2), stream,
             keys, z);
#pragma unroll
    for (int u = 0; u < 3; ++u)
      if (i + u < c.n_steps) sum += z[u];
  }
  const float w = sum * sdt;
  const float x = (c.r - 0.5f * c.sigma * c.sigma) * c.t + c.sigma * w;
  const float s = c.s0 * __expf(x);
  const float disc = __expf(-c.r * c.t);
  const float itm = s > c.strike ? 1.f : 0.f;
  const float pay = disc * itm * (s - c.strike);
  const float sb = disc * itm;  // dP/dS_T
  g[0] = pay;
  g[1] = sb * s / c.s0;                                   // delta
  g[2] = sb * s * (w - c.sigma * c.t);                    // vega
  g[3] = -c.t * pay + sb * s * c.t;                       // rho
  g[4] = g[5] = g[6] = g[7] = 0.f;
}

// Per-path constants of the Heston step, each "+ dt a" and "+ b dw" one FMA.
// The log-spot state carries ln(S / S0) - r t (the rate and the spot come
// in at maturity), so its roundings are those of numbers below 1, and the
// variance takes its increment, formed at its own magnitude, in one
// addition.  A constant's rounding acts on every step alike, and near v = 0
// the tangents amplify it by 1 / sqrt(v) and more: the constants are
// rounded once from float64, and sqrt(dt) keeps its low part.
struct HestonConst {
  float sdt, sdt_lo;      // sqrt(dt)
  float mdt2;             // -dt / 2
  float mdtk, theta;      // -dt kappa
  float xi, rho, s1r;
};

__device__ __forceinline__ HestonConst heston_const(const Contract& c) {
  const double dt = (double)c.t / c.n_steps, sdt = sqrt(dt);
  HestonConst k;
  k.sdt = (float)sdt;
  k.sdt_lo = (float)(sdt - (double)k.sdt);
  k.mdt2 = (float)(-0.5 * dt);
  k.mdtk = (float)(-dt * c.kappa);
  k.theta = c.theta;
  k.xi = c.xi;
  k.rho = c.rho;
  k.s1r = (float)sqrt(1.0 - (double)c.rho * c.rho);
  return k;
}

// z sqrt(dt)
__device__ __forceinline__ float heston_dw(const HestonConst& k, float z) {
  return fma_r(z, k.sdt, z * k.sdt_lo);
}

// Forward Heston step from v's truncation vp and its root sq, the
// increments dw0 and cu = rho dw0 + sqrt(1 - rho^2) dw1.
__device__ __forceinline__ void heston_step(const HestonConst& k, float vp,
                                            float sq, float dw0, float cu,
                                            float& x, float& v) {
  x = fma_r(sq, dw0, fma_r(vp, k.mdt2, x));
  v += fma_r(k.xi * sq, cu, k.mdtk * (vp - k.theta));
}

// Discounted payoff and dP/d ln S of the final state.
__device__ __forceinline__ void heston_payoff(const Contract& c, float x,
                                              float& pay, float& xb) {
  const float e = __expf(fma_r(c.r, c.t, x));
  const float disc = __expf(-c.r * c.t);
  // one rounding of S - K, whatever the caller contracts
  const float gain = fma_r(c.s0, e, -c.strike);
  // NaN compares false and stays
  pay = gain <= 0.f ? 0.f : disc * gain;
  xb = gain <= 0.f ? 0.f : disc * (c.s0 * e);
}

// One Heston path with the checkpointed reverse sweep.  ck: this thread's
// checkpoint column (stride `cstride` floats between segments).
__device__ void heston_path(const Contract& c, int64_t p, uint32_t stream,
                            const PhiloxKeys<true>& keys,
                            float* __restrict__ ck, int64_t cstride,
                            float* g) {
  const int n = c.n_steps;
  const HestonConst k = heston_const(c);
  const float dt = c.t / (float)n;
  const uint32_t plo = (uint32_t)p, phi = (uint32_t)(p >> 32);
  float x = 0.f, v = c.v0;
  float z[4];
  const int nseg = (n + kSeg - 1) / kSeg;
  for (int i = 0; i < n; ++i) {
    if (i % kSeg == 0) ck[(int64_t)(i / kSeg) * cstride] = v;
    if ((i & 1) == 0)
      normals4(plo, phi, (uint32_t)(i >> 1), stream, keys, z);
    const float dw0 = heston_dw(k, (i & 1) ? z[2] : z[0]);
    const float dw1 = heston_dw(k, (i & 1) ? z[3] : z[1]);
    const float vp = v > 0.f ? v : 0.f;
    heston_step(k, vp, __builtin_amdgcn_sqrtf(vp), dw0,
                fma_r(k.s1r, dw1, k.rho * dw0), x, v);
  }
  float pay, xb;
  heston_payoff(c, x, pay, xb);
  // adjoints; the log-spot's, xb, is constant (dx'/dx = 1), so the sweep
  // needs the variance states only
  float vb = 0.f;
  float kb = 0.f, tb = 0.f, xib = 0.f, rhob = 0.f;
  const float drho_s = -c.rho / k.s1r;  // d sqrt(1-rho^2) / d rho
  for (int sgi = nseg - 1; sgi >= 0; --sgi) {
    const int i0 = sgi * kSeg;
    float vs_[kSeg], z0s[kSeg], z1s[kSeg];
    float cx = 0.f, cv = ck[(int64_t)sgi * cstride];
#pragma unroll
    for (int u = 0; u < kSeg; ++u) {
      const int i = i0 + u;
      if (i < n) {
        if ((u & 1) == 0)
          normals4(plo, phi, (uint32_t)(i >> 1), stream, keys, z);
        z0s[u] = heston_dw(k, (u & 1) ? z[2] : z[0]);
        z1s[u] = heston_dw(k, (u & 1) ? z[3] : z[1]);
        vs_[u] = cv;
        const float vp = cv > 0.f ? cv : 0.f;
        heston_step(k, vp, __builtin_amdgcn_sqrtf(vp), z0s[u],
                    fma_r(k.s1r, z1s[u], k.rho * z0s[u]), cx, cv);
      }
    }
#pragma unroll
    for (int u = kSeg - 1; u >= 0; --u) {
      const int i = i0 + u;
      if (i < n) {
        const float v0 = vs_[u];
        const float vp = v0 > 0.f ? v0 : 0.f;
        const float sq = __builtin_amdgcn_sqrtf(vp);
        const float dw0 = z0s[u], dw1 = z1s[u];
        const float cu = fma_r(k.s1r, dw1, k.rho * dw0);
        const float sqb = fma_r(xb, dw0, vb * (k.xi * cu));
        float vpb = fma_r(k.mdt2, xb, k.mdtk * vb);
        // d sqrt(v+) / dv+ = 1 / (2 sqrt(v+)) by the hardware reciprocal
        vpb += sq > 0.f ? sqb * 0.5f * __builtin_amdgcn_rcpf(sq) : 0.f;
        kb += vb * dt * (c.theta - vp);
        tb += vb * dt * c.kappa;
        xib += vb * (sq * cu);
        rhob += vb * (k.xi * sq) * fma_r(drho_s, dw1, dw0);
        vb = vb + (v0 > 0.f ? vpb : 0.f);
      }
    }
  }
  g[0] = pay;
  g[1] = xb / c.s0;              // delta
  g[2] = vb;                     // d/dv0
  g[3] = -c.t * pay + xb * c.t;  // rho (rate): x_T carries r T
  g[4] = kb;
  g[5] = tb;
  g[6] = xib;
  g[7] = rhob;
}

// One Heston path with forward-mode (tangent) Greeks: the tangents of
// (x, v) for v0, kappa, theta, xi and rho ride along the forward pass, so
// there is no checkpoint, no second pass and no second draw of the normals
// (which dominate a step's cost).  Same pathwise estimator as the reverse
// sweep above, with the same subgradient 0 at v <= 0: the price depends on
// x_T only, so each Greek is x-bar ("xb" below) times the x-tangent, and
// delta and rho are closed form as in the reverse sweep.
//   x'  <- x' + A v',  A = -dt/2 + h dw0
//   v'  <- v' + (B v' + dv'/dp),  B = -dt kappa + h xi cu
// with h = 1 / (2 sqrt v) and cu = rho dw0 + s dw1, A and B 0 where v <= 0.
// They are the same for the five tangents, so a step is an FMA for x' and an
// FMA and an addition for v' (a select, a product and four FMAs when the
// factors are applied one by one).  B is the increment, not 1 + B: dt kappa
// of 1e-3 would keep 14 bits beside the 1, with the same rounding in every
// step (median error of d/dv0 over a book 1.4e-6, as an increment 1.2e-7).
// Bound by VALU issue: 75 instructions and about 250 cycles a step and wave,
// of which half a Philox block is 66 and the Box-Muller pair 62; five waves
// per SIMD (the launch bound keeps it at 96 registers).  A book of 256
// contracts (8.3e9 GBM and 8.3e9 Heston path-steps) takes 4.47 ms, 5.47 with
// the factors applied one by one, 4.28 with 1 + B.
__device__ void heston_path_tangent(const Contract& c, int64_t p,
                                    uint32_t stream,
                                    const PhiloxKeys<true>& keys, float* g) {
  const int n = c.n_steps;
  const HestonConst k = heston_const(c);
  const double dt = (double)c.t / n;
  const float drho_s = -c.rho / k.s1r;  // d sqrt(1-rho^2) / d rho
  const float mdt = (float)-dt;
  const uint32_t plo = (uint32_t)p, phi = (uint32_t)(p >> 32);
  float x = 0.f, v = c.v0;
  // tangents of (x, v) for v0, kappa, theta, xi, rho
  float tx[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
  float tv[5] = {1.f, 0.f, 0.f, 0.f, 0.f};
  auto step = [&](float z0, float z1) {
    const bool pos = v > 0.f;
    const float vp = pos ? v : 0.f;
    const float sq = __builtin_amdgcn_sqrtf(vp);
    const float dw0 = heston_dw(k, z0), dw1 = heston_dw(k, z1);
    const float cu = fma_r(k.s1r, dw1, k.rho * dw0);
    // d sqrt(v+) / dv+ by the hardware reciprocal (one instruction in
    // place of a correctly rounded division by sq); 0 where the root is, as
    // in the reverse sweep (the hardware root of a subnormal v is 0)
    const float h = sq > 0.f ? 0.5f * __builtin_amdgcn_rcpf(sq) : 0.f;
    const float a = pos ? fma_r(h, dw0, k.mdt2) : 0.f;
    const float b = pos ? fma_r(h * k.xi, cu, k.mdtk) : 0.f;
#pragma unroll
    for (int q = 0; q < 5; ++q) tx[q] = fma_r(a, tv[q], tx[q]);
    tv[0] = fma_r(b, tv[0], tv[0]);
    tv[1] += fma_r(b, tv[1], mdt * (vp - k.theta));               // kappa
    tv[2] += fma_r(b, tv[2], -k.mdtk);                            // theta
    tv[3] += fma_r(b, tv[3], sq * cu);                            // xi
    tv[4] += fma_r(b, tv[4], (k.xi * sq) * fma_r(drho_s, dw1, dw0));  // rho
    // the state update of the reverse-mode path, so both modes price the
    // same paths bit for bit
    heston_step(k, vp, sq, dw0, cu, x, v);
  };
  // two steps per Philox block
  float z[4];
  int i = 0;
  for (; i + 2 <= n; i += 2) {
    normals4(plo, phi, (uint32_t)(i >> 1), stream, keys, z);
    step(z[0], z[1]);
    step(z[2], z[3]);
  }
  if (i < n) {
    normals4(plo, phi, (uint32_t)(i >> 1), stream, keys, z);
    step(z[0], z[1]);
  }
  float pay, xb;
  heston_payoff(c, x, pay, xb);
  g[0] = pay;
  g[1] = xb / c.s0;             // delta
  g[2] = xb * tx[0];            // d/dv0
  g[3] = -c.t * pay + xb * c.t; // rho (rate): x_T carries r T
  g[4] = xb * tx[1];
  g[5] = xb * tx[2];
  g[6] = xb * tx[3];
  g[7] = xb * tx[4];
}

// Persistent kernel: items from `counter`, sums per item into `item_sums`
// [n_items][2 * kStats].
constexpr int kStats = 8;

// kAdjoint false: the kernel has no reverse sweep (a Heston contract that
// asks for adjoint Greeks gets the forward tangents, the same pathwise
// estimator), so it needs far fewer registers and runs more waves per SIMD.
template <bool kAdjoint>
__global__ void __launch_bounds__(kBlockB, kAdjoint ? 3 : 5)
batch_kernel(const tqf_contract* __restrict__ contracts,
             const tqf_work_item* __restrict__ items,
             const int32_t* __restrict__ order, int n_items,
             uint32_t k0, uint32_t k1, int* __restrict__ counter,
             float* __restrict__ ckpt, int64_t ckpt_per_block,
             int max_seg, double* __restrict__ item_sums, int use_counter) {
  __shared__ int s_item;
  __shared__ double red[kBlockB / kWave][2 * kStats];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float* ck = ckpt + (int64_t)blockIdx.x * ckpt_per_block + threadIdx.x;
  PhiloxKeys<true> keys;
  keys.init(k0, k1);
  int next = blockIdx.x;
  for (;;) {
    if (use_counter) {
      __syncthreads();
      if (threadIdx.x == 0) s_item = atomicAdd(counter, 1);
      __syncthreads();
      next = s_item;
    }
    if (next >= n_items) break;
    const int row = order ? order[next] : next;
    const tqf_work_item it = items[row];
    Contract c;
    load_contract(contracts + it.contract, c);
    float acc[2 * kStats];
#pragma unroll
    for (int q = 0; q < 2 * kStats; ++q) acc[q] = 0.f;
    for (int64_t p = it.first_path + threadIdx.x; p < it.first_path + it.n_paths;
         p += kBlockB) {
      float g[kStats];
      if (c.kind == TQF_CONTRACT_GBM)
        gbm_path(c, p, c.stream, keys, g);
      else if (!kAdjoint || c.greeks_mode == TQF_GREEKS_TANGENT ||
               (c.n_steps + kSeg - 1) / kSeg > max_seg)
        // a contract with more steps than the checkpoint workspace holds
        // (n_steps > max_steps) takes the forward tangents, the same
        // estimator, rather than write past its checkpoint column
        heston_path_tangent(c, p, c.stream, keys, g);
      else
        heston_path(c, p, c.stream, keys, ck, kBlockB, g);
#pragma unroll
      for (int q = 0; q < kStats; ++q) {
        acc[q] += g[q];
        acc[kStats + q] += g[q] * g[q];
      }
    }
    // wave reduction (float), then block (double)
#pragma unroll
    for (int q = 0; q < 2 * kStats; ++q) {
      float v = acc[q];
      for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
      if (lane == 0) red[wave][q] = (double)v;
    }
    __syncthreads();
    if (threadIdx.x < 2 * kStats) {
      double s = 0;
      for (int w = 0; w < kBlockB / kWave; ++w) s += red[w][threadIdx.x];
      item_sums[(int64_t)row * 2 * kStats + threadIdx.x] = s;
    }
    __syncthreads();
    if (!use_counter) next += gridDim.x;
  }
}

__global__ void zero_counter_kernel(int* c) { *c = 0; }

// Per contract (one workgroup): sums its items' rows -> mean, SE.  Thread t
// adds column t % 16 of rows t / 16, t / 16 + 16, ... (a wave reads four
// whole rows), then the 16 slices are added in slice order.  One thread per
// contract walked up to 128 rows of 16 doubles by itself: 70 us for 256
// contracts of up to 2^18 paths.
__global__ void __launch_bounds__(256)
batch_finalize_kernel(const double* __restrict__ item_sums,
                      const int* __restrict__ contract_first_item,
                      const int* __restrict__ contract_n_items,
                      const tqf_contract* __restrict__ contracts,
                      double* __restrict__ out) {
  constexpr int kCols = 2 * kStats, kSlices = 256 / kCols;
  __shared__ double red[kSlices][kCols];
  const int c = blockIdx.x;
  const int col = threadIdx.x % kCols, slice = threadIdx.x / kCols;
  const double* rows = item_sums + (int64_t)contract_first_item[c] * kCols;
  const int m = contract_n_items[c];
  double s = 0;
#pragma unroll 4
  for (int i = slice; i < m; i += kSlices) s += rows[(int64_t)i * kCols + col];
  red[slice][col] = s;
  __syncthreads();
  if (threadIdx.x >= kStats) return;
  double s1 = 0, s2 = 0;
  for (int q = 0; q < kSlices; ++q) {
    s1 += red[q][threadIdx.x];
    s2 += red[q][kStats + threadIdx.x];
  }
  const double n = (double)contracts[c].n_paths;
  const double mean = s1 / n;
  double var = n > 1 ? (s2 - n * mean * mean) / (n - 1) : 0.0;
  out[(int64_t)c * kCols + threadIdx.x] = mean;
  out[(int64_t)c * kCols + kStats + threadIdx.x] =
      sqrt((var > 0 ? var : 0) / n);
}

}  // namespace

extern "C" int64_t tqf_batch_workspace_size(int32_t n_items, int32_t n_blocks,
                                            int32_t max_steps) {
  const int64_t nseg = (max_steps + kSeg - 1) / kSeg;
  const int64_t sums = ((int64_t)n_items * 2 * kStats * 8 + 255) & ~(int64_t)255;
  return sums + 256 + (int64_t)n_blocks * kBlockB * nseg * 4;
}

extern "C" int tqf_batch_price(const tqf_contract* contracts,
                               int32_t n_contracts,
                               const tqf_work_item* items,
                               const int32_t* order, int32_t n_items,
                               const int32_t* contract_first_item,
                               const int32_t* contract_n_items, uint64_t seed,
                               int32_t n_blocks, int32_t max_steps,
                               int32_t flags, void* workspace,
                               double* out, void* stream) {
  clear_error();
  TQF_REQUIRE(contracts && items && contract_first_item && contract_n_items &&
                  workspace && out,
              "null argument");
  TQF_REQUIRE(n_contracts >= 1 && n_items >= 1 && n_blocks >= 1,
              "empty batch");
  TQF_REQUIRE(max_steps >= 1 && max_steps <= (1 << 20), "bad max_steps");
  const hipStream_t s = (hipStream_t)stream;
  char* w = (char*)workspace;
  double* item_sums = (double*)w;
  w += ((int64_t)n_items * 2 * kStats * 8 + 255) & ~(int64_t)255;
  int* counter = (int*)w;
  w += 256;
  float* ckpt = (float*)w;
  const int nseg = (max_steps + kSeg - 1) / kSeg;
  const int64_t per_block = (int64_t)kBlockB * nseg;
  hipLaunchKernelGGL(zero_counter_kernel, 1, 1, 0, s, counter);
  const int use_counter = flags & TQF_BATCH_COUNTER;
  if (flags & TQF_BATCH_TANGENT_ONLY)
    hipLaunchKernelGGL(batch_kernel<false>, n_blocks, kBlockB, 0, s, contracts,
                       items, order, n_items, (uint32_t)seed,
                       (uint32_t)(seed >> 32), counter, ckpt, per_block,
                       nseg, item_sums, use_counter);
  else
    hipLaunchKernelGGL(batch_kernel<true>, n_blocks, kBlockB, 0, s, contracts,
                       items, order, n_items, (uint32_t)seed,
                       (uint32_t)(seed >> 32), counter, ckpt, per_block,
                       nseg, item_sums, use_counter);
  hipLaunchKernelGGL(batch_finalize_kernel, n_contracts, 256, 0, s, item_sums,
                     contract_first_item, contract_n_items, contracts, out);
  return check_launch("tqf_batch_price");
}
