// Shared device and host helpers of the tqf HIP library (gfx950, wave64).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <string>

#include "../../include/tqf.h"

namespace tqf {

// ---------------------------------------------------------------- errors --

// Sets the calling thread's error message and returns `code`.
int set_error(int code, const char* fmt, ...);
void clear_error();

#define TQF_REQUIRE(cond, ...)                         \
  do {                                                 \
    if (!(cond)) return ::tqf::set_error(TQF_EINVAL, __VA_ARGS__); \
  } while (0)

// Returns 0 or the launch error (positive hipError_t) with a message.
int check_launch(const char* what);

constexpr int kWave = 64;

// Workgroup barrier that orders LDS only: the fences are limited to the
// local address space, so the wave's outstanding global stores are not
// waited for (__syncthreads waits for them).  For loops that stage data in
// LDS and stream it out: the next stage may overwrite the LDS buffer while
// the previous stage's stores are still in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// ------------------------------------------------------------ Philox4x32 --
// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11): 10 rounds of
// (hi, lo) = mulhilo(M, c) with a Weyl key schedule.
struct u32x4 {
  uint32_t x, y, z, w;
};

// a ^ b ^ c in one instruction.
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) {
  return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
}

// The ten rounds' keys of one (k0, k1), held in vector registers.  A VALU
// instruction on gfx950 issues in 2 cycles per wave when its operands are
// vector registers, inline constants or literals and in 4 when one is a
// scalar register (measured: v_xor_b32 2.5 against 4.4 cycles, v_bitop3_b32
// 2.7 against 4.3), and with scalar keys a round is two plain XORs per word.
// Vector keys make it one three-input v_bitop3_b32: a block of four words
// takes 156 cycles per wave in place of 239, of which the 20 multiplies
// are 91.  The cost is 20 registers (the asm keeps them from being formed
// again at each use), which the float64 kernels do not have to spare: they
// keep scalar keys (kVector false) and gain only the three-input XOR.
template <bool kVector>
struct PhiloxKeys {
  uint32_t k[20];

  __device__ __forceinline__ void init(uint32_t k0, uint32_t k1) {
    constexpr uint32_t W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
#pragma unroll
    for (int r = 0; r < 10; ++r) {
      k[2 * r] = k0;
      k[2 * r + 1] = k1;
      if constexpr (kVector)
        asm volatile("" : "+v"(k[2 * r]), "+v"(k[2 * r + 1]));
      k0 += W0;
      k1 += W1;
    }
  }
};

template <bool kVector>
__device__ __forceinline__ u32x4 philox4x32_10(u32x4 c,
                                               const PhiloxKeys<kVector>& p) {
  constexpr uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u;
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    // one 32x32->64 multiply per word (v_mad_u64_u32) gives both halves
    const uint64_t p0 = (uint64_t)M0 * c.x;
    const uint64_t p1 = (uint64_t)M1 * c.z;
    c = u32x4{xor3((uint32_t)(p1 >> 32), c.y, p.k[2 * r]), (uint32_t)p1,
              xor3((uint32_t)(p0 >> 32), c.w, p.k[2 * r + 1]), (uint32_t)p0};
  }
  return c;
}

// Box-Muller on one word pair.  float: 24-bit uniforms, u in (0, 1];
// v_sin/v_cos take their argument in turns, so 2*pi*t needs no multiply.
__device__ __forceinline__ void box_muller(uint32_t a, uint32_t b, float& z0,
                                           float& z1) {
  const float u = (float)((a >> 8) + 1u) * 0x1p-24f;
  const float t = (float)(b >> 8) * 0x1p-24f;
  // v_log_f32 is log2: -2 ln u = -2 ln2 log2 u (u >= 2^-24, no denormals)
  const float r =
      __builtin_amdgcn_sqrtf(-1.3862943611198906f * __builtin_amdgcn_logf(u));
  z0 = r * __builtin_amdgcn_cosf(t);
  z1 = r * __builtin_amdgcn_sinf(t);
}

__device__ __forceinline__ void box_muller(uint32_t a, uint32_t b, double& z0,
                                           double& z1) {
  const double u = ((double)a + 1.0) * 0x1p-32;
  const double t = (double)b * 0x1p-32;
  const double r = sqrt(-2.0 * log(u));
  double s, c;
  sincospi(2.0 * t, &s, &c);
  z0 = r * c;
  z1 = r * s;
}

// ---------------------------------------------------------------- erfinv --
// float32: erfinv(x) = x P(w), w = -ln(1 - x^2); P is a degree-8 polynomial
// in w - 2.5 (w < 5) or sqrt(w) - 3 (w >= 5).  The form (the variable w, the
// split at w = 5 and the two shifted polynomial variables) is the one M.
// Giles published for single precision ("Approximating the erfinv
// function", GPU Computing Gems Jade Edition, 2011); the coefficients were
// refitted for this library by least squares against scipy
// (csrc/fit_erfinv.py); max relative error 2.9e-7 over float32 inputs with
// 1 - x^2 rounded once.
__device__ __forceinline__ float erfinv_f32(float x) {
  // w = -ln(1 - x^2) = -ln2 log2(1 - x^2); 1 - x^2 >= 2^-24 here, so the
  // raw v_log_f32 needs no denormal scaling
  float w = -0.69314718055994531f *
            __builtin_amdgcn_logf(__builtin_fmaf(-x, x, 1.0f));
  float p;
  if (w < 5.0f) {
    w = w - 2.5f;
    p = 2.798955610e-08f;
    p = __builtin_fmaf(p, w, 3.430734327e-07f);
    p = __builtin_fmaf(p, w, -3.522236486e-06f);
    p = __builtin_fmaf(p, w, -4.389634286e-06f);
    p = __builtin_fmaf(p, w, 2.185773789e-04f);
    p = __builtin_fmaf(p, w, -1.253729840e-03f);
    p = __builtin_fmaf(p, w, -4.177678720e-03f);
    p = __builtin_fmaf(p, w, 2.466407436e-01f);
    p = __builtin_fmaf(p, w, 1.501409417e+00f);
  } else {
    w = __builtin_amdgcn_sqrtf(w) - 3.0f;
    p = -1.435658875e-04f;
    p = __builtin_fmaf(p, w, 6.800158921e-05f);
    p = __builtin_fmaf(p, w, 1.270877357e-03f);
    p = __builtin_fmaf(p, w, -3.640709435e-03f);
    p = __builtin_fmaf(p, w, 5.775239294e-03f);
    p = __builtin_fmaf(p, w, -7.631052573e-03f);
    p = __builtin_fmaf(p, w, 9.433467592e-03f);
    p = __builtin_fmaf(p, w, 1.001674574e+00f);
    p = __builtin_fmaf(p, w, 2.832977048e+00f);
  }
  return p * x;
}

// float64 uses the device math library's erfinv.
__device__ __forceinline__ double erfinv_any(double x) { return erfinv(x); }
__device__ __forceinline__ float erfinv_any(float x) { return erfinv_f32(x); }

// Normal from a Sobol integer, reference transform (multivariate_normal.py:420):
// u = cast(int) * 2^-nd in the working type, z = erfinv((u - .5) * 2) sqrt 2.
template <typename R>
__device__ __forceinline__ R sobol_ref_normal(uint32_t v, R scale) {
  const R u = (R)v * scale;
  return erfinv_any((u - (R)0.5) * (R)2) * (R)1.4142135623730951;
}

// Engine transform of a 32-digit shifted point in float64: q = 2u - 1
// formed exactly from u = (v + 1/2) 2^-32.  (float32 uses the LDS table of
// normals.h.)
__device__ __forceinline__ double sobol_shifted_normal(uint32_t v, double) {
  const double q = ((double)v + 0.5) * 0x1p-31 - 1.0;
  return erfinv(q) * 1.4142135623730951;
}

// Uniform loads through the constant address space: per-step tables that
// every lane reads at the same index become scalar (s_load) loads.
template <typename T>
__device__ __forceinline__ T ld_uniform(const T* p, int64_t i) {
  return ((const __attribute__((address_space(4))) T*)p)[i];
}

// exp(x): 2^n e^r with r = x - n ln 2 (ln 2 in the two parts published with
// Sun's fdlibm: the product of n and the first is exact) and the Taylor sum
// of e^r to r^13 (|r| <= 0.347: remainder 5e-18).  The coefficients come
// through scalar loads and enter the FMAs as scalar operands: 22 float64
// instructions, where the math library's function takes 47 instructions with
// its coefficients moved into vector registers at every call.  0 below -746,
// infinity from 709.79 on (x itself stays in r, so an infinite x reaches the
// sum), NaN for NaN: the comparison is false for it, where fmax would return
// its other operand.
static __constant__ double kExpCoef[12] = {
    1.0 / 6227020800.0, 1.0 / 479001600.0, 1.0 / 39916800.0, 1.0 / 3628800.0,
    1.0 / 362880.0,     1.0 / 40320.0,     1.0 / 5040.0,     1.0 / 720.0,
    1.0 / 120.0,        1.0 / 24.0,        1.0 / 6.0,        0.5};

__device__ __forceinline__ double exp_f64(double x) {
  x = x < -746.0 ? -746.0 : x;
  const double n = __builtin_rint(fmin(x, 710.0) * 1.4426950408889634);
  double r = fma(n, -6.93147180369123816490e-01, x);
  r = fma(n, -1.90821492927058770002e-10, r);
  double p = ld_uniform(kExpCoef, 0);
#pragma unroll
  for (int k = 1; k < 12; ++k) p = fma(p, r, ld_uniform(kExpCoef, k));
  p = fma(p, r, 1.0);
  p = fma(p, r, 1.0);
  return ldexp(p, (int)n);
}

// ------------------------------------------------------------ wave helpers --
__device__ __forceinline__ float read_lane(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ double read_lane(double v, int lane) {
  const int64_t b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffff), lane);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double(((int64_t)hi << 32) | (uint32_t)lo);
}

__device__ __forceinline__ float fma_r(float a, float b, float c) {
  return __builtin_fmaf(a, b, c);
}
__device__ __forceinline__ double fma_r(double a, double b, double c) {
  return __builtin_fma(a, b, c);
}

// max(x, 0) as one integer max on the bit pattern: negative values (and
// -0) have the sign bit set, so they compare below 0; NaN with the sign bit
// clear passes through unchanged.
__device__ __forceinline__ float pos_part(float x) {
  return __int_as_float(max(__float_as_int(x), 0));
}
__device__ __forceinline__ double pos_part(double x) {
  return __longlong_as_double(max(__double_as_longlong(x), 0ll));
}

__device__ __forceinline__ float fast_exp(float x) { return __expf(x); }
__device__ __forceinline__ double fast_exp(double x) { return exp(x); }
__device__ __forceinline__ float fast_sqrt(float x) {
  return __builtin_amdgcn_sqrtf(x);
}
__device__ __forceinline__ double fast_sqrt(double x) { return sqrt(x); }
// a / b: float32 as a times the hardware reciprocal (about 1 ulp each, two
// instructions in place of the correctly rounded division's sequence);
// float64 exact
__device__ __forceinline__ float fast_div(float a, float b) {
  return a * __builtin_amdgcn_rcpf(b);
}
__device__ __forceinline__ double fast_div(double a, double b) {
  return a / b;
}

// log2 Phi(-z) for z >= -0.9 (below, its value at -0.9): -z^2 / (2 ln 2) plus
// a polynomial for the slowly varying rest, held at z = 6.5 beyond (csrc/
// fit_icdf.py): within 4e-7 below z = 1 and 2^-20 of the result up to 6.5,
// 1e-2 of it beyond.  Every constant is an instruction's literal.  1 - Phi(z)
// from erf has lost all its digits at z = 5.4.
__device__ __forceinline__ float log2_normal_tail(float z) {
  z = fmaxf(z, -0.9f);
  const float h = fminf(z, 6.5f);
  float p = -0x1.519f2ap-33f;
  p = __builtin_fmaf(p, h, 0x1.703b14p-28f);
  p = __builtin_fmaf(p, h, -0x1.4d3566p-24f);
  p = __builtin_fmaf(p, h, 0x1.3311c6p-21f);
  p = __builtin_fmaf(p, h, -0x1.dbba8cp-20f);
  p = __builtin_fmaf(p, h, -0x1.501e92p-18f);
  p = __builtin_fmaf(p, h, 0x1.35e5ccp-14f);
  p = __builtin_fmaf(p, h, -0x1.3a9346p-12f);
  p = __builtin_fmaf(p, h, 0x1.ac6d46p-15f);
  p = __builtin_fmaf(p, h, 0x1.c3e500p-8f);
  p = __builtin_fmaf(p, h, -0x1.ad6b6ap-5f);
  p = __builtin_fmaf(p, h, 0x1.0c6a58p-2f);
  p = __builtin_fmaf(p, h, -0x1.26aec6p+0f);
  p = __builtin_fmaf(p, h, -1.0f);
  return __builtin_fmaf(z * -0.72134752f, z, p);
}

inline int dtype_size(int dtype) { return dtype == TQF_F64 ? 8 : 4; }

}  // namespace tqf
