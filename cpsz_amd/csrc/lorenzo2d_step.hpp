// One element of the 2D Lorenzo codec, shared by the wavefront kernels and
// the host emulation used to test the arithmetic on the CPU.
//
// Compressor step (include/sz_compression_utils.hpp:50-65 with
// pred = (L + U) - UL in float, include/sz_prediction.hpp:10-14):
//   diff = x - pred (float, widened); quant_diff = |diff|/E + 1 (double);
//   unpredictable unless quant_diff < 65536 and |x' - x| <= E, where
//   x' = (float)(pred + 2 q E) and q = +-(int)(quant_diff / 2).
// With E = 2^(2 id - 52) a power of two the FP32 form below is exact. With
// a = |diff|/E (exact, a scaling by a power of two):
//   |diff|/E + 1 < 65536   <=>  a < 65535  <=>  q < 32768
//   q = floor((floor(a) + 1) / 2) == floor(fma(|diff|, 1/(2E), 1/2 - 2^-25)):
//       the real (a + 1)/2 has the same floor as (floor(a) + 1)/2. Its FP32
//       rounding moves the floor only at a = 1 - 2^-24, where the tie rounds
//       to 1; the constant 2^-25 below 1/2 keeps that one below 1 and leaves
//       every odd a at its integer (checked over every float a).
//   (float)(pred + 2qE)    ==   fma(q, 2E, pred) in FP32, because
//       2qE is an exact float (|2q| <= 2^16, id <= 81) and a double sum of two
//       floats rounded to float equals the single FP32 rounding (the double
//       sum is exact when the exponents differ by <= 28; otherwise the smaller
//       term is below 1/32 ulp of the larger and both roundings return it).
// Eb code c: 0 = zero precision (always unpredictable), c >= 1: id = c - 1.
// `shift` is log2 of the id base: 2 for the offline codec (E = 4^id eps), 1
// for offline_log (E = 2^id eps, ids <= 62, never the wide path); the
// argument above holds for both, since E stays a power of two.
//
// The steps come in two halves: what depends on the element alone (l2d_prep*,
// l2d_code, run by the wavefront's helper waves) and what depends on the
// prediction (l2d_quantize, l2d_restore), which is the recurrence and is kept
// as short as it can be.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

namespace cpsz {

__host__ __device__ inline uint32_t l2d_bits(float x) {
  uint32_t u;
  __builtin_memcpy(&u, &x, 4);
  return u;
}
__host__ __device__ inline float l2d_float(uint32_t u) {
  float x;
  __builtin_memcpy(&x, &u, 4);
  return x;
}
__host__ __device__ inline uint64_t l2d_bits(double x) {
  uint64_t u;
  __builtin_memcpy(&u, &x, 8);
  return u;
}
__host__ __device__ inline double l2d_double(uint64_t u) {
  double x;
  __builtin_memcpy(&x, &u, 8);
  return x;
}

constexpr float kL2dReject = -32768.f;  // the quantum of code 0

// What the recurrence needs of eb code c: 2E = 2^(shift (c - 1) - 51), or -2
// for zero precision (no error is <= -1).
__host__ __device__ inline float l2d_prep(uint32_t c, int shift) {
  // shift c is c << (shift - 1) for both shifts
  const float e2 = l2d_float((c << (22 + shift)) + ((uint32_t)(76 - shift) << 23));
  return c ? e2 : -2.0f;
}

// Quantizes x against its prediction: returns the reconstruction, the
// quantum q (kL2dReject: unpredictable) in qs. e2 from l2d_prep.
__host__ __device__ inline float l2d_quantize(float pred, float x, float e2, float& qs) {
  const float diff = x - pred;
  const float half_inv = l2d_float(0x7F000000u - l2d_bits(e2));  // 1 / 2E
  const float qf = floorf(fmaf(fabsf(diff), half_inv, 0x1.fffffep-2f));
  const float s = copysignf(qf, diff);
  const float rec = fmaf(s, e2, pred);
  // one comparison on the chain: the error limit is -1 where q is out of range
  const float lim = qf < 32768.f ? 0.5f * e2 : -1.0f;
  const bool ok = fabsf(rec - x) <= lim;
  qs = ok ? s : kL2dReject;
  return ok ? rec : x;
}

// The stream's code of a quantum, q + 32768 (0 for kL2dReject): the low bits
// of the float 2^23 + q + 32768.
__host__ __device__ inline uint16_t l2d_code(float qs) { return (uint16_t)l2d_bits(qs + 8421376.0f); }

// Ids above 81 (2E beyond the float range): the reference's double arithmetic.
__host__ __device__ inline float l2d_quantize_wide(float pred, float x, uint32_t c, float& qs) {
  qs = kL2dReject;
  if (c == 0) return x;
  const double prec = ldexp(1.0, 2 * ((int)c - 1) - 52);
  const double diff = x - pred;
  double qd = fabs(diff) / prec + 1;
  if (qd < 65536) {
    qd = (diff > 0) ? qd : -qd;
    const int qi = (int)(qd / 2);
    const float dec = (float)((double)pred + 2 * qi * prec);
    if (fabs((double)(dec - x)) <= prec) {
      qs = (float)qi;
      return dec;
    }
  }
  return x;
}

// The double instantiation (quantize<double>, include/sz_compression_utils.hpp:50-65,
// prediction rounded to float): the same steps in double. prec = E, or -1 for
// zero precision.
__host__ __device__ inline double l2d_prep64(uint32_t c) {
  return c ? l2d_double((uint64_t)(2 * ((int)c - 1) - 52 + 1023) << 52) : -1.0;
}
__host__ __device__ inline double l2d_quantize(float pred, double x, double prec, float& qs) {
  const double diff = x - (double)pred;
  const double inv = l2d_double(0x7FE0000000000000ull - l2d_bits(prec));  // 1 / E
  // quant_diff = |diff|/E + 1: the quotient is exact, one rounding
  const double qf = floor(0.5 * fma(fabs(diff), inv, 1.0));
  const double s = copysign(qf, diff);
  const double rec = fma(s, 2 * prec, (double)pred);
  const bool ok = (qf < 32768.0) & (fabs(rec - x) <= prec);
  qs = ok ? (float)s : kL2dReject;
  return ok ? rec : x;
}

// Decompressor step (include/sz_decompression_utils.hpp:63-73): q == 0 takes
// the next unpredictable value; otherwise (float)(pred + 2(q - 32768) eb) with
// eb = 0 for stream id 0 and 2^(2 sid - 52) otherwise
// (src/sz_decompress_cp_preserve_2d.cpp:30-33). The element's own part is the
// step 2(q - 32768) eb (exact in float: sid <= 81).
__host__ __device__ inline float l2d_step(uint32_t q, uint32_t sid, int shift) {
  const float step = ldexpf((float)(2 * ((int)q - 32768)), (int)(sid << (shift - 1)) - 52);
  return sid ? step : 0.f;
}
__host__ __device__ inline double l2d_step64(uint32_t q, uint32_t sid) {
  const double step = ldexp((double)(2 * ((int)q - 32768)), 2 * (int)sid - 52);
  return sid ? step : 0.0;
}
__host__ __device__ inline float l2d_restore_wide(float pred, uint32_t q, uint32_t sid, float raw) {
  if (q == 0) return raw;
  const double prec = sid ? ldexp(1.0, 2 * (int)sid - 52) : 0.0;
  return (float)((double)pred + 2 * ((int)q - 32768) * prec);
}

}  // namespace cpsz
