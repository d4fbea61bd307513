// Exact arithmetic mod q = 12289 on FP32 values, for the NewHope transforms.
//
// Values are integers in floats, twiddles plain (no Montgomery factor) and centred
// (|z| <= 6144).  x z is formed exactly inside v_fma_f32 and reduced by k = round(x z / q)
// in two exact steps, q = 3 2^12 + 1: x z - 12288 k = r + k, then minus k.  With |x z| / q
// <= 2^21, 12288 k = 3 k 2^12 and r + k (below 2^24) are exact, and z / q's rounding moves
// k by at most 2^21 2^-23 = 1/4: |r| < 0.76 q.  Five full-rate instructions; the integer
// Montgomery product is three 32-bit multiplies at half that rate and five more.
//
// Bounds (checked on the CPU by tests/c/newhope_f32_test.cpp):
//   mul(x, z)   |x z| <= kMulMax q     -> |result| <= kOut
//   reduce(x)   |x| <= kReduceMax      -> |result| <= kCentred
//   canon(x)    |x| <= kCanonMax       -> x mod q in [0, q), as an integer
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define PQC_NH_F32_HD __host__ __device__
#else
#define PQC_NH_F32_HD
#endif

namespace pqc {
namespace newhope {
namespace fp {
constexpr float kQ = 12289.0f, kQinv = 1.0f / 12289.0f, kM = 12582912.0f;  // kM = 1.5 2^23
constexpr int kMulMax = 1 << 21, kOut = 9340, kCentred = 6145, kReduceMax = 1 << 24, kCanonMax = 1 << 19;
constexpr int kTwiddle = 6144;  // a centred twiddle

// zq = z kQinv
PQC_NH_F32_HD inline float mul(float x, float z, float zq) {
  const float k = __builtin_fmaf(x, zq, kM) - kM;
  return __builtin_fmaf(x, z, k * -12288.0f) - k;
}
PQC_NH_F32_HD inline float mul(float x, float z) { return mul(x, z, z * kQinv); }
// centred residue
PQC_NH_F32_HD inline float reduce(float x) {
  const float k = __builtin_fmaf(x, kQinv, kM) - kM;
  return __builtin_fmaf(k, -kQ, x);
}
// the residue in [0, q) as an integer: k = floor(x / q) as the rounding of
// x / q - 1/2 + 1 / (2 q), whose margin 1 / (2 q) exceeds the float error 2^-18
PQC_NH_F32_HD inline uint32_t canon(float x) {
  const float k = (__builtin_fmaf(x, kQinv, -0.5f + 0.5f / kQ) + kM) - kM;
  return __builtin_bit_cast(uint32_t, __builtin_fmaf(k, -kQ, x + kM)) & 0x3FFFu;
}

// ---- bounds of the transforms -------------------------------------------------------
// Forward: inputs are noise or packed coefficients below 2^14 (kIn); each of log2 N layers
// adds one product.  Inverse: the same inputs; its first log2(N / 64) layers double where
// z = 1, the others add a product.
constexpr int kIn = 1 << 14;
constexpr int log2n(int n) { return n == 1024 ? 10 : 9; }
constexpr int fwd_bound(int n) { return kIn + log2n(n) * kOut; }
constexpr int inv_bound(int n) { return (kIn << (log2n(n) - 6)) + 6 * kOut; }
constexpr bool mul_ok(int x, int z) { return (int64_t)x * z <= (int64_t)kMulMax * 12289; }
static_assert(mul_ok(fwd_bound(1024), kTwiddle) && mul_ok(inv_bound(1024), kTwiddle), "every layer's products");
static_assert(mul_ok(65535, kCentred) && mul_ok(kIn, kIn), "gen_a times a centred value; packed values");
static_assert(fwd_bound(1024) <= kReduceMax && fwd_bound(1024) + kOut <= kCanonMax, "what follows the forward one");
static_assert(kOut + 3 * 12289 <= kCanonMax, "and the inverse one: noise and message added, or v subtracted");
}  // namespace fp
}  // namespace newhope
}  // namespace pqc
