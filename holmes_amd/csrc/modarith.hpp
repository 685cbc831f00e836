// Exact modular arithmetic for primes p < 2^50 on the gfx950 FP64 pipeline.
//
// Residues live in HBM as canonical uint64 in [0, p).  Inside kernels they are held as
// FP64 values that are exact integers ("signed-lazy" form): every value x satisfies
// |x| <= 8 p <= 2^53 and x is congruent to the residue.  FP64 FMA runs at full rate on gfx950
// (one wave64 instruction per SIMD every 4 cycles), while 64-bit integer multiplies are
// built from several 32-bit VALU multiplies; a lazy FP64 modular multiply measured 3.2x
// the throughput of a 32-bit-op Shoup multiply on MI355X, both bit-exact.
//
// Multiplication by a constant w in [0, p) with wp = fl(w / p):
//   q = rint(a * wp),  h = fl(a * w),  l = fma(a, w, -h)   (exact low part of a*w)
//   r = fma(-q, p, h) + l
// For |a| = A p < 2^53:  |fl(a*wp) - a*w/p| <= |a| 2^-52 <= A / 4, so |a*w - q*p| <= (0.5 + A / 4) p
// <= 2.5 p; |a*w| < 2^103 gives |l| <= 2^49, hence |h - q*p| <= 2.5p + 2^49 < 2^53 and the FMA is
// exact; the final sum is the exact integer a*w - q*p, so r == a*w (mod p), |r| <= (0.5 + A / 4) p.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hck {

constexpr int kLogN = 16;
constexpr int kN = 1 << kLogN;
constexpr double kTwo52 = 4503599627370496.0;  // 2^52

struct TwPair {
  double w;   // residue in [0, p) as an exact double
  double wp;  // fl(w / p)
};

__device__ __forceinline__ double u2d(uint64_t x) {
  // x < 2^52: place x in the mantissa of 2^52 and subtract 2^52 (exact).
  return __longlong_as_double((long long)(x | 0x4330000000000000ULL)) - kTwo52;
}

__device__ __forceinline__ uint64_t d2u(double x) {
  // x an integer in [0, 2^52): 2^52 + x has x as its mantissa field.
  return (uint64_t)__double_as_longlong(x + kTwo52) & 0x000FFFFFFFFFFFFFULL;
}

// a * w mod p, signed-lazy result: |r| <= (0.5 + A / 4) p for |a| = A p < 2^53.
__device__ __forceinline__ double mulc(double a, double w, double wp, double p) {
  const double q = __builtin_rint(a * wp);
  const double h = a * w;
  const double l = __builtin_fma(a, w, -h);
  return __builtin_fma(-q, p, h) + l;
}

__device__ __forceinline__ double mulc(double a, const TwPair& t, double p) {
  return mulc(a, t.w, t.wp, p);
}

// x mod p into [-p/2 - 2, p/2 + 2] for exact |x| <= 2^53 (pinv = fl(1/p)): the quotient's estimate is off by
// |x| / p 2^-52 at most.
__device__ __forceinline__ double reduce(double x, double p, double pinv) {
  const double q = __builtin_rint(x * pinv);
  return __builtin_fma(-q, p, x);
}

// x mod p into [0, p) for exact |x| <= 2^53, and for any integer |x| <= 2^61 that is a double: the
// centered remainder (exact, one FMA) lies within p/2 + 2^9, strictly between -p and p (p > 2^19: every prime
// is 1 modulo 2^17, and 6 2^17 + 1 is the first of them).
__device__ __forceinline__ double canon(double x, double p, double pinv) {
  const double r = reduce(x, p, pinv);
  return r < 0.0 ? r + p : r;
}

// a * b mod p for a residue b in [0, p) without a stored companion: the quotient is estimated
// from the product itself, q = rint(fl(a * b) * pinv).  fl(fl(a b) pinv) is within three
// roundings of X = a b / p, so |q - X| <= 0.5 + |X| 3 2^-53, and with |X| < |a| = A p,
//   |r| <= (0.5 + 0.375 A) p   (p < 2^50).
// For |a| < 2^53 (A < 8): |h - q p| <= 3.5 p + 2^49 < 2^53, so the FMA is
// exact and r == a b (mod p).  Twiddle tables store only w (8 bytes), and the product doubles as
// the quotient's input: 6 FP64 operations.
__device__ __forceinline__ double mulv(double a, double b, double p, double pinv) {
  const double h = a * b;
  const double q = __builtin_rint(h * pinv);
  const double l = __builtin_fma(a, b, -h);
  return __builtin_fma(-q, p, h) + l;
}

// The forward transform's stages that reduce their sum operand (stage l of 0 .. 15).  With A the largest
// |x| / p, a stage (u, v) -> (u + w v, u - w v) takes A to 0.5 + 1.375 A, or to 1 + 0.375 A when it
// reduces u.  From canonical words (A = 1) the column stages end at
// 1.88 3.08 4.73 [2.78] 4.32 6.44 [3.42] 5.20 and the row stages at
// 7.65 [3.87] 5.82 [3.19] 4.88 7.21 [3.71] 5.60; from centered words (A = 0.5) at 4.73 and 5.47.  Every
// value stays below 8 p <= 2^53, so all of them are exact.
constexpr bool fwd_reduces(int l) { return l == 3 || l == 6 || l == 9 || l == 11 || l == 14; }

// The same bounds for the compiler: each sum that the kernels leave unreduced has an assertion beside it.
// All are multiples of p; A stands for the largest |x| / p.
constexpr double kExact = 8.0;                // 8 p <= 2^53: every integer up to here is a double
constexpr double kCentered = 0.5 + 0x1p-10;   // p/2 + 2^9 (reduce of an encoder's coefficient; p > 2^19)
constexpr double mulv_bound(double A) { return 0.5 + 0.375 * A; }
constexpr double mulc_bound(double A) { return 0.5 + 0.25 * A; }
// forward stages first .. end - 1 from A: the end's bound, or the peak on the way
constexpr double fwd_bound(int first, int end, double A, bool peak = false) {
  double top = A;
  for (int l = first; l < end; ++l) {
    A = (fwd_reduces(l) ? kCentered : A) + mulv_bound(A);
    top = A > top ? A : top;
  }
  return peak ? top : A;
}
static_assert(fwd_bound(0, 16, 1.0, true) < kExact, "forward transform of canonical words");
static_assert(fwd_bound(0, 16, kCentered, true) < kExact, "forward transform of centered words");
// A transform's output from centered words (what the conversions and the encoder transform).
constexpr double kFwdOut = fwd_bound(0, 16, kCentered);

// Round half away from zero (llround semantics), written out: the library round() of this
// toolchain does not send negative ties away from zero.  trunc, one exact subtraction, one comparison
// and a signed step: no product to contract, so the result is the same in every translation unit.
__device__ __forceinline__ double round_away(double x) {
  const double r = __builtin_trunc(x);
  const double d = x - r;  // exact
  return r + __builtin_copysign(__builtin_fabs(d) >= 0.5 ? 1.0 : 0.0, x);
}

}  // namespace hck
