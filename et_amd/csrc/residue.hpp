// FP64 products by exact integer arithmetic on the int8 matrix cores: the
// number theory shared by the kernels (gemm_residue.hip) and the host checks.
//
// A row a of op(A) and a column b of op(B) are scaled by powers of two and
// rounded to integers, a' = rint(2^ea a), b' = rint(2^eb b), with ||a'||_2 and
// ||b'||_2 at most 2^kNormBits.  By Cauchy-Schwarz |a'.b'| < M / 2 for
// M = m_0 m_1 ... m_15, the product of 16 pairwise coprime moduli of at most 8
// bits, so the integer a'.b' is determined by its residues, and each residue
// is an int8 product with int32 accumulation, without any rounding
// (Chinese remainder theorem; the scheme is Ozaki, Uchino and Imamura's
// "Ozaki scheme II", 2025).  The only errors are the rounding of the operands
// to integers, at most 2^-kNormBits ||a|| per element, and one final rounding to
// double.
//
// So the error is fixed in the norm, 0.41 2^-kNormBits ||a|| ||b|| rms for norms of
// 2^kNormBits (two to four times that for smaller ones), while an FP64 sum of terms of
// random sign has about 0.4 2^-53 of sum |a_k b_k|.  Rows and columns whose large elements
// meet are far more exact than in FP64 (normal ones 15 times); where large elements meet
// small ones the FP64 sum would be, and such outputs go to it: see the guard below.
#pragma once

#include <cmath>
#include <cstdint>

#ifndef ETG_HD
#if defined(__HIPCC__)
#define ETG_HD __host__ __device__
#else
#define ETG_HD
#endif
#endif

namespace etg {
namespace residue {

constexpr int kModuli = 16;
constexpr int kMod[kModuli] = {256, 255, 253, 251, 247, 241, 239, 233, 229, 227, 223, 217, 211, 199, 197, 193};
constexpr int kNormBits = 62;                     // 2 kNormBits < log2(M / 2) = 124.37
// |residue| <= 128 on both sides: the int32 sums hold this many terms
constexpr int64_t kMaxDepth = (int64_t(1) << 17) - 1;
constexpr int kNotFinite = INT32_MIN;             // exponent of a row with an infinity or NaN

constexpr unsigned __int128 product_of_moduli() {
  unsigned __int128 p = 1;
  for (int i = 0; i < kModuli; ++i) p *= unsigned(kMod[i]);
  return p;
}
constexpr unsigned __int128 kM = product_of_moduli();
constexpr double kMDouble = double(kM);

// 2^e mod m
constexpr int pow2_mod(int e, int m) {
  int r = 1 % m;
  for (int i = 0; i < e; ++i) r = r * 2 % m;
  return r;
}

// inverse of M / m_i modulo m_i
constexpr int cofactor_inverse(int i) {
  const int m = kMod[i], c = int((kM / unsigned(m)) % unsigned(m));
  for (int x = 1; x < m; ++x)
    if (c * x % m == 1) return x;
  return 0;
}

// X = sum_i r_i inv_i (M / m_i)  (mod M), so X / M = sum_i r_i f_i (mod 1) with
// f_i = inv_i / m_i.  f_i = (kHi + kLo 2^-40) 2^-40 to 2^-81: sums of 16 terms
// |r_i| <= 128 of either part are exact in FP64, and the 2^-70 M at most that is left
// out (2^-74 rms) is below 2^-5 of the operands' rounding.
constexpr uint64_t fraction80(int i, bool high) {
  const unsigned __int128 num = (unsigned __int128)(unsigned(cofactor_inverse(i))) << 81;
  const unsigned __int128 f = (num / unsigned(kMod[i]) + 1) >> 1;   // rounded to 2^-80
  return high ? uint64_t(f >> 40) : uint64_t(f & ((uint64_t(1) << 40) - 1));
}

constexpr uint32_t kBits23 = 0x4b000000u;         // the float 2^23

struct Constants {
  // residues of an integer given as 8 unsigned bytes of (a' + 2^63): weights of
  // the low and high four bytes, 256^j mod m, and -2^63 - 2^23 mod m with the bits
  // of the float 2^23 on top
  uint32_t low[kModuli], high[kModuli], offset[kModuli];
  uint32_t c[kModuli];                            // 256 - m
  float invf[kModuli];
  double md[kModuli], invd[kModuli];
  double fhi[kModuli], flo[kModuli];
};

constexpr Constants make_constants() {
  Constants c{};
  for (int i = 0; i < kModuli; ++i) {
    const int m = kMod[i];
    uint32_t w[2] = {0, 0};
    for (int j = 0; j < 8; ++j) w[j / 4] |= uint32_t(pow2_mod(8 * j, m) & 0xff) << (8 * (j % 4));
    c.low[i] = w[0];
    c.high[i] = w[1];
    c.offset[i] = kBits23 + uint32_t((2 * m - pow2_mod(63, m) - pow2_mod(23, m)) % m);
    c.c[i] = uint32_t(256 - m);
    c.invf[i] = 1.0f / float(m);
    c.md[i] = double(m);
    c.invd[i] = 1.0 / double(m);
    c.fhi[i] = double(fraction80(i, true));
    c.flo[i] = double(fraction80(i, false));
  }
  return c;
}
constexpr Constants kC = make_constants();

// Scale exponent of a row from its sum of squares, the bits of its largest
// magnitude and its length: ||2^e a|| <= 2^kNormBits.  Where the squares leave
// the range in which their sum is accurate, the norm is bounded by
// sqrt(k) max |a|.
ETG_HD inline int scale_exponent(double sumsq, uint64_t max_bits, int64_t k) {
  if (max_bits == 0) return 0;
  if (max_bits >= 0x7ff0000000000000ull) return kNotFinite;
  int x;
  if (sumsq > 1e-270 && sumsq < 1e290) {
    (void)frexp(sumsq, &x);                       // sumsq < 2^x
    return kNormBits - ((x + 1) >> 1);
  }
  double big;
  static_assert(sizeof(big) == sizeof(max_bits), "double bits");
  __builtin_memcpy(&big, &max_bits, sizeof(big));
  (void)frexp(big, &x);                           // big < 2^x
  int lk = 0;
  while ((int64_t(1) << lk) < k) ++lk;
  return kNormBits - x - ((lk + 1) >> 1);
}

// a' = rint(2^e x) + 2^63 as two 32-bit halves (|a'| < 2^60)
ETG_HD inline void to_integer(double x, int e, uint32_t& lo, uint32_t& hi) {
  const double v = rint(ldexp(x, e));
  const double h = floor(v * 0x1p-32);
  lo = uint32_t(fma(h, -0x1p32, v));
  hi = uint32_t(int32_t(h)) ^ 0x80000000u;
}

ETG_HD inline uint32_t byte_dot(uint32_t a, uint32_t b, uint32_t c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_udot4(a, b, c, false);
#else
  for (int j = 0; j < 4; ++j) c += ((a >> (8 * j)) & 0xffu) * ((b >> (8 * j)) & 0xffu);
  return c;
#endif
}

// Low byte of a number x = 2^23 + v congruent to the integer, in [-128, 127] and
// congruent too, from the bits of the float x (v < 2^23).  x / m is rounded by adding
// 1.5 2^23, which leaves the quotient in the low bits, and x - q m is x + (256 - m) q
// in the low byte.  The FP32 quotient may be one off where x / m is near a half; that
// the result is in range then was checked for every x and every m.
ETG_HD inline uint32_t low_byte(uint32_t x, float inv, uint32_t c) {
  float f;
  __builtin_memcpy(&f, &x, sizeof(f));
  f = fmaf(f, inv, 12582912.0f);
  uint32_t q;
  __builtin_memcpy(&q, &f, sizeof(q));
  return (q & 0xffffffu) * c + x;
}

// Symmetric residue of the integer modulo m_i: its two's complement in the low
// byte of the returned word.  Four operations (two byte dot products, a fused
// multiply-add and an integer one); with the byte sum converted to float and the
// remainder formed there it took seven.
ETG_HD inline uint32_t residue_byte(uint32_t lo, uint32_t hi, int i) {
  if (kMod[i] == 256) return lo;                  // 2^63 is a multiple
  return low_byte(byte_dot(hi, kC.high[i], byte_dot(lo, kC.low[i], kC.offset[i])), kC.invf[i], kC.c[i]);
}

// The same of an int32 sum (FP64 arithmetic, exact; the matrix cores are busy beside it,
// and the four-operation form gained nothing there).
ETG_HD inline uint32_t residue_byte_of_sum(int32_t s, double m, double inv) {
  constexpr double kMagic = 6755399441055744.0;   // 1.5 2^52
  const double t = double(s);
  const double q = fma(t, inv, kMagic) - kMagic;
  const double r = fma(-q, m, t) + kMagic;
  uint64_t bits;
  __builtin_memcpy(&bits, &r, sizeof(bits));
  return uint32_t(bits);
}

// The guard.  The rounding of the operands has an rms error of 0.41 2^kNormBits in a'.b'
// (1/2 / sqrt(3) per element, norms up to 2^kNormBits) whatever the sum, while an FP64
// sum's error goes with sum |a_k b_k|.  Where large elements of the row meet small ones of
// the column that sum is far below ||a|| ||b||, and digits that FP64 would keep are lost.
// So a product also forms Q = sum qa qb of the magnitudes q = |a'| 2^-47, rounded to 8-bit
// floats (5 exponent and 2 fraction bits, 2^30 below the row's norm; at most a ninth up):
// Q is at most 1.24 times sum |a'_k b'_k| 2^-94.  With the rows' norms na and nb in units
// of 2^kNormBits, an output with Q below kThreshold max(na, nb) is formed in FP64; elsewhere
// sum |a'_k b'_k| is at least max(na, nb) 2^(kNormBits + kGuardBits), and the rms error at
// most 0.41 2^-kGuardBits of sum |a_k b_k|, about what an FP64 sum of terms of random sign has.
// With 15 moduli (58 bits) that limit is reached in most 128 x 128 blocks of a molecule's
// products.
constexpr int kGuardBits = 52;                    // 0.82 2^-53
constexpr float kThreshold = 1.24f * float(uint64_t(1) << (kNormBits + kGuardBits - 94));
static_assert(kNormBits <= 62, "the largest magnitude is an 8-bit float");
constexpr float kZeroNorm = -1.0f;                // of a row of zeros: nothing to lose

// Norm of the scaled row in units of 2^kNormBits (1 where it is only bounded; infinite for
// a row that is not finite).
ETG_HD inline float scaled_norm(double sumsq, uint64_t max_bits) {
  if (max_bits == 0) return kZeroNorm;
  if (max_bits >= 0x7ff0000000000000ull) return float(HUGE_VAL);
  if (!(sumsq > 1e-270 && sumsq < 1e290)) return 1.0f;
  int x;
  const double f = frexp(sumsq, &x);
  return float(sqrt((x & 1) ? 0.5 * f : f)) * (1.0f + 0x1p-20f);
}

// From the high half of the integer, floor(a' / 2^32) + 2^31: the top of the FP32 number
// |a'| 2^-32, its exponent from 2^0 on.
ETG_HD inline uint32_t magnitude_byte(uint32_t hi) {
  const int32_t h = int32_t(hi ^ 0x80000000u);
  const float f = float(uint32_t(h ^ (h >> 31)));
  uint32_t bits;
  __builtin_memcpy(&bits, &f, sizeof(bits));
  const int32_t q = int32_t((bits + 0x100000u) >> 21) - (127 << 2);
  return uint32_t(q > 0 ? q : 0);
}

// a'.b' 2^-(ea + eb) from the sums hi = sum_i r_i kHi_i and lo = sum_i r_i kLo_i.
ETG_HD inline double reconstruct(double hi, double lo, int ea, int eb) {
  const double t = hi * 0x1p-40;
  const double frac = (t - rint(t)) + lo * 0x1p-80;   // X / M in [-1/2, 1/2], the first term exact
  return ldexp(frac * kMDouble, -ea - eb);
}

}  // namespace residue
}  // namespace etg
