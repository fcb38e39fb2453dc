// Device-side helpers shared by the kernels (gfx950, wave64).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ga {

// complex value in registers
template <typename T>
struct cplx {
  T re, im;
};

template <typename T>
__device__ __forceinline__ cplx<T> cmul(cplx<T> a, cplx<T> b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
template <typename T>
__device__ __forceinline__ cplx<T> cadd(cplx<T> a, cplx<T> b) {
  return {a.re + b.re, a.im + b.im};
}
template <typename T>
__device__ __forceinline__ cplx<T> csub(cplx<T> a, cplx<T> b) {
  return {a.re - b.re, a.im - b.im};
}
template <typename T>
__device__ __forceinline__ cplx<T> cconj(cplx<T> a) {
  return {a.re, -a.im};
}
template <typename T>
__device__ __forceinline__ cplx<T> cmuli(cplx<T> a) {  // a * i
  return {-a.im, a.re};
}

// exp(2 pi i q / d) for 0 <= q < d, accurate to the type's rounding
__device__ __forceinline__ cplx<double> expi_frac(int64_t q, int64_t d, double) {
  double s, c;
  sincospi(2.0 * double(q) / double(d), &s, &c);
  return {c, s};
}
__device__ __forceinline__ cplx<float> expi_frac(int64_t q, int64_t d, float) {
  // reduce in double so the float argument stays exact to rounding
  double s, c;
  sincospi(2.0 * double(q) / double(d), &s, &c);
  return {float(c), float(s)};
}

// Legendre seed lambda_mm = c_m sin^m(theta) in the scaled form used by the
// recurrence kernels: value = p * 2^(600 k), k <= 0, p in (2^-601 |c_m|, |c_m|].
// sin^m is formed by binary powering with exact exponent bookkeeping.
constexpr int kScaleBits = 600;

// sin^m(theta) = rm 2^E (E <= 0), with exact exponent bookkeeping
__device__ __forceinline__ void sin_power(double sth, int m, double &rm, long long &E) {
  int es;
  double b = frexp(sth, &es);  // sth = b 2^es, b in [0.5, 1)
  double bm = b;
  rm = 1.0;
  int er = 0, eb = 0;
  int mm = m;
  while (mm) {
    if (mm & 1) {
      int t;
      rm = frexp(rm * bm, &t);
      er += eb + t;
    }
    mm >>= 1;
    if (mm) {
      int t;
      bm = frexp(bm * bm, &t);
      eb = 2 * eb + t;
    }
  }
  E = (long long)er + (long long)m * (long long)es;  // <= 0
}

__device__ __forceinline__ void legendre_seed(double cm, double sth, int m, double &p,
                                              int &k) {
  double rm;
  long long E;
  sin_power(sth, m, rm, E);
  const long long negE = -E;
  k = -int(negE / kScaleBits);
  const int rem = int(E + (long long)kScaleBits * (negE / kScaleBits));  // in (-600, 0]
  p = ldexp(cm * rm, rem);
}

// Seeds of the spin-s recurrences at l0 = max(m, s) for one ring:
// +s: K sin^{m+s}(t/2) cos^{|m-s|}(t/2), -s: K' sin^{|m-s|}(t/2) cos^{m+s}(t/2),
// with K = mant 2^exp (signed mantissa) from the plan's seed table.  The powers
// are formed as mantissa and exact binary exponent: b^n = mant 2^e.
__device__ __forceinline__ void scaled_power(double b, int n, double &mant, long long &e) {
  int eb;
  const double bm0 = frexp(b, &eb);
  double rm = 1.0, bm = bm0;
  long long er = 0, ebb = 0;
  int nn = n;
  while (nn) {
    if (nn & 1) {
      int t;
      rm = frexp(rm * bm, &t);
      er += ebb + t;
    }
    nn >>= 1;
    if (nn) {
      int t;
      bm = frexp(bm * bm, &t);
      ebb = 2 * ebb + t;
    }
  }
  mant = rm;
  e = er + (long long)n * eb;
}

// value = mant 2^E (E <= 0 in use) in the scaled form p 2^(600 k), k <= 0
__device__ __forceinline__ void to_scaled(double mant, long long E, double &p, int &k) {
  if (E > 0) {  // cannot exceed O(1) values, but keep the representation valid
    p = ldexp(mant, int(E));
    k = 0;
    return;
  }
  const long long negE = -E;
  k = -int(negE / kScaleBits);
  const int rem = int(E + (long long)kScaleBits * (negE / kScaleBits));
  p = ldexp(mant, rem);
}

// The scaled form of the FP64 stages: value = p 2^(600 k), k <= 0, where a
// scaled value (k < 0) is held below 2^-300.  Such a p stands for a number
// below 2^-900 of its own magnitude, so a kernel may use it as if it were the
// value: the error it makes is below 2^-200 of the operand it multiplies (a
// chunk of 16 recurrence steps grows a value by less than 2^100), and no
// step needs a test.  rescale_low is called once per chunk and moves a value
// that has passed 2^-300 up one scale.
constexpr int kLowBits = 300;

__device__ __forceinline__ void to_scaled_low(double mant, long long E, double &p, int &k) {
  const long long negE = -E;
  k = negE < kLowBits + kScaleBits ? 0 : -int((negE - kLowBits) / kScaleBits);
  p = ldexp(mant, int(E - (long long)kScaleBits * k));
}

// the seed lambda_mm in that form
__device__ __forceinline__ void legendre_seed_low(double cm, double sth, int m, double &p,
                                                  int &k) {
  double rm;
  long long E;
  sin_power(sth, m, rm, E);
  to_scaled_low(cm * rm, E, p, k);
}

__device__ __forceinline__ void rescale_low(double &p0, double &p1, int &k) {
  const bool up = k < 0 && fabs(p1) > 0x1p-300;
  const double f = up ? 0x1p-600 : 1.0;
  p1 *= f;
  p0 *= f;
  k += up;
}

// One row of the normalised recurrence of the FP64 stages, X = 2x, h = gam / 2 - 1
// (d_h64); the new value is in p1.  Two operations: the coefficient gam x, rounded
// once, and the step, from (p0, p1) = (y_{l-2}, y_{l-1}).  The row of l = m (h = -1)
// yields the seed from p1 = 0 and p0 = -seed.
//
// For m = 0, 1 the coefficients tend to 2x so fast that the rounding of gam x is the
// same for most rows, which adds up over a long recurrence.  There DIFF carries
// the difference p0 = y_{l-1} - y_{l-2} (at first the seed), with gam x - 2 as its
// coefficient, for one operation more (map2alm without iterations at nside 512,
// lmax 1023: 171 -> 178 us, the workgroup of m = 0 being the longest).  Below lmax
// 832 the whole error stays under that of the (a, b) form without it (nside 512,
// lmax 820: 0.9556e-14 against 0.9553e-14; lmax 880: 1.027e-14 against 1.017e-14).
//
// Error of lambda, RMS over all (l, m) and rings (weighted by their pixels), at
// nside 64, lmax 128; 256, 512; 512, 1023; 1024, 2048: as a (x lambda_{l-1} - b
// lambda_{l-2}) 2.06e-15, 6.2e-15, 1.17e-14, 2.28e-14; this form 1.91e-15, 6.0e-15,
// 1.15e-14, 2.25e-14 (without DIFF 1.21e-14 and 2.38e-14 in the last two); with
// gam and c from products in double precision 2.81e-15, 7.9e-15, 1.41e-14, 3.04e-14.
// Most of what is left is the seed's (sin^m by repeated squaring).
__device__ __forceinline__ bool norm_diff(int lmax, int m) { return m < 2 && lmax >= 832; }

template <bool DIFF>
__device__ __forceinline__ void norm_step(double h, double X, double &p0, double &p1) {
  if (DIFF) {
    p0 = fma(fma(1.0 + h, X, -2.0), p1, p0);
    p1 += p0;
  } else {
    const double y = fma(fma(h, X, X), p1, -p0);
    p0 = p1;
    p1 = y;
  }
}

// ---- sums over the lanes of a wave
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, int(uint32_t(u)), CTRL, 0xF, 0xF, false);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, int(uint32_t(u >> 32)), CTRL, 0xF, 0xF, false);
  return __builtin_bit_cast(double, (uint64_t(hi) << 32) | lo);
}
// lanes with `bit` unset get a summed over the lane and its partner, the
// others b; the partner (CTRL) has the other `bit`
template <int CTRL>
__device__ __forceinline__ double halve(double a, double b, bool bit) {
  const double keep = bit ? b : a, send = bit ? a : b;
  return keep + dpp_move<CTRL>(send);
}
template <bool ROWS16>
__device__ __forceinline__ double halve_swap(double a, double b) {
  const uint64_t ua = __builtin_bit_cast(uint64_t, a), ub = __builtin_bit_cast(uint64_t, b);
  // (X, Y) -> ([X_lo | Y_lo], [X_hi | Y_hi]) over halves of the wave, or over
  // even and odd rows of 16 lanes
  uint32_t l0, l1, h0, h1;
  if (ROWS16) {
    const auto l = __builtin_amdgcn_permlane16_swap(uint32_t(ua), uint32_t(ub), false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(uint32_t(ua >> 32), uint32_t(ub >> 32), false, false);
    l0 = l[0]; l1 = l[1]; h0 = h[0]; h1 = h[1];
  } else {
    const auto l = __builtin_amdgcn_permlane32_swap(uint32_t(ua), uint32_t(ub), false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(uint32_t(ua >> 32), uint32_t(ub >> 32), false, false);
    l0 = l[0]; l1 = l[1]; h0 = h[0]; h1 = h[1];
  }
  return __builtin_bit_cast(double, (uint64_t(h0) << 32) | l0) +
         __builtin_bit_cast(double, (uint64_t(h1) << 32) | l1);
}

// The 32 sums v[0..31] over the 64 lanes of a wave: lane L returns sum L / 2.
// Every exchange halves the number of sums a lane carries while it adds the
// partner's half, about 125 instructions in all.
__device__ __forceinline__ double wave_sums32(const double (&v)[32], int lane) {
  double a[16], b[8], c[4], d[2];
#pragma unroll
  for (int q = 0; q < 16; ++q) a[q] = halve_swap<false>(v[q], v[q + 16]);
#pragma unroll
  for (int q = 0; q < 8; ++q) b[q] = halve_swap<true>(a[q], a[q + 8]);
#pragma unroll
  for (int q = 0; q < 4; ++q) c[q] = halve<0x128>(b[q], b[q + 4], lane & 8);  // row_ror:8
#pragma unroll
  for (int q = 0; q < 2; ++q) d[q] = halve<0x141>(c[q], c[q + 2], lane & 4);  // row_half_mirror
  const double e = halve<0x1B>(d[0], d[1], lane & 2);                          // quad_perm [3,2,1,0]
  return e + dpp_move<0xB1>(e);                                                // quad_perm [1,0,3,2]
}

// ---- Philox4x32-10 (Salmon, Moraes, Dror, Shaw 2011), counter-based
struct u32x4 {
  uint32_t v[4];
};

__device__ __forceinline__ u32x4 philox4x32_10(u32x4 c, uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const uint64_t p0 = uint64_t(0xD2511F53u) * c.v[0];
    const uint64_t p1 = uint64_t(0xCD9E8D57u) * c.v[2];
    const uint32_t hi0 = uint32_t(p0 >> 32), lo0 = uint32_t(p0);
    const uint32_t hi1 = uint32_t(p1 >> 32), lo1 = uint32_t(p1);
    c = u32x4{{hi1 ^ c.v[1] ^ k0, lo1, hi0 ^ c.v[3] ^ k1, lo0}};
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  return c;
}

// a double in [0, 1) with 53 random bits from two words (27 + 26 bits)
__device__ __forceinline__ double uniform53(uint32_t a, uint32_t b) {
  return (double(a >> 5) * 67108864.0 + double(b >> 6)) * 0x1p-53;
}

// (m, ring group) of this block of a grid of m_run8_blocks (see common.h)
__device__ __forceinline__ bool decode_m_run8(int lmax, int nrg, int &m, int &rg) {
  const int b = blockIdx.x, xcd = b & 7, kq = b >> 3;
  const int mq = kq / nrg;
  rg = kq - mq * nrg;
  m = 64 * (mq >> 3) + 8 * xcd + (mq & 7);
  return m <= lmax;
}

// full 64-bit lane masks
__device__ __forceinline__ bool wave_any(bool v) { return __any(v); }
__device__ __forceinline__ bool wave_all(bool v) { return __all(v); }

}  // namespace ga
