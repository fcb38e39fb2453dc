// FFT pieces shared by the ring stages (FP32 and FP64, gfx950): in-place
// radix-2^K passes over arrays in LDS, Bluestein convolutions, twiddles.
#pragma once

#include "common.h"
#include "device.h"

namespace ga {
namespace {

template <typename T>
struct tab_t;
template <>
struct tab_t<float> {
  using type = float2;
};
template <>
struct tab_t<double> {
  using type = double2;
};

template <typename T>
__device__ __forceinline__ cplx<T> ld(const typename tab_t<T>::type *p, int64_t i) {
  auto v = p[i];
  return {v.x, v.y};
}

__device__ __forceinline__ int ilog2(int x) { return 31 - __clz(x); }

// LDS work arrays insert one pad element after every 32 complex floats or 16
// complex doubles (256 bytes: all 64 banks), which removes the bank conflicts
// of the short-span butterflies and of the bit-reversed scatter.
template <typename T>
constexpr int kPadShift = sizeof(T) == 8 ? 4 : 5;
template <typename T = float>
__device__ __forceinline__ int pad(int i) {
  return i + (i >> kPadShift<T>);
}
template <typename T = float>
__host__ __device__ inline int padded_len(int n) {
  return n + (n >> kPadShift<T>) + 1;
}

__device__ __forceinline__ cplx<float> expi_q(int q, int d, float) {
  float s, c;
  sincospif(2.0f * float(q) / float(d), &s, &c);
  return {c, s};
}
__device__ __forceinline__ cplx<double> expi_q(int q, int d, double) {
  double s, c;
  sincospi(2.0 * double(q) / double(d), &s, &c);
  return {c, s};
}

__device__ __forceinline__ int blu_len(int r) {
  int L = 1;
  while (L < 2 * r - 1) L <<= 1;
  return L;
}

// e^{2 pi i k / 16} for k = 0..15: cos and sin
template <typename T>
__device__ __forceinline__ T c16(int k) {
  switch (k & 15) {
    case 0: return T(1);
    case 1: case 15: return T(0.92387953251128674);
    case 2: case 14: return T(0.70710678118654752);
    case 3: case 13: return T(0.38268343236508977);
    case 4: case 12: return T(0.0);
    case 5: case 11: return T(-0.38268343236508977);
    case 6: case 10: return T(-0.70710678118654752);
    case 7: case 9: return T(-0.92387953251128674);
    default: return T(-1);
  }
}
template <typename T>
__device__ __forceinline__ T s16(int k) {
  return c16<T>(k - 4);
}

// v e^{SIGN 2 pi i k / 16} (k a compile-time constant after unrolling)
template <int SIGN, typename T>
__device__ __forceinline__ cplx<T> rot16(cplx<T> v, int k) {
  k &= 15;
  if (k == 0) return v;
  if (k == 4) return SIGN > 0 ? cplx<T>{-v.im, v.re} : cplx<T>{v.im, -v.re};
  if (k == 8) return cplx<T>{-v.re, -v.im};
  if (k == 12) return SIGN > 0 ? cplx<T>{v.im, -v.re} : cplx<T>{-v.im, v.re};
  const T c = c16<T>(k), sn = SIGN * s16<T>(k);
  return cplx<T>{v.re * c - v.im * sn, v.re * sn + v.im * c};
}

template <typename T = float>
__device__ __forceinline__ cplx<T> twid(const typename tab_t<T>::type *__restrict__ tw, int idx,
                                        int sign) {
  const auto w = tw[idx];
  return cplx<T>{w.x, sign * w.y};
}

// One pass fusing K radix-2 stages with half-spans h0, 2 h0, .., 2^(K-1) h0
// (DIT: stages in increasing span; DIF: decreasing) on A arrays of length N.
// Group = elements base + q h0 (q < 2^K), base = blk 2^K h0 + b, b < h0.
// base has zeros in the bits that q h0 can set, so the sum never carries and
// its padded slots are
//   pad(base + q h0) = pad(base) + q h0 + (q h0 >> kPadShift),
// offsets that are the same for every thread of the pass.  tw holds
// e^{2 pi i j / 2^ltw}.
template <int K, int NT, bool DIT, int SIGN, typename T>
__device__ __forceinline__ void fused_pass(cplx<T> *X, int ldx, int A, int N, int h0,
                                           const typename tab_t<T>::type *__restrict__ tw, int ltw) {
  constexpr int R = 1 << K;
  const int lh0 = ilog2(h0);
  const int lg = ilog2(N) - K;  // groups per array = N / R
  const int total = A << lg;
  int off[R];
#pragma unroll
  for (int q = 0; q < R; ++q) off[q] = (q << lh0) + ((q << lh0) >> kPadShift<T>);
  for (int gg = threadIdx.x; gg < total; gg += NT) {
    const int a = gg >> lg, g = gg & ((1 << lg) - 1);
    const int b = g & (h0 - 1), blk = g >> lh0;
    const int base = (blk << (K + lh0)) + b;
    cplx<T> *Y = X + a * ldx + pad<T>(base);
    cplx<T> v[R];
#pragma unroll
    for (int q = 0; q < R; ++q) v[q] = Y[off[q]];
    // ws[s] = e^{SIGN 2 pi i b / (2^(s+1) h0)}: one table value per stage
    cplx<T> ws[K];
#pragma unroll
    for (int s = 0; s < K; ++s) ws[s] = twid<T>(tw, b << (ltw - s - 1 - lh0), SIGN);
#pragma unroll
    for (int ss = 0; ss < K; ++ss) {
      const int s = DIT ? ss : K - 1 - ss;
      const int d = 1 << s;
#pragma unroll
      for (int q = 0; q < R; ++q) {
        if (q & d) continue;
        // twiddle of this pair: ws[s] e^{SIGN 2 pi i (q mod d) / (2 d)}
        const cplx<T> t = rot16<SIGN>(ws[s], (q & (d - 1)) * (16 >> (s + 1)));
        if (DIT) {
          const cplx<T> y = cmul(v[q + d], t);
          const cplx<T> x = v[q];
          v[q] = cadd(x, y);
          v[q + d] = csub(x, y);
        } else {
          const cplx<T> x = v[q], y = v[q + d];
          v[q] = cadd(x, y);
          v[q + d] = cmul(csub(x, y), t);
        }
      }
    }
#pragma unroll
    for (int q = 0; q < R; ++q) Y[off[q]] = v[q];
  }
  __syncthreads();
}

// full power-of-two transform of A arrays: DIT (bit-reversed in, natural out)
// or DIF (natural in, bit-reversed out)
template <int NT, bool DIT, int SIGN, typename T>
__device__ __forceinline__ void fused_fft(cplx<T> *X, int ldx, int A, int N,
                                          const typename tab_t<T>::type *__restrict__ tw, int twlen) {
  const int lN = ilog2(N), ltw = ilog2(twlen);
  if (DIT) {
    for (int l = 0; l < lN;) {
      const int K = lN - l >= 4 ? 4 : lN - l;
      switch (K) {
        case 4: fused_pass<4, NT, true, SIGN>(X, ldx, A, N, 1 << l, tw, ltw); break;
        case 3: fused_pass<3, NT, true, SIGN>(X, ldx, A, N, 1 << l, tw, ltw); break;
        case 2: fused_pass<2, NT, true, SIGN>(X, ldx, A, N, 1 << l, tw, ltw); break;
        default: fused_pass<1, NT, true, SIGN>(X, ldx, A, N, 1 << l, tw, ltw); break;
      }
      l += K;
    }
  } else {
    for (int l = lN; l > 0;) {  // stages with half-spans 2^(l-1) down to 1
      const int K = l >= 4 ? 4 : l;
      const int h0 = 1 << (l - K);
      switch (K) {
        case 4: fused_pass<4, NT, false, SIGN>(X, ldx, A, N, h0, tw, ltw); break;
        case 3: fused_pass<3, NT, false, SIGN>(X, ldx, A, N, h0, tw, ltw); break;
        case 2: fused_pass<2, NT, false, SIGN>(X, ldx, A, N, h0, tw, ltw); break;
        default: fused_pass<1, NT, false, SIGN>(X, ldx, A, N, h0, tw, ltw); break;
      }
      l -= K;
    }
  }
}

// The middle of a Bluestein convolution as one pass: the last forward DIF
// pass (K stages, half-spans 2^(K-1) .. 1), the product with the chirp
// spectrum (stored bit-reversed, i.e. in the order the DIF leaves the
// values) and the first inverse DIT pass (half-spans 1 .. 2^(K-1)) act on the
// same groups of 2^K consecutive elements, whose twiddles are the constant
// rotations alone; one LDS round trip instead of three.
template <int K, int NT, typename T>
__device__ __forceinline__ void mid_pass(cplx<T> *X, int ldx, int A, int L,
                                         const typename tab_t<T>::type *__restrict__ bspec) {
  constexpr int R = 1 << K;
  const int lg = ilog2(L) - K;
  const int total = A << lg;
  for (int gg = threadIdx.x; gg < total; gg += NT) {
    const int a = gg >> lg, g = gg & ((1 << lg) - 1);
    const int base = g << K;
    cplx<T> *Y = X + a * ldx + pad<T>(base);  // a group never straddles a pad
    cplx<T> v[R];
#pragma unroll
    for (int q = 0; q < R; ++q) v[q] = Y[q];
#pragma unroll
    for (int s = K - 1; s >= 0; --s) {
      const int d = 1 << s;
#pragma unroll
      for (int q = 0; q < R; ++q) {
        if (q & d) continue;
        const cplx<T> tq = rot16<-1>(cplx<T>{T(1), T(0)}, (q & (d - 1)) * (16 >> (s + 1)));
        const cplx<T> x = v[q], y = v[q + d];
        v[q] = cadd(x, y);
        v[q + d] = cmul(csub(x, y), tq);
      }
    }
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const auto b = bspec[base + q];
      v[q] = cmul(v[q], cplx<T>{b.x, b.y});
    }
#pragma unroll
    for (int s = 0; s < K; ++s) {
      const int d = 1 << s;
#pragma unroll
      for (int q = 0; q < R; ++q) {
        if (q & d) continue;
        const cplx<T> tq = rot16<1>(cplx<T>{T(1), T(0)}, (q & (d - 1)) * (16 >> (s + 1)));
        const cplx<T> y = cmul(v[q + d], tq);
        const cplx<T> x = v[q];
        v[q] = cadd(x, y);
        v[q + d] = csub(x, y);
      }
    }
#pragma unroll
    for (int q = 0; q < R; ++q) Y[q] = v[q];
  }
  __syncthreads();
}

// Bluestein convolution of A arrays of length L = 2^lN in place: forward DIF
// passes (K = 4, half-spans down to 2^(l0)), the middle pass (K = l0 <= 4,
// with the chirp spectrum), inverse DIT passes mirroring the forward ones;
// natural order in and out.
template <int NT, typename T>
__device__ __forceinline__ void bluestein_conv(cplx<T> *X, int ldx, int A, int L,
                                               const typename tab_t<T>::type *__restrict__ tw, int twlen,
                                               const typename tab_t<T>::type *__restrict__ bspec) {
  const int lN = ilog2(L), ltw = ilog2(twlen);
  int l = lN;
  for (; l > 4; l -= 4) fused_pass<4, NT, false, -1>(X, ldx, A, L, 1 << (l - 4), tw, ltw);
  switch (l) {
    case 4: mid_pass<4, NT>(X, ldx, A, L, bspec); break;
    case 3: mid_pass<3, NT>(X, ldx, A, L, bspec); break;
    case 2: mid_pass<2, NT>(X, ldx, A, L, bspec); break;
    default: mid_pass<1, NT>(X, ldx, A, L, bspec); break;
  }
  for (int lo = l; lo < lN; lo += 4) fused_pass<4, NT, true, 1>(X, ldx, A, L, 1 << lo, tw, ltw);
}

}  // namespace
}  // namespace ga
