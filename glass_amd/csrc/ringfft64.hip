// Per-ring Fourier stage of the FP64 transforms (one map, or one pair of maps).
//
// As in FP32, a ring of n = 4 r pixels is one complex transform of two real
// ones, split into four of length r (radix-2^K passes in LDS for a power of two,
// Bluestein convolutions otherwise).  The two real transforms are the two maps
// of a pair (spin) or, for one map, the north and the south ring of a ring
// pair, which have the same length and the same phi0: one complex transform
// serves both, where a ring by itself would leave the imaginary part empty.
//
// A of the four transforms run together on A arrays in LDS, as many as fit the
// launch's share (4 for short rings, 1 for the longest), so that short
// transforms still give every thread work in each pass.  The threads of a
// workgroup follow the longest ring: 64 for r <= 64 up to 512.
//
// The synthesis can subtract its result from a given map in the store (the
// residual of the analysis iterations), the analysis can weight the pixels in
// the load, each in place of a pass of its own.
//
// Bound: LDS round trips and barriers of the passes; HBM traffic (the ring
// coefficients once, the pixels once) is a third of the time at large nside.
// Measured at nside 1024, lmax 2048, one map: 140 us synthesis, 128 us analysis (one
// ring at a time, radix-4 stages of one array, a pass for the residual: 396
// and 350 us, and 48 for the residual).  The synthesis' fold keeps the loads of
// four bins in flight, past lmax too, instead of one loop after another with a
// wait in each: the whole alm2map 764 -> 751 us there, 50 -> 39 at nside 100,
// lmax 700, 24 -> 20 at nside 128, lmax 256.
#include <algorithm>

#include "common.h"
#include "device.h"
#include "kernels.h"
#include "ringfft.h"

namespace ga {

namespace {

using c64 = cplx<double>;

// the two real transforms of an item: coefficients at f[q] + m stride, pixels
// at map offset px[q]; has1: the second exists
struct ring_item {
  int ring, n;
  bool has1;
  int64_t f[2], px[2];
  int stride;
};

__device__ __forceinline__ ring_item decode_item(int S, int lmax, int nrings, int64_t npix,
                                                 const int64_t *__restrict__ ring_start,
                                                 const int32_t *__restrict__ ring_n) {
  ring_item it;
  const int b = blockIdx.x;
  it.ring = b;
  it.stride = S;
  const int64_t row = lmax + 1;
  if (S == 1) {  // ring pair b; the equator ring (the last one) is alone
    const int south = nrings - 1 - b;
    it.has1 = south != b;
    it.f[0] = b * row;
    it.f[1] = south * row;
    it.px[0] = ring_start[b];
    it.px[1] = ring_start[south];
  } else {  // ring b of the maps 0 and 1
    it.has1 = true;
    it.f[0] = b * row * 2;
    it.f[1] = it.f[0] + 1;
    it.px[0] = ring_start[b];
    it.px[1] = npix + ring_start[b];
  }
  it.n = ring_n[b];
  return it;
}

__device__ __forceinline__ int bit_rev(int k, int bits) {
  return bits ? int(__brev(unsigned(k)) >> (32 - bits)) : 0;
}

// The inverse length-r DFTs of H[.][0..3] (k1 = t + c NT) in place, A at a
// time; CONJ: the forward DFT, as the conjugate of the inverse of the
// conjugate.
template <int NT, int C, int A, bool CONJ>
__device__ __forceinline__ void sub_dfts(c64 (&H)[C][4], int r, int64_t boff, c64 *X,
                                         const double2 *__restrict__ blu,
                                         const double2 *__restrict__ tw, int twlen) {
  const int t = threadIdx.x;
  const bool bl = boff >= 0;
  const int L = bl ? blu_len(r) : r;
  const int bits = ilog2(L), ldx = padded_len<double>(L);
  const double2 *__restrict__ chirp = blu + (bl ? boff : 0);
#pragma unroll
  for (int q0 = 0; q0 < 4; q0 += A) {
    __syncthreads();  // X free
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int k1 = t + c * NT;
      if (k1 < r) {
        c64 cj = {1.0, 0.0};
        if (bl) cj = ld<double>(chirp, k1);
        const int pos = bl ? k1 : bit_rev(k1, bits);
#pragma unroll
        for (int a = 0; a < A; ++a) {
          c64 v = H[c][q0 + a];
          if (CONJ) v = cconj(v);
          X[a * ldx + pad<double>(pos)] = bl ? cmul(v, cj) : v;
        }
      }
    }
    if (bl) {
#pragma unroll
      for (int a = 0; a < A; ++a)
        for (int j = r + t; j < L; j += NT) X[a * ldx + pad<double>(j)] = c64{0.0, 0.0};
    }
    __syncthreads();
    if (bl)
      bluestein_conv<NT>(X, ldx, A, L, tw, twlen, chirp + r);
    else
      fused_fft<NT, true, 1>(X, ldx, A, L, tw, twlen);
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int j1 = t + c * NT;
      if (j1 < r) {
        c64 cj = {1.0, 0.0};
        if (bl) cj = ld<double>(chirp, j1);
#pragma unroll
        for (int a = 0; a < A; ++a) {
          c64 v = X[a * ldx + pad<double>(j1)];
          if (bl) v = cmul(v, cj);
          H[c][q0 + a] = CONJ ? cconj(v) : v;
        }
      }
    }
  }
}

// as many arrays at a time as the launch's LDS (cap elements) holds
template <int NT, int C, bool CONJ>
__device__ __forceinline__ void all_dfts(c64 (&H)[C][4], int r, int64_t boff, c64 *X, int cap,
                                         const double2 *__restrict__ blu,
                                         const double2 *__restrict__ tw, int twlen) {
  const int ldx = padded_len<double>(boff >= 0 ? blu_len(r) : r);
  if (4 * ldx <= cap)
    sub_dfts<NT, C, 4, CONJ>(H, r, boff, X, blu, tw, twlen);
  else if (2 * ldx <= cap)
    sub_dfts<NT, C, 2, CONJ>(H, r, boff, X, blu, tw, twlen);
  else
    sub_dfts<NT, C, 1, CONJ>(H, r, boff, X, blu, tw, twlen);
}

// e^{2 pi i k / n}, from the table for a power of two
__device__ __forceinline__ c64 root_n(int k, int n, bool pow2, const double2 *__restrict__ tw,
                                      int twlen) {
  if (pow2) return ld<double>(tw, int64_t(k) * (twlen / n));
  return expi_q(k, n, 0.0);
}

template <int NT, int C>
__global__ __launch_bounds__(NT) void ring_synth64_kernel(
    int lmax, int nrings, int S, const int64_t *__restrict__ ring_start,
    const int32_t *__restrict__ ring_n, const int64_t *__restrict__ blu_off,
    const double2 *__restrict__ blu, const double2 *__restrict__ tw, int twlen, int cap,
    const c64 *__restrict__ F, double *__restrict__ maps, int64_t npix,
    const double *__restrict__ ref) {
  extern __shared__ char smem_raw[];
  c64 *X = reinterpret_cast<c64 *>(smem_raw);
  const ring_item it = decode_item(S, lmax, nrings, npix, ring_start, ring_n);
  const int t = threadIdx.x, n = it.n, r = n >> 2;
  const int64_t boff = blu_off[r];
  const c64 *__restrict__ f0 = F + it.f[0], *__restrict__ f1 = F + it.f[1];
  // coefficient m of both transforms as one complex value f0 + i f1, or the
  // conjugate term conj(f0) + i conj(f1)
  // (0 past lmax, read at lmax: no branch, so that loads are issued together)
  auto term = [&](int m, bool conj) {
    const int64_t i = int64_t(min(m, lmax)) * it.stride;
    const c64 a = f0[i];
    c64 b = {0.0, 0.0};
    if (it.has1) b = f1[i];
    const c64 v = conj ? c64{a.re + b.im, b.re - a.im} : c64{a.re - b.im, a.im + b.re};
    return m <= lmax ? v : c64{0.0, 0.0};
  };

  // ---- aliasing fold: bin k collects F_m for m = k (mod n) and conj(F_m) for
  // m = -k (mod n), m <= lmax
  c64 H[C][4];
  const int Q = NT / n;  // small rings: Q threads per bin, partial sums meet in LDS
  if (Q >= 2) {
    const int q = t / n, k = t - q * n;
    c64 s = {0.0, 0.0};
    if (q < Q) {
      for (int j = q; j * n <= lmax; j += 4 * Q) {
        c64 u[4], v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          u[i] = term((j + i * Q) * n + k, false);
          v[i] = term((j + i * Q + 1) * n - k, true);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) s = cadd(cadd(s, u[i]), v[i]);
      }
      X[t] = s;
    }
    __syncthreads();
#pragma unroll
    for (int k2 = 0; k2 < 4; ++k2) {
      c64 h = {0.0, 0.0};
      if (t < r)
        for (int j = 0; j < Q; ++j) h = cadd(h, X[j * n + t + r * k2]);
      H[0][k2] = h;
    }
  } else {
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int k1 = t + c * NT;
#pragma unroll
      for (int k2 = 0; k2 < 4; ++k2) H[c][k2] = c64{0.0, 0.0};
      // the four bins of k1 together: eight (or sixteen) loads in flight
      for (int m0 = 0; k1 < r && m0 <= lmax; m0 += n) {
        c64 u[4], v[4];
#pragma unroll
        for (int k2 = 0; k2 < 4; ++k2) {
          u[k2] = term(m0 + k1 + r * k2, false);
          v[k2] = term(m0 + n - k1 - r * k2, true);
        }
#pragma unroll
        for (int k2 = 0; k2 < 4; ++k2) H[c][k2] = cadd(cadd(H[c][k2], u[k2]), v[k2]);
      }
    }
  }
  // ---- radix-4 split
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int k1 = t + c * NT;
    const c64 w1 = root_n(k1 < r ? k1 : 0, n, boff < 0, tw, twlen);
    const c64 w2 = cmul(w1, w1), w3 = cmul(w2, w1);
    const c64 s02 = cadd(H[c][0], H[c][2]), d02 = csub(H[c][0], H[c][2]);
    const c64 s13 = cadd(H[c][1], H[c][3]), d13 = cmuli(csub(H[c][1], H[c][3]));
    H[c][0] = cadd(s02, s13);
    H[c][1] = cmul(cadd(d02, d13), w1);
    H[c][2] = cmul(csub(s02, s13), w2);
    H[c][3] = cmul(csub(d02, d13), w3);
  }
  all_dfts<NT, C, false>(H, r, boff, X, cap, blu, tw, twlen);

  // ---- pixels 4 j1 + j2
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int j1 = t + c * NT;
    if (j1 >= r) continue;
#pragma unroll
    for (int j2 = 0; j2 < 4; ++j2) {
      const int64_t p0 = it.px[0] + 4 * j1 + j2, p1 = it.px[1] + 4 * j1 + j2;
      maps[p0] = ref ? ref[p0] - H[c][j2].re : H[c][j2].re;
      if (it.has1) maps[p1] = ref ? ref[p1] - H[c][j2].im : H[c][j2].im;
    }
  }
}

// Analysis: pixels -> F[ring][m] = w e^{-i m phi0} DFT(f)_{m mod n}
template <int NT, int C>
__global__ __launch_bounds__(NT) void ring_anal64_kernel(
    int lmax, int nrings, const int64_t *__restrict__ ring_start,
    const int32_t *__restrict__ ring_n, const int32_t *__restrict__ ring_pnum,
    const int64_t *__restrict__ blu_off, const double2 *__restrict__ blu,
    const double2 *__restrict__ tw, int twlen, int cap, const double *__restrict__ maps,
    int64_t npix, const double *__restrict__ pixw, double wc, double weight, c64 *__restrict__ F) {
  extern __shared__ char smem_raw[];
  c64 *X = reinterpret_cast<c64 *>(smem_raw);
  const ring_item it = decode_item(1, lmax, nrings, npix, ring_start, ring_n);
  const int t = threadIdx.x, n = it.n, r = n >> 2;
  const int64_t boff = blu_off[r];
  c64 H[C][4];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int j1 = t + c * NT;
#pragma unroll
    for (int j2 = 0; j2 < 4; ++j2) {
      c64 v = {0.0, 0.0};
      if (j1 < r) {
        const int64_t p0 = it.px[0] + 4 * j1 + j2, p1 = it.px[1] + 4 * j1 + j2;
        v.re = maps[p0];
        if (it.has1) v.im = maps[p1];
        if (pixw) {
          v.re *= pixw[p0] * wc;
          if (it.has1) v.im *= pixw[p1] * wc;
        }
      }
      H[c][j2] = v;
    }
  }
  all_dfts<NT, C, true>(H, r, boff, X, cap, blu, tw, twlen);
  // bins k1 + r k2: sum_j2 (-i)^(j2 k2) e^{-2 pi i j2 k1 / n} D_j2[k1]
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int k1 = t + c * NT;
    const c64 w1 = cconj(root_n(k1 < r ? k1 : 0, n, boff < 0, tw, twlen));
    const c64 w2 = cmul(w1, w1), w3 = cmul(w2, w1);
    const c64 y0 = H[c][0], y1 = cmul(H[c][1], w1), y2 = cmul(H[c][2], w2), y3 = cmul(H[c][3], w3);
    const c64 s02 = cadd(y0, y2), d02 = csub(y0, y2);
    const c64 s13 = cadd(y1, y3), d13 = cmuli(csub(y3, y1));  // -i (y1 - y3)
    H[c][0] = cadd(s02, s13);
    H[c][1] = cadd(d02, d13);
    H[c][2] = csub(s02, s13);
    H[c][3] = csub(d02, d13);
  }
  // The two real transforms are split with the partner bin n - k, and every m
  // = k (mod n) gets weight e^{-i m phi0} times its bin; phi0 = pi / n or 0.
  const bool shifted = ring_pnum[it.ring] != 0;
  auto put = [&](int m, c64 av, c64 partner) {
    const c64 bv = cconj(partner);
    const c64 d0 = {0.5 * (av.re + bv.re), 0.5 * (av.im + bv.im)};
    const c64 d1 = {0.5 * (av.im - bv.im), -0.5 * (av.re - bv.re)};  // (a - b) / (2 i)
    const c64 ph = shifted ? cconj(expi_q(m % (2 * n), 2 * n, 0.0)) : c64{1.0, 0.0};
    const c64 v0 = cmul(d0, ph);
    F[it.f[0] + m] = c64{weight * v0.re, weight * v0.im};
    if (it.has1) {
      const c64 v1 = cmul(d1, ph);
      F[it.f[1] + m] = c64{weight * v1.re, weight * v1.im};
    }
  };
  if (n <= lmax && padded_len<double>(n) <= cap) {
    // several m per bin: all bins to LDS, the threads go over m (a polar ring
    // of four bins has lmax / 4 values of m for each)
    __syncthreads();
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int k1 = t + c * NT;
#pragma unroll
      for (int k2 = 0; k2 < 4; ++k2)
        if (k1 < r) X[pad<double>(k1 + r * k2)] = H[c][k2];
    }
    __syncthreads();
    for (int m = t; m <= lmax; m += NT) {
      const int k = m % n;
      put(m, X[pad<double>(k)], X[pad<double>(k ? n - k : 0)]);
    }
    return;
  }
  // one or a few m per bin: the partner (r - k1) + r (3 - k2) (r ((4 - k2) mod 4)
  // for k1 = 0) is exchanged through LDS two bins at a time, first k2 = 2, 3
  // for the outputs of k2 = 0, 1, then the others
  const int ldx = padded_len<double>(r);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    __syncthreads();
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int k1 = t + c * NT;
      if (k1 < r) {
        X[pad<double>(k1)] = H[c][2 - 2 * h];
        X[ldx + pad<double>(k1)] = H[c][3 - 2 * h];
      }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int k1 = t + c * NT;
      if (k1 >= r) continue;
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int k2 = 2 * h + b, k = k1 + r * k2;
        const int p1 = k1 ? r - k1 : 0, p2 = k1 ? 3 - k2 : (4 - k2) & 3;
        const c64 av = H[c][k2];
        const c64 pv = p2 == k2 ? av : X[(p2 - (2 - 2 * h)) * ldx + pad<double>(p1)];
        for (int m = k; m <= lmax; m += n) put(m, av, pv);
      }
    }
  }
}

// LDS elements of a launch: four arrays of the longest transform if that stays
// within kLds64, else two, else one
constexpr int kLds64 = 4800;  // complex doubles: 75 KiB, two workgroups per CU
int lds_elements(const ga_plan *p, int least) {
  const int ldx = padded_len<double>(p->max_L);
  int n = 4 * ldx;
  if (n > kLds64) n = 2 * ldx;
  if (n > kLds64) n = ldx;
  return std::max(n, least);
}

}  // namespace

#define GA_RING64(KERNEL, ...)                                                                   \
  do {                                                                                          \
    GA_CHECK_HIP(hipFuncSetAttribute((const void *)KERNEL,                                       \
                                     hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));     \
    hipLaunchKernelGGL(KERNEL, dim3(unsigned(nitem)), dim3(NT), lds, stream, __VA_ARGS__);       \
  } while (0)

template <int NT, int C>
static int launch_synth64(const ga_plan *p, int S, const double *F, double *maps,
                          const double *ref, hipStream_t stream) {
  const int cap = lds_elements(p, NT);
  const size_t lds = size_t(cap) * sizeof(c64);
  GA_REQUIRE(lds <= 160 * 1024, GA_ERR_UNSUPPORTED, "ring synthesis needs %zu bytes of LDS", lds);
  const int nitem = S == 1 ? p->npairs : p->nrings;
  auto kfn = ring_synth64_kernel<NT, C>;
  GA_RING64(kfn, p->lmax, p->nrings, S, p->d_ring_start, p->d_ring_n, p->d_blu_off, p->d_blu64,
            p->d_tw64, p->tw_len, cap, reinterpret_cast<const c64 *>(F), maps, p->npix, ref);
  GA_LAUNCH_CHECK();
  return GA_OK;
}

template <int NT, int C>
static int launch_anal64(const ga_plan *p, const double *maps, const double *pixw, double wc,
                         double *F, hipStream_t stream) {
  const int cap = lds_elements(p, 2 * padded_len<double>(p->max_r));
  const size_t lds = size_t(cap) * sizeof(c64);
  GA_REQUIRE(lds <= 160 * 1024, GA_ERR_UNSUPPORTED, "ring analysis needs %zu bytes of LDS", lds);
  const int nitem = p->npairs;
  auto kfn = ring_anal64_kernel<NT, C>;
  GA_RING64(kfn, p->lmax, p->nrings, p->d_ring_start, p->d_ring_n, p->d_ring_pnum,
            p->d_blu_off, p->d_blu64, p->d_tw64, p->tw_len, cap, maps, p->npix, pixw, wc,
            4.0 * M_PI / double(p->npix), reinterpret_cast<c64 *>(F));
  GA_LAUNCH_CHECK();
  return GA_OK;
}

// Threads and k1 values per thread by the longest ring.  Whole alm2map at a small
// band limit (the rings are most of it), against half as many threads with twice
// the values and twice as many with half of them: nside 128 15.2, 15.2, 14.9 us; 200
// 21.6, 24.5, 26.0; 300 33.6, 40.9, 40.5; 512 43.8, 50.8, 52.8; 1024 124, 142, 159; 2048
// 681, 776, 963; the analysis likewise (below 129 64 threads are as good for the
// synthesis, but 17.1 against 15.6 us for the analysis).
#define GA_RING64_SIZES(FN, ...)                                                   \
  do {                                                                            \
    if (p->max_r <= 64) return FN<64, 1>(__VA_ARGS__);                            \
    if (p->max_r <= 128) return FN<128, 1>(__VA_ARGS__);                          \
    if (p->max_r <= 256) return FN<256, 1>(__VA_ARGS__);                          \
    if (p->max_r <= 512) return FN<256, 2>(__VA_ARGS__);                          \
    if (p->max_r <= 1024) return FN<256, 4>(__VA_ARGS__);                         \
    if (p->max_r <= 2048) return FN<512, 4>(__VA_ARGS__);                         \
    GA_REQUIRE(p->max_r <= 4096, GA_ERR_UNSUPPORTED,                              \
               "ring length 4 * %d not supported", p->max_r);                     \
    return FN<512, 8>(__VA_ARGS__);                                               \
  } while (0)

int launch_ring_synth_f64(const ga_plan *p, int S, const double *F, double *maps,
                          const double *ref, hipStream_t s) {
  GA_REQUIRE(S == 1 || S == 2, GA_ERR_INVALID, "one map or one pair of maps, not %d", S);
  GA_RING64_SIZES(launch_synth64, p, S, F, maps, ref, s);
}

int launch_ring_anal_f64(const ga_plan *p, const double *maps, const double *pixw, double wc,
                         double *F, hipStream_t s) {
  // the largest nside whose belt ring, padded, fits LDS as a whole, which is the
  // limit of the entry point; the kernel holds at most half a ring there (136 KB at
  // nside 4096, checked in launch_anal64)
  GA_REQUIRE(p->nside <= 2482, GA_ERR_UNSUPPORTED, "ring analysis: nside %d too large", p->nside);
  GA_RING64_SIZES(launch_anal64, p, maps, pixw, wc, F, s);
}

}  // namespace ga
