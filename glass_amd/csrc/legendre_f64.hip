// Plain FP64 Legendre stage of the scalar synthesis (one map, no MFMA).
//
// A lane owns RPL ring pairs of one m and runs the associated-Legendre recurrence
// in l for their cos(theta) in FP64, from the seed lambda_mm = c_m sin^m theta.  It
// accumulates the l-sums of a_lm lambda_lm split by the parity of l - m (static in
// the unrolled loop), which gives the north ring and its south mirror at once:
//     F_m(theta)      = E + O,   F_m(pi - theta) = E - O,
// because lambda_lm(-x) = (-1)^(l+m) lambda_lm(x).
//
// Coefficients and alm are wave-uniform: scalar loads, kRows rows at a time,
// which serve all RPL pairs.  Values far below the range that matters are kept
// scaled (to_scaled_low) and rescaled every 2 kRows rows, so no step has a test.
// NORM runs the normalised form y_l = lambda_l / c_l, two operations a step
// instead of three, against alm that a first pass has multiplied by c_l; the
// plain form a (x lambda_{l-1} - b lambda_{l-2}) reads the alm as they are and
// saves that launch.  (As (a x) lambda_{l-1} - (a b) lambda_{l-2} it would be one
// operation deep instead of two, but the sums' errors 3 to 17 % larger.)
//
// Bound: FP64 issue, 4 (NORM) or 5 operations per (l, m, ring pair).  Measured at
// nside 1024, lmax 2048: 705 us (one pair per lane, a test of the scale and
// three operations in each step: 1377 us), of which the seeds take 80 us and
// the stores 20.  Issuing each batch of scalar loads one turn ahead changed
// nothing (716 against 711 us), four pairs per lane neither.
#include <algorithm>

#include "common.h"
#include "device.h"
#include "kernels.h"

namespace ga {

namespace {

constexpr int kRows = 8;           // rows per batch of scalar loads
constexpr int64_t kManyWaves = 12288;  // see launch_legendre_synth_f64

enum { kPlain, kNorm, kDiff };  // forms of the recurrence

template <int RPL>
struct synth_state {
  double x[RPL], p0[RPL], p1[RPL];  // x: cos(theta), twice that in the normalised forms
  double2 acc[2][RPL];              // by the parity of l - m
  int k[RPL];

  // one row: c = (a, b) or (h, -)
  template <int FORM>
  __device__ __forceinline__ void step(int par, double2 c, double2 a) {
#pragma unroll
    for (int j = 0; j < RPL; ++j) {
      if (FORM == kPlain) {
        const double y = c.x * fma(x[j], p1[j], -(c.y * p0[j]));
        p0[j] = p1[j];
        p1[j] = y;
      } else {
        norm_step<FORM == kDiff>(c.x, x[j], p0[j], p1[j]);
      }
      acc[par][j].x = fma(p1[j], a.x, acc[par][j].x);
      acc[par][j].y = fma(p1[j], a.y, acc[par][j].y);
    }
  }
};

template <int FORM>
__device__ __forceinline__ double2 row_coef(const double *__restrict__ t, int i) {
  return FORM == kPlain ? reinterpret_cast<const double2 *>(t)[i] : double2{t[i], 0.0};
}

// the nl rows of one m
template <int FORM, int RPL>
__device__ __forceinline__ void synth_rows(synth_state<RPL> &s, int nl,
                                           const double *__restrict__ c,
                                           const double2 *__restrict__ a) {
  bool scaled = true;  // wave-uniform: some value of the wave may still be scaled
  int i = 0;
  for (; i + kRows <= nl; i += kRows) {
    double2 cv[kRows], av[kRows];
#pragma unroll
    for (int q = 0; q < kRows; ++q) cv[q] = row_coef<FORM>(c, i + q);
#pragma unroll
    for (int q = 0; q < kRows; ++q) av[q] = a[i + q];
#pragma unroll
    for (int q = 0; q < kRows; ++q) s.template step<FORM>(q & 1, cv[q], av[q]);
    if (scaled && (i & kRows)) {
      bool any = false;
#pragma unroll
      for (int j = 0; j < RPL; ++j) {
        rescale_low(s.p0[j], s.p1[j], s.k[j]);
        any |= s.k[j] < 0;
      }
      scaled = wave_any(any);
    }
  }
  // the last rows (the turns leave i even), loaded together
  double2 cv[kRows - 1], av[kRows - 1];
#pragma unroll
  for (int q = 0; q < kRows - 1; ++q) {
    const int r = min(i + q, nl - 1);
    cv[q] = row_coef<FORM>(c, r);
    av[q] = a[r];
  }
#pragma unroll
  for (int q = 0; q < kRows - 1; ++q)
    if (i + q < nl) s.template step<FORM>(q & 1, cv[q], av[q]);
}

// (two pairs per lane in the registers of seven waves per SIMD: 763 us for alm2map
// at nside 1024, lmax 2048, 799 at six)
template <int RPL, bool NORM>
__global__ __launch_bounds__(256, RPL == 2 ? 7 : 1) void legendre_synth_f64_kernel(
    int lmax, int npairs, int nrings, int nrg, const double *__restrict__ z,
    const double *__restrict__ sth, const double *__restrict__ tab /* h, or (a, b) */,
    const double *__restrict__ cm, const int32_t *__restrict__ ring_pnum,
    const int32_t *__restrict__ ring_pden, const double2 *__restrict__ alm,
    double2 *__restrict__ F) {
  int m, rg;
  if (!decode_m_run8(lmax, nrg, m, rg)) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int rp0 = (rg * (blockDim.x >> 6) + wave) * 64 * RPL + lane;
  if (rp0 - lane >= npairs) return;  // wave-uniform; the kernel has no barriers
  const bool diff = NORM && norm_diff(lmax, m);
  synth_state<RPL> s;
#pragma unroll
  for (int j = 0; j < RPL; ++j) {
    const int rp = min(rp0 + 64 * j, npairs - 1);
    s.x[j] = NORM ? 2.0 * z[rp] : z[rp];
    s.p1[j] = 0.0;
    legendre_seed_low(cm[m], sth[rp], m, s.p0[j], s.k[j]);
    // the first row (h = -1, or (a, b) = (1, -1)) yields the seed
    if (NORM && !diff) s.p0[j] = -s.p0[j];
    s.acc[0][j] = s.acc[1][j] = double2{0.0, 0.0};
  }
  const int64_t base = hp_index(lmax, m, m);
  const double2 *__restrict__ a = alm + base;
  const double *__restrict__ c = tab + (NORM ? 1 : 2) * base;
  const int nl = lmax + 1 - m;
  if (!NORM) synth_rows<kPlain>(s, nl, c, a);
  else if (diff) synth_rows<kDiff>(s, nl, c, a);
  else synth_rows<kNorm>(s, nl, c, a);

  const int64_t stride = lmax + 1;
#pragma unroll
  for (int j = 0; j < RPL; ++j) {
    const int rp = rp0 + 64 * j;
    if (rp >= npairs) continue;
    double2 e = s.acc[0][j], o = s.acc[1][j];
    if (m == 0) e.y = o.y = 0.0;  // Im a_l0 is ignored (real map)
    // ring phase e^{i m phi0}, phi0 = 2 pi pnum / pden (the same on the south mirror)
    const int pnum = ring_pnum[rp], pden = ring_pden[rp];
    double ps = 0.0, pc = 1.0;
    if (pnum) sincospi(2.0 * double((int64_t(m) * pnum) % pden) / double(pden), &ps, &pc);
    const double nr = e.x + o.x, ni = e.y + o.y, sr = e.x - o.x, si = e.y - o.y;
    F[int64_t(rp) * stride + m] = double2{nr * pc - ni * ps, nr * ps + ni * pc};
    if (rp < npairs - 1)
      F[int64_t(nrings - 1 - rp) * stride + m] = double2{sr * pc - si * ps, sr * ps + si * pc};
  }
}

__global__ __launch_bounds__(256) void scale_alm_kernel(int64_t n, const double2 *__restrict__ alm,
                                                        const double *__restrict__ c,
                                                        double2 *__restrict__ out) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i < n) out[i] = double2{alm[i].x * c[i], alm[i].y * c[i]};
}

template <int RPL, bool NORM>
int launch(const ga_plan *p, const double *alm, double *F, hipStream_t stream) {
  const int nw = std::min(4, (p->npairs + 64 * RPL - 1) / (64 * RPL));
  const int nrg = (p->npairs + 64 * RPL * nw - 1) / (64 * RPL * nw);
  hipLaunchKernelGGL((legendre_synth_f64_kernel<RPL, NORM>), dim3(m_run8_blocks(p->lmax, nrg)),
                     dim3(64 * nw), 0, stream, p->lmax, p->npairs, p->nrings, nrg, p->d_z, p->d_sth,
                     NORM ? p->d_h64 : reinterpret_cast<const double *>(p->d_ab), p->d_cm,
                     p->d_ring_pnum, p->d_ring_pden, reinterpret_cast<const double2 *>(alm),
                     reinterpret_cast<double2 *>(F));
  GA_LAUNCH_CHECK();
  return GA_OK;
}

}  // namespace

int launch_legendre_synth_f64(const ga_plan *p, const double *alm, double *F, double *scratch,
                              size_t scratch_doubles, hipStream_t stream) {
  // The normalised form saves an operation in five and, with two pairs per
  // lane, half the scalar loads, but costs the launch of the scaling pass and
  // the wait between the two, and half the waves.  Whole alm2map by waves of one
  // pair per lane, plain / normalised: 4104 (nside 256, lmax 512) 35 / 59 us; 9000
  // (300, 899) 100 / 109; 10413 (400, 800) 112 / 110; 12816 (512, 800) 114 / 113; 14416
  // (512, 900) 145 / 126; 16384 (512, 1023) 158 / 147; 35232 (1024, 1100) 373 / 316.
  const int64_t waves = int64_t(p->lmax + 1) * ((p->npairs + 63) / 64);
  if (waves < kManyWaves || scratch_doubles < size_t(2 * p->nalm))
    return launch<1, false>(p, alm, F, stream);
  hipLaunchKernelGGL(scale_alm_kernel, dim3(unsigned((p->nalm + 255) / 256)), dim3(256), 0, stream,
                     p->nalm, reinterpret_cast<const double2 *>(alm), p->d_c64,
                     reinterpret_cast<double2 *>(scratch));
  GA_LAUNCH_CHECK();
  return launch<2, true>(p, scratch, F, stream);
}

}  // namespace ga
