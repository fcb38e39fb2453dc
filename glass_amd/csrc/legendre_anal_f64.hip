// Plain FP64 Legendre stage of the analysis (one map):
//   a_lm = sum_rp lambda_lm(theta_rp) Q_p[rp],   Q_0 = F_N + F_S, Q_1 = F_N - F_S,
// p the parity of l - m, F the weighted, phase-removed ring coefficients.
//
// A workgroup of up to four waves takes one m; a lane owns RPL ring pairs, whose
// recurrences (the normalised form y_l = lambda_l / c_l, two operations a step,
// norm_step) and Q stay in registers.  The sum runs over lanes, so each lane first adds
// its own pairs for kRows rows of l (32 real sums in registers), and the wave
// then reduces all 32 sums at once: every exchange halves the number of sums
// a lane carries while it adds the partner's half (permlane swaps, then DPP
// moves), so the 32 sums cost about 125 instructions together instead of a
// six-step butterfly each.  The waves' results meet in LDS in a fixed order,
// and one of the waves multiplies them by c_l and stores them.
// Values far below the range that matters are kept scaled (to_scaled_low) and
// rescaled once per kRows rows, so no step has a test.
//
// Bound: FP64 issue, 4 RPL operations per row and wave plus about 8 for the
// reduction.  RPL grows with the number of ring pairs (1, 2, 4, 8 up to 256,
// 512, 1024 pairs and above), so that one workgroup covers an m and small
// maps still have four waves for each.  Measured at nside 1024, lmax 2048:
// 878 us (a butterfly of each sum through LDS shuffles: 4803 us); nside 256,
// lmax 512: 48 us (482 us).
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "device.h"
#include "kernels.h"

namespace ga {

namespace {

constexpr int kRows = 16;        // l rows per reduction
constexpr int kSums = 2 * kRows;  // (re, im) of each
static_assert(kSums == 32, "wave_sums32");

// the values of kRows rows on the wave's ring pairs and each lane's part of their
// sums (re, im)
template <int RPL, bool DIFF>
__device__ __forceinline__ void anal_rows(const double (&h)[kRows], const double (&X)[RPL],
                                          double (&p0)[RPL], double (&p1)[RPL],
                                          const double2 (&q)[2][RPL], double (&v)[kSums]) {
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
#pragma unroll
    for (int j = 0; j < RPL; ++j) {
      norm_step<DIFF>(h[i], X[j], p0[j], p1[j]);
      const double y = p1[j];
      v[2 * i] = j == 0 ? y * q[i & 1][j].x : fma(y, q[i & 1][j].x, v[2 * i]);
      v[2 * i + 1] = j == 0 ? y * q[i & 1][j].y : fma(y, q[i & 1][j].y, v[2 * i + 1]);
    }
    __builtin_amdgcn_sched_barrier(0);  // rows in order: registers
  }
}

template <int RPL>
__global__ __launch_bounds__(256, RPL == 8 ? 2 : 3) void legendre_anal_f64_kernel(
    int lmax, int npairs, int nrings, int nrg, const double *__restrict__ z,
    const double *__restrict__ sth, const double *__restrict__ h,
    const double *__restrict__ c, const double *__restrict__ cm,
    const double2 *__restrict__ F, double *__restrict__ out /* [slot][idx] (re, im) */,
    int64_t slot_stride, int accumulate) {
  __shared__ double red[2][4][kSums];
  int m, rg;
  if (!decode_m_run8(lmax, nrg, m, rg)) return;  // whole workgroup
  const int nw = blockDim.x >> 6, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int rp0 = (rg * nw + wave) * 64 * RPL + lane;
  const int64_t base = hp_index(lmax, m, m);

  const bool diff = norm_diff(lmax, m);
  double X[RPL], p0[RPL], p1[RPL];
  int k[RPL];
  double2 q[2][RPL];
#pragma unroll
  for (int j = 0; j < RPL; ++j) {
    const int rp = rp0 + 64 * j;
    const int rpc = min(rp, npairs - 1);
    X[j] = 2.0 * z[rpc];
    p1[j] = 0.0;
    legendre_seed_low(cm[m], sth[rpc], m, p0[j], k[j]);
    if (!diff) p0[j] = -p0[j];  // the first row (h = -1) yields the seed
    double2 fn = {0.0, 0.0}, fs = {0.0, 0.0};
    if (rp < npairs) fn = F[int64_t(rp) * (lmax + 1) + m];
    if (rp < npairs - 1) fs = F[int64_t(nrings - 1 - rp) * (lmax + 1) + m];
    q[0][j] = double2{fn.x + fs.x, fn.y + fs.y};
    q[1][j] = double2{fn.x - fs.x, fn.y - fs.y};
  }

  h += base;
  const int nl = lmax + 1 - m;
  bool scaled = true;  // wave-uniform: some value of the wave may still be scaled
  out += 2 * (int64_t(rg) * slot_stride + base);
  // the coefficient table is padded: the rows past lmax in the last turn are
  // computed and not stored
  auto all_rows = [&](auto form) {
    int buf = 0, turn = 0;
    for (int i0 = 0; i0 < nl; i0 += kRows) {
      double hv[kRows], v[kSums];
#pragma unroll
      for (int i = 0; i < kRows; ++i) hv[i] = h[i0 + i];
      anal_rows<RPL, form.value>(hv, X, p0, p1, q, v);
      const double sum = wave_sums32(v, lane);
      if (!(lane & 1)) red[buf][wave][lane >> 1] = sum;
      if (scaled) {
        bool any = false;
#pragma unroll
        for (int j = 0; j < RPL; ++j) {
          rescale_low(p0[j], p1[j], k[j]);
          any |= k[j] < 0;
        }
        scaled = wave_any(any);
      }
      __syncthreads();
      if (wave == turn && lane < kSums) {
        double s = red[buf][0][lane];
        for (int w = 1; w < nw; ++w) s += red[buf][w][lane];
        const int i = i0 + (lane >> 1);
        if (i < nl) {
          s = (m == 0 && (lane & 1)) ? 0.0 : s * c[base + i];
          double *o = out + 2 * int64_t(i0) + lane;
          *o = accumulate ? *o + s : s;
        }
      }
      buf ^= 1;  // the other buffer was read before this turn's barrier
      turn = turn + 1 == nw ? 0 : turn + 1;
    }
  };
  if (diff) all_rows(std::true_type());
  else all_rows(std::false_type());
}

}  // namespace

int launch_legendre_anal_f64(const ga_plan *p, const double *F, double *alm, double *partial,
                             bool accumulate, hipStream_t stream) {
  // the fewest pairs per lane whose four waves cover an m: fewer need several
  // workgroups and partial sums per m, twice as many halve the waves (whole
  // map2alm, and with twice as many: nside 128, lmax 256 27 and 28 us; 256, 512 54
  // and 65; 300, 767 114 and 150; 512, 1023 180 and 220)
  int rpl = 1;
  while (rpl < 8 && 256 * rpl < p->npairs) rpl *= 2;
  const int nw = std::min(4, (p->npairs + 64 * rpl - 1) / (64 * rpl));
  const int nrg = (p->npairs + 64 * rpl * nw - 1) / (64 * rpl * nw);
  GA_REQUIRE(nrg == 1 || nrg <= anal_partial_slots(p), GA_ERR_UNSUPPORTED,
             "partial slots %d > %d", nrg, anal_partial_slots(p));
  // one workgroup per m adds to the alm itself; several leave partial sums
  double *out = nrg == 1 ? alm : partial;
#define GA_ANAL64(RPL_)                                                                          \
  hipLaunchKernelGGL(legendre_anal_f64_kernel<RPL_>, dim3(m_run8_blocks(p->lmax, nrg)),           \
                     dim3(64 * nw), 0, stream, p->lmax, p->npairs, p->nrings, nrg, p->d_z,        \
                     p->d_sth, p->d_h64, p->d_c64, p->d_cm, reinterpret_cast<const double2 *>(F), \
                     out, p->nalm, nrg == 1 && accumulate)
  if (rpl == 1) GA_ANAL64(1);
  else if (rpl == 2) GA_ANAL64(2);
  else if (rpl == 4) GA_ANAL64(4);
  else GA_ANAL64(8);
#undef GA_ANAL64
  GA_LAUNCH_CHECK();
  if (nrg == 1) return GA_OK;
  return launch_reduce_partials_f64(p->nalm, nrg, partial, alm, accumulate, stream);
}

}  // namespace ga
