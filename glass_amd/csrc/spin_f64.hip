// Spin-s synthesis Legendre stage in plain FP64 (one pair of maps), s = 1, 2.
//
//   Q_m = sum_l E F+ + i B F-,  U_m = sum_l B F+ - i E F-,
//   F+- = -(lambda+ +- (-1)^s lambda-) / 2
// with lambda+- the normalised Wigner-d functions of spin +s and -s; the south
// ring of a pair follows from F+(pi - t) = sigma F+(t), F-(pi - t) = -sigma F-(t),
// sigma = (-1)^(l+m+s).
//
// A lane owns one ring pair of one m and runs both recurrences from l0 = max(m, s).
// The sums are linear in lambda, so it accumulates lambda+ and lambda- against E
// and B as they come (eight FMAs a step, split by the parity of l - l0, which is
// static in the unrolled loop) and forms Q and U once, after the loop; the two
// recurrence steps cost six more operations.  E, B and the recurrence
// coefficients are wave-uniform and arrive by scalar loads, kChunk rows at a
// time.  Coefficients below the spin (l < s, which a spin-s field does not have)
// are not read.  Values far below the range that matters are kept scaled
// (to_scaled_low) and rescaled once per chunk, so no step has a test.  Skipping
// the sums while a whole wave is scaled would save 1 to 5 % (nside 300, 1024),
// but a coefficient that is not finite would then not reach every ring.
//
// Bound: FP64 issue, 14 operations per (l, m, ring pair).  Measured at nside
// 300, lmax 767 (E and B): 141 us (chunks of 4 rows 169 us, two ring pairs per
// lane 185 us); 3820 us when the sums were combined at every step into an
// array indexed by the parity at run time, which lived in scratch memory.
#include "common.h"
#include "device.h"
#include "kernels.h"

namespace ga {

namespace {

constexpr int kChunk = 8;  // rows per batch of scalar loads

struct spin_state {
  double x, a0, a1, b0, b1;  // (l-2, l-1) of +s and -s
  int kp, km;
  // [parity of l - l0]: lambda+ E, lambda+ B, lambda- E, lambda- B
  double2 pe[2], pb[2], me[2], mb[2];

  // one recurrence step; the new values are in a1, b1
  __device__ __forceinline__ void advance(double A, double AB, double C) {
    const double n1 = fma(fma(A, x, AB), a1, -(C * a0));
    const double n2 = fma(fma(A, x, -AB), b1, -(C * b0));
    a0 = a1;
    a1 = n1;
    b0 = b1;
    b1 = n2;
  }
  __device__ __forceinline__ void add(int par, double2 e, double2 b) {
    axpy(a1, e, pe[par]);
    axpy(a1, b, pb[par]);
    axpy(b1, e, me[par]);
    axpy(b1, b, mb[par]);
  }
  static __device__ __forceinline__ void axpy(double v, double2 c, double2 &acc) {
    acc.x = fma(v, c.x, acc.x);
    acc.y = fma(v, c.y, acc.y);
  }
  __device__ __forceinline__ void rescale() {
    rescale_low(a0, a1, kp);
    rescale_low(b0, b1, km);
  }
  __device__ __forceinline__ bool any_scaled() const { return wave_any(kp < 0 || km < 0); }
};

__global__ __launch_bounds__(256) void spin_synth_f64_kernel(
    int lmax, int npairs, int nrings, int spin, int nrg, const double *__restrict__ z,
    const double *__restrict__ sth, const double *__restrict__ tab /* (A, A B, C) per (l, m) */,
    const double2 *__restrict__ seeds /* [+s | -s][m]: (signed mantissa, exponent) */,
    const int32_t *__restrict__ ring_pnum, const int32_t *__restrict__ ring_pden,
    const double2 *__restrict__ E, const double2 *__restrict__ B, double2 *__restrict__ Fo) {
  int m, rg;
  if (!decode_m_run8(lmax, nrg, m, rg)) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int rp = (rg * 4 + wave) * 64 + lane;
  if (rp - lane >= npairs) return;  // wave-uniform; the kernel has no barriers

  spin_state s;
  const int l0 = m > spin ? m : spin;
  const double2 kp = seeds[m], km = seeds[lmax + 1 + m];
  {
    const int rpc = min(rp, npairs - 1);
    const double x = z[rpc], st = sth[rpc];
    double sh = sqrt(0.5 * (1.0 - x)), ch = sqrt(0.5 * (1.0 + x));
    if (x > 0.5) sh = st / (2.0 * ch);
    else if (x < -0.5) ch = st / (2.0 * sh);
    const int dif = m > spin ? m - spin : spin - m;
    double ms1, ms2, mc1, mc2;
    long long es1, es2, ec1, ec2;
    scaled_power(sh, m + spin, ms1, es1);
    scaled_power(ch, dif, mc1, ec1);
    scaled_power(sh, dif, ms2, es2);
    scaled_power(ch, m + spin, mc2, ec2);
    int t;
    double v = frexp(kp.x * ms1 * mc1, &t), sp, sm;
    to_scaled_low(v, (long long)kp.y + es1 + ec1 + t, sp, s.kp);
    v = frexp(km.x * ms2 * mc2, &t);
    to_scaled_low(v, (long long)km.y + es2 + ec2 + t, sm, s.km);
    // the (0, 0, -1) row at l0 turns (seed, 0) into the seed
    s.x = x;
    s.a0 = sp;
    s.b0 = sm;
    s.a1 = s.b1 = 0.0;
#pragma unroll
    for (int p = 0; p < 2; ++p)
      s.pe[p] = s.pb[p] = s.me[p] = s.mb[p] = double2{0.0, 0.0};
  }

  const int64_t base = hp_index(lmax, m, m);
  const double *__restrict__ cf = tab + 3 * base;
  const double2 *__restrict__ e = E + base, *__restrict__ b = B + base;
  const int nl = lmax + 1 - m;
  int i = l0 - m;
  bool scaled = s.any_scaled();  // wave-uniform
  for (; i + kChunk <= nl; i += kChunk) {
    double c[3 * kChunk];
    double2 ev[kChunk], bv[kChunk];
#pragma unroll
    for (int q = 0; q < 3 * kChunk; ++q) c[q] = cf[3 * i + q];
#pragma unroll
    for (int q = 0; q < kChunk; ++q) ev[q] = e[i + q];
#pragma unroll
    for (int q = 0; q < kChunk; ++q) bv[q] = b[i + q];
#pragma unroll
    for (int q = 0; q < kChunk; ++q) {
      s.advance(c[3 * q], c[3 * q + 1], c[3 * q + 2]);
      s.add(q & 1, ev[q], bv[q]);
    }
    if (scaled) {
      s.rescale();
      scaled = s.any_scaled();
    }
  }
#pragma unroll
  for (int q = 0; q < kChunk - 1; ++q)  // the last rows
    if (i + q < nl) {
      s.advance(cf[3 * (i + q)], cf[3 * (i + q) + 1], cf[3 * (i + q) + 2]);
      s.add(q & 1, e[i + q], b[i + q]);
    }

  const double sg = (spin & 1) ? -1.0 : 1.0;
  const int64_t stride = 2 * int64_t(lmax + 1);  // output [ring][m][Q, U]
  if (rp >= npairs) return;
  // ring phase e^{i m phi0} (the same on the south mirror)
  const int pnum = ring_pnum[rp], pden = ring_pden[rp];
  double ps = 0.0, pc = 1.0;
  if (pnum) sincospi(2.0 * double((int64_t(m) * pnum) % pden) / double(pden), &ps, &pc);
  const cplx<double> ph = {pc, ps};
  cplx<double> qa[2], qb[2], ua[2], ub[2];  // by the parity of l - l0
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    double2 PE = s.pe[p], PB = s.pb[p], ME = s.me[p], MB = s.mb[p];
    if (m == 0) PE.y = PB.y = ME.y = MB.y = 0.0;  // Im a_l0 is ignored (real maps)
    const cplx<double> pE = {-0.5 * (PE.x + sg * ME.x), -0.5 * (PE.y + sg * ME.y)};  // E F+
    const cplx<double> mE = {-0.5 * (PE.x - sg * ME.x), -0.5 * (PE.y - sg * ME.y)};  // E F-
    const cplx<double> pB = {-0.5 * (PB.x + sg * MB.x), -0.5 * (PB.y + sg * MB.y)};
    const cplx<double> mB = {-0.5 * (PB.x - sg * MB.x), -0.5 * (PB.y - sg * MB.y)};
    qa[p] = pE;
    qb[p] = cmuli(mB);
    ua[p] = pB;
    ub[p] = cplx<double>{mE.im, -mE.re};  // -i E F-
  }
  // sigma = (-1)^(l + m + s) = south on even, -south on odd l - l0
  const double south = ((l0 + m + spin) & 1) ? -1.0 : 1.0;
  const cplx<double> qn = cadd(cadd(qa[0], qb[0]), cadd(qa[1], qb[1]));
  const cplx<double> un = cadd(cadd(ua[0], ub[0]), cadd(ua[1], ub[1]));
  const cplx<double> qs = cadd(csub(qa[0], qb[0]), csub(qb[1], qa[1]));
  const cplx<double> us = cadd(csub(ua[0], ub[0]), csub(ub[1], ua[1]));
  const cplx<double> q0 = cmul(qn, ph), u0 = cmul(un, ph);
  double2 *o = Fo + int64_t(rp) * stride + 2 * m;
  o[0] = double2{q0.re, q0.im};
  o[1] = double2{u0.re, u0.im};
  if (rp < npairs - 1) {
    const cplx<double> q1 = cmul(qs, ph), u1 = cmul(us, ph);
    o = Fo + int64_t(nrings - 1 - rp) * stride + 2 * m;
    o[0] = double2{south * q1.re, south * q1.im};
    o[1] = double2{south * u1.re, south * u1.im};
  }
}

}  // namespace

int launch_spin_synth_f64(const ga_plan *p, int spin, const double *E, const double *B, double *Fo,
                          hipStream_t stream) {
  GA_REQUIRE(spin >= 1 && spin <= 2 && p->d_spin[spin] && p->d_spin_seed[spin], GA_ERR_INVALID,
             "spin %d tables not prepared (call ga_plan_prepare_spin)", spin);
  const int nrg = (p->npairs + 255) / 256;
  hipLaunchKernelGGL(spin_synth_f64_kernel, dim3(m_run8_blocks(p->lmax, nrg)), dim3(256), 0, stream,
                     p->lmax, p->npairs, p->nrings, spin, nrg, p->d_z, p->d_sth, p->d_spin[spin],
                     p->d_spin_seed[spin], p->d_ring_pnum, p->d_ring_pden,
                     reinterpret_cast<const double2 *>(E), reinterpret_cast<const double2 *>(B),
                     reinterpret_cast<double2 *>(Fo));
  GA_LAUNCH_CHECK();
  return GA_OK;
}

}  // namespace ga
