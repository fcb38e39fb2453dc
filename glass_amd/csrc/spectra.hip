// Angular power spectrum <-> angular correlation function on Gauss-Legendre
// nodes, the transforms of the Gaussian-spectra solver (glass/grf/_solver.py
// :27-148 and glass/grf/_core.py:141-184, where the transformcl package does
// them).
//
//   corr(x_k) = sum_l (2l+1) / (4 pi) cl_l P_l(x_k)                (cl2corr)
//   cl_l      = 2 pi sum_k w_k corr(x_k) P_l(x_k)                   (corr2cl)
//
// With n Gauss-Legendre nodes (x_k, w_k) and n coefficients l < n the pair is
// exact (products P_l P_l' of degree < 2n - 1 are integrated exactly), so
// corr2cl(cl2corr(cl)) = cl to rounding.  P_l by a recurrence in l in FP64, one
// lane per node; corr2cl reduces 32 l at a time over the 64 nodes of a wave and
// then over waves in a fixed order, so the result does not depend on scheduling.
// The nodes come from Newton's method on P_n from the asymptotic first guess
// cos(pi (i + 3/4) / (n + 1/2)), one thread per node pair (x, -x).
#include "common.h"
#include "device.h"
#include "kernels.h"

namespace ga {
namespace {

__global__ __launch_bounds__(256) void gl_nodes_kernel(int n, double *__restrict__ x,
                                                       double *__restrict__ w) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (n + 1) / 2) return;
  double z = cos(M_PI * (double(i) + 0.75) / (double(n) + 0.5));
  double dp = 1.0;
  for (int it = 0; it < 100; ++it) {
    double p0 = 1.0, p1 = z;
    for (int k = 2; k <= n; ++k) {
      const double p2 = (double(2 * k - 1) * z * p1 - double(k - 1) * p0) / double(k);
      p0 = p1;
      p1 = p2;
    }
    dp = double(n) * (z * p1 - p0) / (z * z - 1.0);
    const double dz = p1 / dp;
    z -= dz;
    if (fabs(dz) < 1e-13) break;  // quadratic convergence: the step left ~dz^2
  }
  {  // derivative at the converged node
    double p0 = 1.0, p1 = z;
    for (int k = 2; k <= n; ++k) {
      const double p2 = (double(2 * k - 1) * z * p1 - double(k - 1) * p0) / double(k);
      p0 = p1;
      p1 = p2;
    }
    dp = double(n) * (z * p1 - p0) / (z * z - 1.0);
  }
  const double wi = 2.0 / ((1.0 - z * z) * dp * dp);
  // ascending order: x[n - 1 - i] = +z (z > 0 for i < n / 2), x[i] = -z
  x[n - 1 - i] = z;
  w[n - 1 - i] = wi;
  x[i] = -z;
  w[i] = wi;
  if ((n & 1) && i == n / 2) x[i] = 0.0;
}

// P_l by differences: with D_l = P_l - P_{l-1} and s = 1 / l,
//   D_l = (1 - s) D_{l-1} + (2 - s) (x - 1) P_{l-1},   P_l = P_{l-1} + D_l.
// Near x = 1, where the three-term form loses most (its coefficients tend to the
// constants 2 x and 1, whose rounding then pushes the same way row after row),
// both terms are small.  A node x < 0 takes P_l(x) = (-1)^l P_l(-x): its odd rows
// count with the other sign.  Error of (2l + 1) P_l against its value, RMS over all
// rows and nodes at n = nl = 200, 1000, 6147: 1.7e-15, 8.0e-15, 4.1e-14; the
// three-term form with a division in every step 7.8e-15, 3.3e-13, 3.7e-12, with
// rounded coefficients for each row 6.3e-14, 3.6e-13, 4.1e-12.
//
// Lane i works out the row l0 + i (its division would otherwise be done by every
// lane in every step) into LDS, from where all lanes read it.  From (D, P) = (1, 0)
// the row of l = 0 (s = 0) yields P_0 = 1.
__device__ __forceinline__ double legendre_row(int l) { return l == 0 ? 0.0 : 1.0 / l; }
__device__ __forceinline__ double legendre_step(double s, double xm, double xm2, double &d,
                                                double &p) {
  d = fma(fma(-s, xm, xm2), p, fma(-s, d, d));
  p += d;
  return p;
}

// One wave, 64 nodes.  Bound: the serial recurrence (one wave on each of n / 64
// CUs): 89 us at nl = n = 6147 (97 us as the three-term form with two rounded
// coefficients for each row; with the division in every step and a load of cl_l
// waited for in it 823 us).
__global__ __launch_bounds__(64) void cl2corr_kernel(int nl, const double *__restrict__ cl, int n,
                                                     const double *__restrict__ x,
                                                     double *__restrict__ corr) {
  __shared__ double row[2][64];
  __shared__ double c[2][64];
  const int lane = threadIdx.x, k = blockIdx.x * 64 + lane;
  const double xk = x[min(k, n - 1)];
  const double xm = fabs(xk) - 1.0, xm2 = 2.0 * xm;
  auto fill = [&](int buf, int l0) {
    const int l = l0 + lane;
    // rows past nl have c = 0 and s = 2, which only turns the sign of D: their
    // values stay finite where P_l grows without bound (|x| > 1)
    row[buf][lane] = l < nl ? legendre_row(l) : 2.0;
    c[buf][lane] = l < nl ? cl[l] * (double(2 * l + 1) / (4.0 * M_PI)) : 0.0;
  };
  double d = 1.0, p = 0.0, acc[2] = {0.0, 0.0};  // sums of the even and odd rows
  int buf = 0;
  fill(0, 0);
  __syncthreads();
  for (int l0 = 0; l0 < nl; l0 += 64, buf ^= 1) {
    if (l0 + 64 < nl) fill(buf ^ 1, l0 + 64);
    // 16 rows to registers while the 16 before them are run: a wave that is
    // alone on its CU hides no latency
    double r[4][16];
    double cv[4][16];
#pragma unroll
    for (int q = 0; q <= 4; ++q) {
      if (q < 4) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          r[q][j] = row[buf][16 * q + j];
          cv[q][j] = c[buf][16 * q + j];
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (q > 0) {
#pragma unroll
        for (int j = 0; j < 16; ++j)
          acc[j & 1] = fma(cv[q - 1][j], legendre_step(r[q - 1][j], xm, xm2, d, p), acc[j & 1]);
      }
    }
    __syncthreads();
  }
  if (k < n) corr[k] = xk < 0.0 ? acc[0] - acc[1] : acc[0] + acc[1];
}

// part[wave][l]: 2 pi sum over the wave's nodes of w_k corr_k P_l(x_k), 32 rows
// of l reduced over the wave at a time.  Bound as above, the reduction adding
// half: 159 us at n = nl = 6147 (a shuffle butterfly for every l: 2076 us).
__global__ __launch_bounds__(64) void corr2cl_kernel(int n, const double *__restrict__ x,
                                                     const double *__restrict__ w,
                                                     const double *__restrict__ corr, int nl,
                                                     double *__restrict__ part) {
  __shared__ double row[2][32];
  const int lane = threadIdx.x, k = blockIdx.x * 64 + lane;
  const bool ok = k < n;
  const double xk = ok ? x[k] : 1.0;
  const double xm = fabs(xk) - 1.0, xm2 = 2.0 * xm;
  const double a = ok ? 2.0 * M_PI * w[k] * corr[k] : 0.0;
  const double ap[2] = {a, xk < 0.0 ? -a : a};  // for even and odd rows
  double *__restrict__ out = part + int64_t(blockIdx.x) * nl;
  auto fill = [&](int buf, int l0) {
    if (lane < 32) row[buf][lane] = legendre_row(l0 + lane);
  };
  double d = 1.0, p = 0.0;
  int buf = 0;
  double r[32];  // rows 0..15 of a turn are loaded before the reduction of the last one
  fill(0, 0);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 16; ++j) r[j] = row[0][j];
  for (int l0 = 0; l0 < nl; l0 += 32) {
#pragma unroll
    for (int j = 16; j < 32; ++j) r[j] = row[buf][j];
    buf ^= 1;
    fill(buf, l0 + 32);
    __builtin_amdgcn_sched_barrier(0);
    double v[32];
#pragma unroll
    for (int j = 0; j < 32; ++j) v[j] = ap[j & 1] * legendre_step(r[j], xm, xm2, d, p);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 16; ++j) r[j] = row[buf][j];
    __builtin_amdgcn_sched_barrier(0);
    const double s = wave_sums32(v, lane);
    const int l = l0 + (lane >> 1);
    if (!(lane & 1) && l < nl) out[l] = s;
  }
}

// cl[l] = the waves' parts, four interleaved sums added in order
__global__ __launch_bounds__(256) void corr2cl_sum_kernel(int nl, int nwaves,
                                                          const double *__restrict__ part,
                                                          double *__restrict__ cl) {
  __shared__ double red[4][64];
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int l = blockIdx.x * 64 + lane;
  double acc = 0.0;
  if (l < nl)
    for (int wv = g; wv < nwaves; wv += 4) acc += part[int64_t(wv) * nl + l];
  red[g][lane] = acc;
  __syncthreads();
  if (g == 0 && l < nl) cl[l] = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
}

}  // namespace
}  // namespace ga

using namespace ga;

extern "C" int ga_legendre_nodes(int32_t n, double *x, double *w, void *stream) {
  clear_error();
  GA_REQUIRE(n >= 1 && x && w, GA_ERR_INVALID, "invalid argument");
  const int half = (n + 1) / 2;
  hipLaunchKernelGGL(gl_nodes_kernel, dim3((half + 255) / 256), dim3(256), 0, (hipStream_t)stream,
                     n, x, w);
  GA_LAUNCH_CHECK();
  return GA_OK;
}

extern "C" int ga_cl2corr(int32_t nl, const double *cl, int32_t n, const double *x, double *corr,
                          void *stream) {
  clear_error();
  GA_REQUIRE(nl >= 1 && n >= 1 && cl && x && corr, GA_ERR_INVALID, "invalid argument");
  hipLaunchKernelGGL(cl2corr_kernel, dim3((n + 63) / 64), dim3(64), 0, (hipStream_t)stream, nl,
                     cl, n, x, corr);
  GA_LAUNCH_CHECK();
  return GA_OK;
}

extern "C" int ga_corr2cl_workspace_size(int32_t n, int32_t nl, size_t *bytes) {
  clear_error();
  GA_REQUIRE(bytes && n >= 1 && nl >= 1, GA_ERR_INVALID, "invalid argument");
  *bytes = size_t((n + 63) / 64) * size_t(nl) * sizeof(double);
  return GA_OK;
}

extern "C" int ga_corr2cl(int32_t n, const double *x, const double *w, const double *corr,
                          int32_t nl, double *cl, void *ws, size_t ws_bytes, void *stream) {
  clear_error();
  GA_REQUIRE(n >= 1 && nl >= 1 && x && w && corr && cl && ws, GA_ERR_INVALID, "invalid argument");
  const int nwaves = (n + 63) / 64;
  const size_t need = size_t(nwaves) * size_t(nl) * sizeof(double);
  GA_REQUIRE(ws_bytes >= need, GA_ERR_WORKSPACE, "workspace %zu < %zu bytes", ws_bytes, need);
  hipStream_t s = (hipStream_t)stream;
  double *part = static_cast<double *>(ws);
  hipLaunchKernelGGL(corr2cl_kernel, dim3(nwaves), dim3(64), 0, s, n, x, w, corr, nl, part);
  GA_LAUNCH_CHECK();
  hipLaunchKernelGGL(corr2cl_sum_kernel, dim3((nl + 63) / 64), dim3(256), 0, s, nl, nwaves, part,
                     cl);
  GA_LAUNCH_CHECK();
  return GA_OK;
}
