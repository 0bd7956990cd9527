// generic_far.hip — L2L and L2P for any expansion order (runtime p), used
// when p exceeds the register-resident templated kernels (the M2L of those
// orders is m2l_rot.hip's).
#include "common.h"
#include "internal.h"

namespace fmmh {

__device__ __forceinline__ int deg_of(int e) {
  int n = (int)sqrt((double)e);
  while (n * n > e) n--;
  while ((n + 1) * (n + 1) <= e) n++;
  return n;
}

__device__ __forceinline__ cplx cmul_(cplx a, cplx b) {
  return cplx{a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}

constexpr int GEN_T = 256;

// ------------------------------------------------------------- L2L, L2P
__device__ void upsilon_column_far(int p, double x, double y, double z, int m, cplx* tab) {
  const double r2 = x * x + y * y + z * z;
  cplx u = cplx{1.0, 0.0};
  for (int j = 1; j <= m; j++) {
    const double f = 1.0 / (double)(2 * j);
    u = cmul_(cplx{x * f, y * f}, u);
  }
  const double sgn = (m & 1) ? -1.0 : 1.0;
  cplx u1 = u, u2 = cplx{0.0, 0.0};
  for (int n = m; n <= p; n++) {
    cplx un;
    if (n == m) {
      un = u;
    } else {
      const double a = (double)(2 * n - 1) * z;
      const double ic = 1.0 / (double)(n * n - m * m);
      const double bb = (n >= m + 2) ? r2 : 0.0;
      un = cplx{(a * u1.re - bb * u2.re) * ic, (a * u1.im - bb * u2.im) * ic};
      u2 = u1;
      u1 = un;
    }
    tab[hidx(n, m)] = un;
    if (m > 0) tab[hidx(n, -m)] = cplx{sgn * un.re, -sgn * un.im};
  }
}

__global__ void __launch_bounds__(GEN_T) k_l2l_gen(int p, const uint32_t* __restrict__ cells,
                                                  DevCells c, cplx* __restrict__ locals) {
  extern __shared__ cplx u[];
  const int D = hdim(p);
  const uint32_t ch = cells[blockIdx.x];
  const int32_t pa = c.parent[ch];
  if (pa < 0) return;
  for (int m = threadIdx.x; m <= p; m += GEN_T)
    upsilon_column_far(p, c.cx[pa] - c.cx[ch], c.cy[pa] - c.cy[ch], c.cz[pa] - c.cz[ch], m, u);
  __syncthreads();
  const cplx* fp = locals + (size_t)pa * D;
  cplx* fc = locals + (size_t)ch * D;
  for (int e = threadIdx.x; e < D; e += GEN_T) {
    const int n = deg_of(e), m = e - n * (n + 1);
    double sr = 0.0, si = 0.0;
    for (int k = 0; k <= p - n; k++)
      for (int l = -k; l <= k; l++) {
        const cplx a = u[hidx(k, l)], b = fp[hidx(n + k, m + l)];
        sr = fma(a.re, b.re, fma(a.im, b.im, sr));
        si = fma(a.re, b.im, fma(-a.im, b.re, si));
      }
    fc[e].re += sr;
    fc[e].im += si;
  }
}

constexpr int GEN_PMAX = FMMH_MAX_P;

__global__ void __launch_bounds__(64) k_l2p_gen(int p, const uint32_t* __restrict__ leaf_ids,
                                               DevCells c, DevBodies b,
                                               const cplx* __restrict__ locals,
                                               const double* __restrict__ lap,
                                               double4* __restrict__ far) {
  extern __shared__ cplx F[];
  const int D = hdim(p);
  const uint32_t leaf = leaf_ids[blockIdx.x];
  for (int e = threadIdx.x; e < D; e += 64) F[e] = locals[(size_t)leaf * D + e];
  __syncthreads();
  const double cxl = c.cx[leaf], cyl = c.cy[leaf], czl = c.cz[leaf];
  const uint32_t f0 = c.first[leaf], e0 = f0 + c.count[leaf];
  for (uint32_t k = f0 + threadIdx.x; k < e0; k += 64) {
    const double x = cxl - b.x[k], y = cyl - b.y[k], z = czl - b.z[k];
    const double r2 = x * x + y * y + z * z;
    cplx U[GEN_PMAX + 1], U1[GEN_PMAX + 1], U2[GEN_PMAX + 1];
    double p00 = 0.0, p11r = 0.0, p11i = 0.0, p10r = 0.0;
    for (int kk = 0; kk <= p; kk++) {
      if (kk == 0) {
        U[0] = cplx{1.0, 0.0};
      } else {
        const double a = (double)(2 * kk - 1) * z;
        for (int q = 0; q < kk; q++) {
          const double ic = 1.0 / (double)(kk * kk - q * q);
          const double bb = (q + 2 <= kk) ? r2 : 0.0;
          const cplx u2 = (q + 2 <= kk) ? U2[q] : cplx{0.0, 0.0};
          U[q] = cplx{(a * U1[q].re - bb * u2.re) * ic, (a * U1[q].im - bb * u2.im) * ic};
        }
        const double f = 1.0 / (double)(2 * kk);
        U[kk] = cmul_(cplx{x * f, y * f}, U1[kk - 1]);
      }
      for (int l = -kk; l <= kk; l++) {
        double ar, ai;  // conj(Y_k^l)
        if (l >= 0) {
          ar = U[l].re;
          ai = -U[l].im;
        } else {
          const double sg = ((-l) & 1) ? -1.0 : 1.0;
          ar = sg * U[-l].re;
          ai = sg * U[-l].im;
        }
        const cplx f00 = F[hidx(kk, l)];
        p00 += ar * f00.re - ai * f00.im;
        if (kk + 1 <= p) {
          const cplx f11 = F[hidx(kk + 1, l + 1)], f10 = F[hidx(kk + 1, l)];
          p11r += ar * f11.re - ai * f11.im;
          p11i += ar * f11.im + ai * f11.re;
          p10r += ar * f10.re - ai * f10.im;
        }
      }
      for (int q = 0; q <= kk; q++) {
        U2[q] = U1[q];
        U1[q] = U[q];
      }
    }
    double4 o = make_double4(-p11r, -p11i, -p10r, p00);
    if (lap) l2p_trace_walk(lap, c.parent, c.cx, c.cy, c.cz, leaf, b.x[k], b.y[k], b.z[k], o);
    far[k] = o;
  }
}

void launch_l2l_gen(int p, const uint32_t* cells, uint32_t cnt, DevCells c, cplx* locals,
                    hipStream_t s) {
  if (cnt == 0) return;
  hipLaunchKernelGGL(k_l2l_gen, dim3(cnt), dim3(GEN_T), (size_t)hdim(p) * sizeof(cplx), s, p,
                     cells, c, locals);
}

void launch_l2p_gen(int p, const uint32_t* leaf_ids, uint32_t nleaves, DevCells c, DevBodies b,
                    const cplx* locals, const double* lap, double4* far, hipStream_t s) {
  if (nleaves == 0) return;
  hipLaunchKernelGGL(k_l2p_gen, dim3(nleaves), dim3(64), (size_t)hdim(p) * sizeof(cplx), s, p,
                     leaf_ids, c, b, locals, lap, far);
}

}  // namespace fmmh
