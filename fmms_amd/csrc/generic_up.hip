// generic_up.hip — P2M and M2M for any expansion order (runtime p), used
// when p exceeds the register-resident templated kernels (compiled
// -ffp-contract=off). Results are bit-identical to the reference
// (moments.rs:30-90): the same recursions and the same summation order, each
// entry owned by one thread.
#include <algorithm>

#include "common.h"
#include "internal.h"

namespace fmmh {

// Column m (both signs) of Upsilon(r) into tab (harmonic.rs:141-173).
__device__ void upsilon_column_gen(int p, double x, double y, double z, int m, cplx* tab) {
  const double r2 = x * x + y * y + z * z;
  cplx u = cplx{1.0, 0.0};
  for (int j = 1; j <= m; j++) u = cmul(cscale(cplx{x, y}, 1.0 / (double)(2 * j)), u);
  const double sgn = (m % 2 == 0) ? 1.0 : -1.0;
  cplx u1 = u, u2 = cz();
  for (int n = m; n <= p; n++) {
    cplx un;
    if (n == m) {
      un = u;
    } else {
      const double a = (double)(2 * n - 1) * z;
      const double c = (double)(n * n - m * m);
      const cplx p2 = (n >= m + 2) ? u2 : cz();
      un = cscale(csub(cscale(u1, a), cscale(p2, r2)), 1.0 / c);
      u2 = u1;
      u1 = un;
    }
    tab[hidx(n, m)] = un;
    if (m > 0) tab[hidx(n, -m)] = cscale(cconj(un), sgn);
  }
}

// P2M, one thread per (leaf, m), a few leaves per block: the column of each
// body's Upsilon is recomputed in order and added to the entries (n, +-m) the
// thread owns, which stay in LDS until the leaf is done (adding them straight
// into the moments array was a dependent memory round trip per entry and body),
// with the recursion's reciprocals from a table.
constexpr int P2MG_T = 256;

__global__ void __launch_bounds__(P2MG_T) k_p2m_gen(int p, int nlf,
                                                   const uint32_t* __restrict__ leaf_ids,
                                                   uint32_t nleaves, DevCells c, DevBodies b,
                                                   cplx* __restrict__ moments) {
  extern __shared__ cplx gsh[];
  const int D = hdim(p);
  cplx* acc = gsh;                        // [nlf][D]
  double* inv = (double*)(acc + nlf * D);  // 1 / (n^2 - m^2), hpos; entry (n, n): 1 / (2n)
  const uint32_t l0 = blockIdx.x * (uint32_t)nlf;
  const int nl = (int)min((uint32_t)nlf, nleaves - l0);
  for (int i = threadIdx.x; i < hnpos(p); i += P2MG_T) {
    int n = 0;
    while ((n + 1) * (n + 2) / 2 <= i) n++;
    const int m = i - n * (n + 1) / 2;
    inv[i] = m == n ? 1.0 / (double)(2 * n) : 1.0 / (double)(n * n - m * m);
  }
  for (int i = threadIdx.x; i < nl * D; i += P2MG_T) acc[i] = cz();
  __syncthreads();
  const int li = threadIdx.x / (p + 1), m = threadIdx.x - li * (p + 1);
  if (li < nl) {
    const uint32_t id = leaf_ids[l0 + li];
    const double zx = c.cx[id], zy = c.cy[id], zz = c.cz[id];
    cplx* out = acc + li * D;
    const double sgn = (m % 2 == 0) ? 1.0 : -1.0;
    const uint32_t f = c.first[id], e = f + c.count[id];
    for (uint32_t k = f; k < e; k++) {
      const double4 q = b.xyzm[k];
      const double x = q.x - zx, y = q.y - zy, z = q.z - zz;
      const double r2 = x * x + y * y + z * z;
      const double ms = q.w;
      cplx u = cplx{1.0, 0.0};
      for (int j = 1; j <= m; j++) u = cmul(cscale(cplx{x, y}, inv[hpos(j, j)]), u);
      cplx u1 = u, u2 = cz();
      for (int n = m; n <= p; n++) {
        cplx un;
        if (n == m) {
          un = u;
        } else {
          const double a = (double)(2 * n - 1) * z;
          const cplx p2 = (n >= m + 2) ? u2 : cz();
          un = cscale(csub(cscale(u1, a), cscale(p2, r2)), inv[hpos(n, m)]);
          u2 = u1;
          u1 = un;
        }
        out[hidx(n, m)] = cadd(out[hidx(n, m)], cscale(un, ms));
        if (m > 0) out[hidx(n, -m)] = cadd(out[hidx(n, -m)], cscale(cscale(cconj(un), sgn), ms));
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < nl * D; i += P2MG_T) {
    const int lf = i / D;
    moments[(size_t)leaf_ids[l0 + lf] * D + (i - lf * D)] = acc[i];
  }
}

// M2M: the children of a cell in passes of nch, their Upsilon tables and
// moments staged in LDS, one thread per (child, output entry). A thread's sum
// is its child's part of one entry, from zero, in the reference's (k, l)
// order; the parts are then added to the entry in octant order, so every
// entry is the reference's sum bit for bit. A level near the root has few
// cells, so a cell's entries are cut over blockIdx.y (slices of M2MG_T / nch).
// One block per cell that took the children one after another, reading their
// moments from memory term by term, spent 530 us a level at p = 24 (30k
// bodies, eight levels: 4.25 ms); the latency of one entry's serial sum (up
// to 313 terms) now bounds it.
constexpr int M2MG_T = 1024;

__global__ void __launch_bounds__(M2MG_T) k_m2m_gen(int p, int nch,
                                                   const uint32_t* __restrict__ cells, DevCells c,
                                                   cplx* __restrict__ moments) {
  extern __shared__ cplx gsh[];
  const int D = hdim(p);
  const uint32_t id = cells[blockIdx.x];
  if (c.leaf[id]) return;
  cplx* u = gsh;              // [nch][D]
  cplx* mo = gsh + nch * D;   // [nch][D]
  cplx* part = mo + nch * D;  // [M2MG_T]
  const double zx = c.cx[id], zy = c.cy[id], zz = c.cz[id];
  const int32_t* ch = c.children + (size_t)id * 8;
  const int per = M2MG_T / nch;
  const int g = threadIdx.x / per, j = threadIdx.x - g * per;
  const int e = blockIdx.y * per + j;
  int n = 0;
  while ((n + 1) * (n + 1) <= e) n++;
  const int m = e - n * (n + 1);
  cplx out = cz();
  for (int o0 = 0; o0 < 8; o0 += nch) {
    __syncthreads();
    for (int i = threadIdx.x; i < nch * (p + 1); i += M2MG_T) {
      const int o = i / (p + 1), q = ch[o0 + o];
      if (q >= 0)
        upsilon_column_gen(p, c.cx[q] - zx, c.cy[q] - zy, c.cz[q] - zz, i - o * (p + 1), u + o * D);
    }
    for (int i = threadIdx.x; i < nch * D; i += M2MG_T) {
      const int o = i / D, q = ch[o0 + o];
      if (q >= 0) mo[i] = moments[(size_t)q * D + (i - o * D)];
    }
    __syncthreads();
    if (e < D && ch[o0 + g] >= 0) {
      const cplx* uc = u + g * D;
      const cplx* mc = mo + g * D;
      cplx s = cz();
      for (int k = 0; k <= n; k++) {
        const int nk = n - k;
        const int lo = max(-k, m - nk), hi = min(k, m + nk);
        for (int l = lo; l <= hi; l++) s = cadd(s, cmul(uc[hidx(k, l)], mc[hidx(nk, m - l)]));
      }
      part[threadIdx.x] = s;
    }
    __syncthreads();
    if (g == 0 && e < D)
      for (int o = 0; o < nch; o++)
        if (ch[o0 + o] >= 0) out = cadd(out, part[o * per + j]);
  }
  if (g == 0 && e < D) moments[(size_t)id * D + e] = out;
}

void launch_p2m_gen(int p, const uint32_t* leaf_ids, uint32_t nleaves, DevCells c, DevBodies b,
                    cplx* moments, hipStream_t s) {
  if (nleaves == 0) return;
  // leaves per block: one thread per column, at most about 60 KB of accumulators
  const size_t D = (size_t)hdim(p);
  const int nlf = std::max(1, std::min(P2MG_T / (p + 1), (int)(60 * 1024 / (D * sizeof(cplx)))));
  const size_t lds = (size_t)nlf * D * sizeof(cplx) + (size_t)hnpos(p) * sizeof(double);
  hipLaunchKernelGGL(k_p2m_gen, dim3((nleaves + nlf - 1) / nlf), dim3(P2MG_T), lds, s, p, nlf,
                     leaf_ids, nleaves, c, b, moments);
}

hipError_t launch_m2m_gen(int p, const uint32_t* cells, uint32_t cnt, DevCells c, cplx* moments,
                          hipStream_t s) {
  if (cnt == 0) return hipSuccess;
  // children per pass: as many as leave tables and moments within 150 KB (4 up to p = 31)
  const size_t D = (size_t)hdim(p);
  int nch = 8;
  while (nch > 1 && (2 * (size_t)nch * D + M2MG_T) * sizeof(cplx) > 150 * 1024) nch /= 2;
  const size_t lds = (2 * (size_t)nch * D + M2MG_T) * sizeof(cplx);
  const int per = M2MG_T / nch;
  const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_m2m_gen),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(k_m2m_gen, dim3(cnt, (D + per - 1) / per), dim3(M2MG_T), lds, s, p, nch, cells,
                     c, moments);
  return hipSuccess;
}

}  // namespace fmmh
