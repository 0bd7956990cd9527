// m2l_rot.hip — M2L of the runtime orders (p > TEMPLATED_MAX_P) by the
// rotation route of rotation.rs:106-435 (Dehnen 2014 A.6.1) on the FP64
// matrix cores: z-phase, x<->z swap, z-phase, swap, axial M2L along z, and
// the inverse rotation — O(p^3) per pair.
//
// Basis. With the coefficients scaled by g_n^m = sqrt((n-m)!(n+m)!) every swap
// matrix is orthogonal and, a swap being its own inverse, symmetric: one
// matrix D_n serves all four products, and the diagonals reduce to g on the
// source moments, 1/g on both sides of the axial sum and g on the result.
// Only m >= 0 is held (X_n^{-m} = (-1)^m conj X_n^m on every side), which
// splits D_n into a real-part matrix D[m][l] + (-1)^l D[m][-l] and an
// imaginary-part matrix D[m][l] - (-1)^l D[m][-l]. Half the entries of each
// vanish: in the real part m and l have the parity of their sum equal to
// n's, in the imaginary part opposite. So a product is four dense blocks of
// about (n/2 x n/2).
//
// Mapping. One block per chunk of a target's sources, NP pairs at a time: the
// pairs are the columns of v_mfma_f64_16x16x4 and a wave takes whole degrees.
// The instruction's output layout (row 4 i + lane / 16, column lane % 16 in
// register i) is its B-operand layout, so a product's result is multiplied by
// its phase in registers and is the next product's operand as it stands. The
// matrices are read in A-operand order (one coalesced 512-byte load per
// instruction, from L2, shared by the 16 pairs). Only the axial sum, which
// couples the degrees, goes through LDS.
//
// What bounds it at p = 24: vector instructions (about 41k per wave and batch
// of 16 pairs against 850 matrix instructions) and their latency at two waves
// a SIMD. Measured, 670k directed pairs at p = 24 (30k bodies, evaluation
// 145.4 -> 14.1 ms with this kernel alone, 9.4 with M2M and the others of later):
// the kernel before this one (one pair at a time per block, full-length matrices
// read from L2 for every pair) took 136.7 ms, this one 6.4 ms. W kept for every
// (k, m), half of it unread, held one block a CU: 7.6 ms.
// It replaces the per-pair naive convolution of 11 <= p < 20 too, and rounds no
// worse: against the 80-bit sum of the same moments and lists the far forces are
// off by 1e-16 in the median at p = 11 .. 19 (3e-16 by convolution), by 2.5e-15 at
// most in the 99th percentile on a clumped system (2.9e-15), and every degree's
// locals, in the norm of their power, by 2.2e-15 (2.0e-15).
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "common.h"
#include "internal.h"
#include "m2l_chunk.h"

namespace fmmh {

typedef double v4d __attribute__((ext_vector_type(4)));

constexpr int ROT_WAVES = 4;  // 8: 15.2 ms, 16: 16.9 ms against 14.0 ms (order 24, whole evaluation)
constexpr int ROT_T = 64 * ROT_WAVES;
constexpr int NP = 16;  // pairs per batch: the matrix instruction's columns

// Rows of one parity block, K-steps of 4, 16-row tiles (the same for both
// parities of a degree: the odd block is at most one row shorter).
__host__ __device__ constexpr int rot_rows(int n) { return n / 2 + 1; }
__host__ __device__ constexpr int rot_steps(int n) { return (rot_rows(n) + 3) / 4; }
__host__ __device__ constexpr int rot_tiles(int n) { return (rot_rows(n) + 15) / 16; }
// W, the axial sum's input: rows m = 0..min(k, p - k) of each degree k
// (n >= m and n + k <= p leave no others), degree after degree.
__host__ __device__ constexpr int rot_wrow(int p, int k) {
  const int h = p / 2 + 1;  // degrees 0..p/2 have k + 1 rows
  return k <= h ? k * (k + 1) / 2 : h * (h + 1) / 2 + (k - h) * (2 * p - k - h + 3) / 2;
}
// doubles of degree n in the A-operand table: [part][row parity][tile][step][lane]
__host__ __device__ constexpr int rot_words(int n) { return 4 * rot_tiles(n) * rot_steps(n) * 64; }

struct Cx {
  double re, im;
};
__device__ __forceinline__ Cx cxmul(Cx a, Cx b) {
  return Cx{fma(a.re, b.re, -(a.im * b.im)), fma(a.re, b.im, a.im * b.re)};
}
// b^q by squaring (error growth of log2 q products, not q).
__device__ __forceinline__ Cx cxpow(Cx b, int q) {
  Cx r = Cx{1.0, 0.0};
  while (q) {
    if (q & 1) r = cxmul(r, b);
    b = cxmul(b, b);
    q >>= 1;
  }
  return r;
}

// Row of register i of a parity block in the lane's group (sub = lane / 16).
__device__ __forceinline__ int rot_row(int po, int i, int sub) { return 2 * sub + (po + 8 * i); }

// One vector of a degree in operand layout: [row parity][register]; ST =
// rot_steps(n) registers per parity (register i: row 4 i + lane / 16).
template <int ST>
struct RotVec {
  double re[2][ST], im[2][ST];
};
// D_n in registers: [part][row parity][tile][step], both products of a side use it.
template <int ST>
struct RotMat {
  static constexpr int NT = (ST + 3) / 4;
  double a[4 * NT * ST];
  __device__ __forceinline__ void load(const double* __restrict__ tab, int lane) {
#pragma unroll
    for (int i = 0; i < 4 * NT * ST; i++) a[i] = tab[i * 64 + lane];
  }
};

// y = D_n x (both parts, both row parities). KP = n % 2: the input parity
// that feeds row parity po is po ^ KP in the real part, the other one in the
// imaginary part.
template <int ST, int KP>
__device__ __forceinline__ void rot_product(const RotMat<ST>& mat, const RotVec<ST>& x,
                                            RotVec<ST>& y) {
  constexpr int NT = RotMat<ST>::NT;
#pragma unroll
  for (int t = 0; t < NT; t++) {
    v4d acc[4] = {};
#pragma unroll
    for (int s = 0; s < ST; s++)
#pragma unroll
      for (int q = 0; q < 4; q++) {  // four independent chains
        const int po = q & 1;
        const double xi = q < 2 ? x.re[po ^ KP][s] : x.im[po ^ KP ^ 1][s];
        acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(mat.a[(q * NT + t) * ST + s], xi, acc[q], 0, 0, 0);
      }
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (4 * t + i < ST) (q < 2 ? y.re[q & 1] : y.im[q & 1])[4 * t + i] = acc[q][i];
  }
}

// x *= e (conjugated when CONJ) row by row, e from the pair's power table.
// Only the last register can hold rows past n (rot_steps(n) = n / 8 + 1);
// they are zero (the matrix rows are), so any finite factor serves there.
template <int ST, bool CONJ>
__device__ __forceinline__ void rot_phase(const Cx* __restrict__ e, int p, int sub, int col,
                                          RotVec<ST>& x) {
#pragma unroll
  for (int po = 0; po < 2; po++)
#pragma unroll
    for (int i = 0; i < ST; i++) {
      const int m = i < ST - 1 ? rot_row(po, i, sub) : min(rot_row(po, i, sub), p);
      const Cx f = e[m * NP + col];
      const double fi = CONJ ? -f.im : f.im;
      const double re = x.re[po][i], im = x.im[po][i];
      x.re[po][i] = fma(re, f.re, -(im * fi));
      x.im[po][i] = fma(re, fi, im * f.re);
    }
}

struct RotTables {
  const double* d;     // D_n in A-operand order
  const double* g;     // g_n^m, hpos order
  const double* ig;    // 1 / g_n^m
  const double* fact;  // j!
  uint32_t off[FMMH_MAX_P + 1];  // start of degree n in d
};

// Sums v[j] over the 16 lanes of each group; lane j of the group gets sum j.
__device__ __forceinline__ double reduce_scatter16(double (&v)[16], int lane) {
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) {
    const bool up = (lane & o) != 0;
#pragma unroll
    for (int i = 0; i < o; i++) {
      const double keep = up ? v[i + o] : v[i], send = up ? v[i] : v[i + o];
      v[i] = keep + __shfl_xor(send, o, 64);
    }
  }
  return v[0];
}

// Source side of degree k: moments -> rotated and scaled, conj(w)/g into LDS
// (rows m <= p - k: the axial sum reads no others).
template <int ST, int KP>
__device__ __forceinline__ void rot_source(int p, int k, const RotTables& rt,
                                           const cplx* __restrict__ ms, bool have, int lane,
                                           const Cx* __restrict__ ea, const Cx* __restrict__ eb,
                                           Cx* __restrict__ W) {
  const int col = lane & 15, sub = lane >> 4;
  RotMat<ST> mat;
  RotVec<ST> x, y;
  cplx v[2][ST];
  double gl[2][ST];
#pragma unroll
  for (int po = 0; po < 2; po++)
#pragma unroll
    for (int i = 0; i < ST; i++) {
      const int l = i < ST - 1 ? rot_row(po, i, sub) : min(rot_row(po, i, sub), k);
      v[po][i] = ms[hidx(k, l)];
      gl[po][i] = rt.g[hpos(k, l)];
    }
  mat.load(rt.d + rt.off[k], lane);
#pragma unroll
  for (int po = 0; po < 2; po++)
#pragma unroll
    for (int i = 0; i < ST; i++) {
      const int l = rot_row(po, i, sub);
      // conj(M) g e^{il(alpha - pi/2)}; absent pairs and rows are zero
      const bool ok = i < ST - 1 ? have : have && l <= k;
      const Cx f = ea[(i < ST - 1 ? l : min(l, k)) * NP + col];
      const double vr = ok ? v[po][i].re * gl[po][i] : 0.0, vi = ok ? v[po][i].im * gl[po][i] : 0.0;
      x.re[po][i] = fma(vr, f.re, vi * f.im);
      x.im[po][i] = fma(vr, f.im, -(vi * f.re));
    }
  rot_product<ST, KP>(mat, x, y);
  rot_phase<ST, false>(eb, p, sub, col, y);
  rot_product<ST, KP>(mat, y, x);
  const int mmax = min(k, p - k);
#pragma unroll
  for (int po = 0; po < 2; po++)
#pragma unroll
    for (int i = 0; i < ST; i++) {
      const int m = rot_row(po, i, sub);
      if (m <= mmax) {
        const double s = rt.ig[hpos(k, m)];
        W[(rot_wrow(p, k) + m) * NP + col] = Cx{x.re[po][i] * s, -x.im[po][i] * s};
      }
    }
}

// Axial sum of the rows of register I (m = 8 I .. 8 I + 7 over the lane groups):
// X_m = g_n^-1 sum_{k = m}^{p - n} conj(w_k^m) g_k^-1 a_{n+k}. The first
// eight degrees read rows past their own (they are other rows of W, finite)
// with a zero factor; rows past n end up with a zero scale.
template <int ST, int I>
__device__ __forceinline__ void rot_axial(int p, int n, int sub, int col, const RotTables& rt,
                                          const double* __restrict__ fa, const Cx* __restrict__ W,
                                          RotVec<ST>& x) {
  double re[2] = {0.0, 0.0}, im[2] = {0.0, 0.0};
  const double* a = fa + (n + 8 * I) * NP + col;
  const int k1 = min(8 * I + 8, p - n + 1);
  const Cx* w0 = W + (rot_wrow(p, 8 * I) + rot_row(0, I, sub)) * NP + col;
#pragma unroll 4
  for (int k = 8 * I; k < k1; k++) {
    const double av = *a;
#pragma unroll
    for (int po = 0; po < 2; po++) {
      const Cx w = w0[po * NP];
      const double f = rot_row(po, I, sub) <= k ? av : 0.0;
      re[po] = fma(w.re, f, re[po]);
      im[po] = fma(w.im, f, im[po]);
    }
    a += NP;
    w0 += (min(k, p - k) + 1) * NP;
  }
#pragma unroll 4
  for (int k = 8 * I + 8; k <= p - n; k++) {
    const double av = *a;
#pragma unroll
    for (int po = 0; po < 2; po++) {
      const Cx w = w0[po * NP];
      re[po] = fma(w.re, av, re[po]);
      im[po] = fma(w.im, av, im[po]);
    }
    a += NP;
    w0 += (min(k, p - k) + 1) * NP;
  }
#pragma unroll
  for (int po = 0; po < 2; po++) {
    const int m = rot_row(po, I, sub);
    const double s = m <= min(n, p - n) ? rt.ig[hpos(n, min(m, n))] : 0.0;
    x.re[po][I] = re[po] * s;
    x.im[po][I] = im[po] * s;
  }
}

// Target side of degree n: axial sum from LDS, inverse rotation, sum over the
// batch's pairs; lane (sub, j) of acc[t] holds component j of tile t.
template <int ST, int KP>
__device__ __forceinline__ void rot_target(int p, int n, const RotTables& rt, bool have, int lane,
                                           const Cx* __restrict__ ea, const Cx* __restrict__ eb,
                                           const double* __restrict__ fa, const Cx* __restrict__ W,
                                           double* acc) {
  const int col = lane & 15, sub = lane >> 4;
  RotMat<ST> mat;
  RotVec<ST> x, y;
  mat.load(rt.d + rt.off[n], lane);
  const int ax = rot_steps(min(n, p - n));  // rows m <= min(n, p - n)
#define FMMH_ROT_AXIAL(I)                                                                  \
  if constexpr (ST > I) {                                                                  \
    if (ax > I) {                                                                          \
      rot_axial<ST, I>(p, n, sub, col, rt, fa, W, x);                                      \
    } else {                                                                               \
      x.re[0][I] = x.im[0][I] = x.re[1][I] = x.im[1][I] = 0.0;                             \
    }                                                                                      \
  }
  FMMH_ROT_AXIAL(0)
  FMMH_ROT_AXIAL(1)
  FMMH_ROT_AXIAL(2)
  // min(n, p - n) <= 20: no rows beyond register 2
  if constexpr (ST > 3) {
#pragma unroll
    for (int i = 3; i < ST; i++) x.re[0][i] = x.im[0][i] = x.re[1][i] = x.im[1][i] = 0.0;
  }
#undef FMMH_ROT_AXIAL
  if (!have) {
#pragma unroll
    for (int po = 0; po < 2; po++)
#pragma unroll
      for (int i = 0; i < ST; i++) x.re[po][i] = x.im[po][i] = 0.0;
  }
  rot_product<ST, KP>(mat, x, y);
  rot_phase<ST, true>(eb, p, sub, col, y);
  rot_product<ST, KP>(mat, y, x);
  rot_phase<ST, false>(ea, p, sub, col, x);  // e^{im(alpha + pi/2)} = (-1)^m e^{im(alpha - pi/2)}
#pragma unroll
  for (int t = 0; t < RotMat<ST>::NT; t++) {
    double v[16];
#pragma unroll
    for (int po = 0; po < 2; po++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const bool in = 4 * t + i < ST;
        const double re = in ? x.re[po][in ? 4 * t + i : 0] : 0.0;
        const double im = in ? x.im[po][in ? 4 * t + i : 0] : 0.0;
        v[(po * 4 + i) * 2] = po ? -re : re;
        v[(po * 4 + i) * 2 + 1] = po ? -im : im;
      }
    acc[t] += reduce_scatter16(v, lane);
  }
}

// Calls f with ST = rot_steps(k) and KP = k % 2 as template arguments.
template <int STMAX, class F>
__device__ __forceinline__ void rot_dispatch(int k, F f) {
  const int st = rot_steps(k);
#define FMMH_ROT_CASE(S)                                                       \
  if (STMAX >= S && st == S) {                                                 \
    if (k & 1)                                                                 \
      f(std::integral_constant<int, (STMAX >= S ? S : 1)>{}, std::integral_constant<int, 1>{}); \
    else                                                                       \
      f(std::integral_constant<int, (STMAX >= S ? S : 1)>{}, std::integral_constant<int, 0>{}); \
  }
  FMMH_ROT_CASE(1)
  FMMH_ROT_CASE(2)
  FMMH_ROT_CASE(3)
  FMMH_ROT_CASE(4)
  FMMH_ROT_CASE(5)
  FMMH_ROT_CASE(6)
#undef FMMH_ROT_CASE
}

// LDS: W [rot_wrow(p, p + 1)][16], e^{im(alpha - pi/2)} and e^{im beta}
// [p+1][16], a_q [p+1][16]: 59 KB at p = 24 (two blocks a CU), 139 KB at p = 40.
__host__ __device__ constexpr size_t rot_lds_bytes(int p) {
  return (size_t)NP * ((size_t)rot_wrow(p, p + 1) * 16 + (size_t)(p + 1) * 40);
}

// Chunks c0, c0 + 1, ... (one per block) into part[0], part[1], ...
template <int STMAX>
__global__ void __launch_bounds__(ROT_T) k_m2l_rot(int p, uint32_t c0,
                                                  const M2lChunk* __restrict__ chunks,
                                                  const uint64_t* __restrict__ skeys,
                                                  uint64_t smask, DevCells c,
                                                  const cplx* __restrict__ moments, double soft2,
                                                  RotTables rt, cplx* __restrict__ part) {
  extern __shared__ Cx rot_lds[];
  // degrees a wave takes: p, p - 8, ... in snake order over the waves
  constexpr int PMAX = STMAX == 4 ? 31 : FMMH_MAX_P, NT = (STMAX + 3) / 4;
  constexpr int SL = (PMAX + ROT_WAVES) / ROT_WAVES;
  const int D = hdim(p), NH = hnpos(p);
  Cx* W = rot_lds;
  Cx* ea = W + rot_wrow(p, p + 1) * NP;
  Cx* eb = ea + (p + 1) * NP;
  double* fa = (double*)(eb + (p + 1) * NP);
  const uint32_t ci = xcd_block(blockIdx.x, gridDim.x);
  const M2lChunk ck = chunks[c0 + ci];
  const double tx = c.cx[ck.target], ty = c.cy[ck.target], tz = c.cz[ck.target];
  const int lane = threadIdx.x & 63, wave = wave_uniform((int)(threadIdx.x >> 6));
  double acc[SL][NT];
#pragma unroll
  for (int s = 0; s < SL; s++)
#pragma unroll
    for (int t = 0; t < NT; t++) acc[s][t] = 0.0;
  for (uint32_t b = ck.begin; b < ck.end; b += NP) {
    const int cnt = (int)min((uint32_t)NP, ck.end - b);
    __syncthreads();
    for (int i = threadIdx.x; i < NP * (p + 1); i += ROT_T) {
      const int pr = i % NP, q = i / NP;
      // pair geometry (rotation.rs:267-290): r = s_target - z_source
      const uint32_t src = (uint32_t)(skeys[b + min(pr, cnt - 1)] & smask);
      const double x = tx - c.cx[src], y = ty - c.cy[src], z = tz - c.cz[src];
      const double h2 = x * x + y * y, r2 = h2 + z * z;
      const double h = sqrt(h2), r = sqrt(r2);
      const double ih = h > 0.0 ? 1.0 / h : 0.0, ir = 1.0 / r;
      const double ca = h > 0.0 ? x * ih : 1.0, sa = y * ih;
      ea[i] = cxpow(Cx{sa, -ca}, q);
      eb[i] = cxpow(Cx{z * ir, h * ir}, q);
      // axial harmonic derivatives of the (softened) kernel: q! R^q / s^{2q+1}
      const double s2 = r2 + soft2;
      double v = 1.0 / sqrt(s2), t = r / s2;
      for (int e = q; e; e >>= 1) {
        if (e & 1) v *= t;
        t *= t;
      }
      fa[i] = rt.fact[q] * v;
    }
    __syncthreads();
    const int pr = lane & 15;
    const bool have = pr < cnt;  // absent columns hold zeros
    const uint32_t src = (uint32_t)(skeys[b + min(pr, cnt - 1)] & smask);
    const cplx* ms = moments + (size_t)src * D;
    for (int s = 0; s < SL; s++) {
      const int k = p - (s * ROT_WAVES + ((s & 1) ? ROT_WAVES - 1 - wave : wave));
      if (k < 0) continue;
      rot_dispatch<STMAX>(k, [&](auto st, auto kp) {
        rot_source<decltype(st)::value, decltype(kp)::value>(p, k, rt, ms, have, lane, ea, eb, W);
      });
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < SL; s++) {
      const int n = p - (s * ROT_WAVES + ((s & 1) ? ROT_WAVES - 1 - wave : wave));
      if (n < 0) continue;
      rot_dispatch<STMAX>(n, [&](auto st, auto kp) {
        rot_target<decltype(st)::value, decltype(kp)::value>(p, n, rt, have, lane, ea, eb, fa, W,
                                                                 acc[s]);
      });
    }
  }
  // acc[s][t], lane (sub, j): component j % 2 of row 4 (4 t + (j / 2) % 4) + sub
  // of parity j / 8
  double* out = (double*)(part + (size_t)ci * NH);
#pragma unroll
  for (int s = 0; s < SL; s++) {
    const int n = p - (s * ROT_WAVES + ((s & 1) ? ROT_WAVES - 1 - wave : wave));
    if (n < 0) continue;
#pragma unroll
    for (int t = 0; t < NT; t++) {
      const int j = lane & 15;
      const int m = (j >> 3) + 2 * (4 * (4 * t + ((j >> 1) & 3)) + (lane >> 4));
      if (m <= n) out[2 * hpos(n, m) + (j & 1)] = acc[s][t];
    }
  }
}

// locals[t] = g * sum over the target's chunk partials in chunk order, both
// signs of m; targets without sources get 0. part holds the chunks c0..c1-1: a
// target whose chunks go on past c1 keeps its sum so far, unscaled, in the
// m >= 0 entries, and the next slice adds to it, so the slices change no sum.
__global__ void __launch_bounds__(256) k_m2l_reduce_rot(int p, uint32_t nc, uint32_t c0, uint32_t c1,
                                                       const uint4* __restrict__ plan,
                                                       const cplx* __restrict__ part,
                                                       const double* __restrict__ g,
                                                       cplx* __restrict__ locals) {
  const int NH = hnpos(p);
  const uint32_t t = blockIdx.x;
  const uint32_t b = plan[t].x, e1 = plan[t + 1].x;
  const bool none = b == e1;  // no sources: written once, with the first slice
  if (none ? c0 > 0u : e1 <= c0 || b >= c1) return;
  const bool begun = !none && b < c0, done = none || e1 <= c1;
  cplx* out = locals + (size_t)t * hdim(p);
  for (int e = threadIdx.x; e < NH; e += 256) {
    int n = (int)((sqrt(8.0 * e + 1.0) - 1.0) * 0.5);
    while (n * (n + 1) / 2 > e) n--;
    while ((n + 1) * (n + 2) / 2 <= e) n++;
    const int m = e - n * (n + 1) / 2;
    cplx s = begun ? out[hidx(n, m)] : cplx{0.0, 0.0};
    for (uint32_t k = max(b, c0); k < min(e1, c1); k++) {
      const cplx v = part[(size_t)(k - c0) * NH + e];
      s.re += v.re;
      s.im += v.im;
    }
    if (!done) {
      out[hidx(n, m)] = s;
      continue;
    }
    s.re *= g[e];
    s.im *= g[e];
    out[hidx(n, m)] = s;
    if (m > 0) {
      const double sg = (m & 1) ? -1.0 : 1.0;
      out[hidx(n, -m)] = cplx{sg * s.re, -sg * s.im};
    }
  }
}

// ------------------------------------------------------------- host side
// Swap matrices B_n of Dehnen 2014 eq. 63 (rotation.rs:137-211), taken to the
// orthogonal basis, folded to m >= 0, split by parity and laid out as
// A operands; then g, 1/g and the factorials. Built once per context.
void rot_tables_host(int p, std::vector<double>& tab, std::vector<uint32_t>& off) {
  auto boff = [](int n) { return n == 0 ? 0 : n * (4 * n * n - 1) / 3; };
  std::vector<double> sw((size_t)(p + 1) * (4 * p * p + 8 * p + 3) / 3, 0.0);
  sw[0] = 1.0;
  for (int n = 1; n <= p; n++) {
    const int nb = 2 * n + 1, pnb = 2 * n - 1, o = boff(n), po = boff(n - 1);
    // entry (M, L) of B_{n-1}, zero outside |M|,|L| <= n-1
    auto prev = [&](int M, int L) -> double {
      if (M < -(n - 1) || M > n - 1 || L < -(n - 1) || L > n - 1) return 0.0;
      return sw[po + (M + n - 1) * pnb + (L + n - 1)];
    };
    for (int M = -n; M <= n; M++)
      for (int L = -n; L <= n; L++) {
        double v;
        if (M > -n && M < n)
          v = (prev(M, L - 1) - prev(M, L + 1)) * 0.5;
        else if (M == n)
          v = (prev(n - 1, L - 1) + prev(n - 1, L + 1) + 2.0 * prev(n - 1, L)) * 0.5;
        else
          v = (prev(1 - n, L - 1) + prev(1 - n, L + 1) - 2.0 * prev(1 - n, L)) * 0.5;
        sw[o + (M + n) * nb + (L + n)] = v;
      }
  }
  std::vector<double> f(2 * p + 1, 1.0);
  for (size_t i = 1; i < f.size(); i++) f[i] = f[i - 1] * (double)i;
  auto g = [&](int n, int m) { return std::sqrt(f[n - m]) * std::sqrt(f[n + m]); };
  off.assign(FMMH_MAX_P + 1, 0);
  size_t words = 0;
  for (int n = 0; n <= p; n++) {
    off[n] = (uint32_t)words;
    words += rot_words(n);
  }
  const int NH = hnpos(p);
  tab.assign(words + 2 * (size_t)NH + p + 1, 0.0);
  for (int n = 0; n <= p; n++) {
    const int nb = 2 * n + 1, tiles = rot_tiles(n), steps = rot_steps(n);
    const double* B = sw.data() + boff(n);
    for (int part = 0; part < 2; part++)
      for (int po = 0; po < 2; po++)
        for (int t = 0; t < tiles; t++)
          for (int s = 0; s < steps; s++)
            for (int lane = 0; lane < 64; lane++) {
              const int m = po + 2 * (16 * t + (lane & 15));
              const int pi = po ^ (n & 1) ^ part;
              const int l = pi + 2 * (4 * s + (lane >> 4));
              double v = 0.0;
              if (m <= n && l <= n && !(part == 1 && (l == 0 || m == 0))) {
                const double sg = ((l & 1) != 0) != (part == 1) ? -1.0 : 1.0;
                v = B[(m + n) * nb + (l + n)];
                if (l > 0) v += sg * B[(m + n) * nb + (n - l)];
                v *= g(n, l) / g(n, m);
              }
              tab[off[n] + (size_t)(((part * 2 + po) * tiles + t) * steps + s) * 64 + lane] = v;
            }
  }
  for (int n = 0; n <= p; n++)
    for (int m = 0; m <= n; m++) {
      tab[words + hpos(n, m)] = g(n, m);
      tab[words + NH + hpos(n, m)] = 1.0 / g(n, m);
    }
  for (int j = 0; j <= p; j++) tab[words + 2 * (size_t)NH + j] = f[j];
}

static RotTables rot_view(int p, const double* tab, const std::vector<uint32_t>& off) {
  RotTables r;
  const size_t words = (size_t)off[p] + rot_words(p);
  r.d = tab;
  r.g = tab + words;
  r.ig = r.g + hnpos(p);
  r.fact = r.ig + hnpos(p);
  std::copy(off.begin(), off.end(), r.off);
  return r;
}

template <int STMAX>
static hipError_t rot_t(int p, const M2lChunk* ck, uint32_t c0, uint32_t nchunks,
                        const uint64_t* skeys, uint64_t smask, DevCells c, const cplx* moments, double soft2,
                        const RotTables& rt, cplx* part, hipStream_t s) {
  const size_t lds = rot_lds_bytes(p);
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_m2l_rot<STMAX>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_m2l_rot<STMAX>), dim3(nchunks), dim3(ROT_T), lds, s, p, c0, ck, skeys,
                     smask, c, moments, soft2, rt, part);
  return hipSuccess;
}

hipError_t launch_m2l_rot(int p, uint32_t nc, const void* chunks, uint32_t nchunks,
                          const uint4* plan, const uint64_t* skeys, int sbits, DevCells c,
                          const cplx* moments, double soft2, const double* tab,
                          const std::vector<uint32_t>& off, cplx* part, size_t slice, cplx* locals,
                          hipStream_t s) {
  const uint64_t smask = (1ull << sbits) - 1ull;
  const RotTables rt = rot_view(p, tab, off);
  const M2lChunk* ck = (const M2lChunk*)chunks;
  if (nc == 0) return hipSuccess;
  uint32_t c0 = 0;
  do {  // once without chunks: every local is 0
    const uint32_t m = (uint32_t)std::min<size_t>(slice, nchunks - c0);
    if (m) {
      const hipError_t e =
          p <= 31 ? rot_t<4>(p, ck, c0, m, skeys, smask, c, moments, soft2, rt, part, s)
                  : rot_t<6>(p, ck, c0, m, skeys, smask, c, moments, soft2, rt, part, s);
      if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k_m2l_reduce_rot, dim3(nc), dim3(256), 0, s, p, nc, c0, c0 + m, plan, part,
                       rt.g, locals);
    c0 += m;
  } while (c0 < nchunks);
  return hipSuccess;
}

}  // namespace fmmh
