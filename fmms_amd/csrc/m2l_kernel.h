// m2l_kernel.h — far-field M2L on gfx950 (FP64, and FP32 in the mixed form;
// FMA contraction on).
//
// F_B[n,m] += sum_{k<=p-n} sum_{|l|<=k} conj(M_A[k,l]) Theta_{n+k}^{m+l}(s_B - z_A)
// (crates/fmm translate.rs:47-136). The reference evaluates each accepted
// pair mutually into both cells' locals; here the directed entries are
// grouped by target (sorted (target, source) keys), so every local is
// written by exactly one reduction, in a fixed order, with no atomics.
//
// Mapping: one thread per chunk of at most m2l_chunk sources of one target. Per
// source the thread streams Theta degree by degree (three-term recursion,
// two previous columns in registers) against the source multipole held in
// registers, accumulating the m >= 0 half of F (the m < 0 half follows from
// F_n^{-m} = (-1)^m conj(F_n^m)). P is a template parameter so every index
// is static and all operands live in registers. Partials of the chunks of a
// target are then summed in chunk order by k_m2l_reduce.
#pragma once
#include "common.h"
#include "internal.h"
#include "m2l_chunk.h"

namespace fmmh {

// The chunk length (sources per thread) is a context parameter,
// fmmh_tuning.m2l_chunk (default 32).

__device__ __forceinline__ void cmac(cplxf& f, float ar, float ai, float br, float bi) {
  f.re = fmaf(ar, br, f.re);
  f.re = fmaf(-ai, bi, f.re);
  f.im = fmaf(ar, bi, f.im);
  f.im = fmaf(ai, br, f.im);
}

// f += a * (br + i bi) for a real factor a.
__device__ __forceinline__ void cmac_real(cplxf& f, float a, float br, float bi) {
  f.re = fmaf(a, br, f.re);
  f.im = fmaf(a, bi, f.im);
}

__device__ __forceinline__ double m2l_rsqrt(double x) { return rsqrt(x); }
__device__ __forceinline__ float m2l_rsqrt(float x) {
  const float y = rsqrtf(x);
  return y * fmaf(-0.5f * x * y, y, 1.5f);  // one Newton step on the hardware estimate
}

// FP32 (mixed form): F (m>=0 half, hpos layout) += M2L of source multipole M
// (m>=0 half) at r, term by term (softening as in m2l_accumulate64). on:
// whether the lane has a pair (else Theta is 0 and nothing is added); mid()
// runs before the products of degree MID.
template <int P, int H, int MID, typename R, typename C, class Mid>
__device__ __forceinline__ void m2l_accumulate(bool on, R x, R y, R z, R soft2, const C* M, C* F,
                                               Mid mid) {
  const R rr2 = x * x + y * y + z * z;
  const R r2 = rr2 + soft2;
  const R ir = m2l_rsqrt(r2);
  const R ir2 = ir * ir;
  const R ks = soft2 > R(0) ? rr2 * ir2 : R(1);
  C T[P + 1], T1[P + 1], T2[P + 1];
#pragma unroll
  for (int s = 0; s <= P; s++) {
    // Theta_s^q, q = 0..s (harmonic.rs:91-129 recursion, Dehnen eq. 52/54)
    if (s == 0) {
      T[0] = C{on ? ir : R(0), R(0)};
    } else {
      const R a = (R)(2 * s - 1) * z;
#pragma unroll
      for (int q = 0; q <= P; q++) {
        if (q > s) continue;
        if (q + 2 <= s) {
          const R bq = (R)((s - 1) * (s - 1) - q * q) * ks;
          T[q].re = (a * T1[q].re - bq * T2[q].re) * ir2;
          T[q].im = q == 0 ? R(0) : (a * T1[q].im - bq * T2[q].im) * ir2;  // Theta_s^0 is real
        } else if (q == s - 1) {
          T[q].re = a * T1[q].re * ir2;
          T[q].im = q == 0 ? R(0) : a * T1[q].im * ir2;
        } else {  // q == s: (2s-1)(x+iy)/r^2 * Theta_{s-1}^{s-1}
          const R f = (R)(2 * s - 1) * ir2;
          const R wr = x * f, wi = y * f;
          T[q].re = wr * T1[s - 1].re - wi * T1[s - 1].im;
          T[q].im = wr * T1[s - 1].im + wi * T1[s - 1].re;
        }
      }
    }
    if (s == MID) mid(T[s].re);
    // all terms with n + k == s
#pragma unroll
    for (int n = 0; n <= P; n++) {
      if (n > s) continue;
      if (H != 2 && (n & 1) != H) continue;
      const int k = s - n;
#pragma unroll
      for (int m = 0; m <= P; m++) {
        if (m > n) continue;
#pragma unroll
        for (int l = -P; l <= P; l++) {
          if (l < -k || l > k) continue;
          // conj(M_k^l): l >= 0 direct; l < 0 via M_k^l = (-1)^l conj(M_k^{-l})
          R ar, ai;
          if (l >= 0) {
            ar = M[hpos(k, l)].re;
            ai = -M[hpos(k, l)].im;
          } else {
            const R sg = ((-l) & 1) ? R(-1) : R(1);
            ar = sg * M[hpos(k, -l)].re;
            ai = sg * M[hpos(k, -l)].im;
          }
          const int q = m + l;
          R br, bi;
          if (q >= 0) {
            br = T[q].re;
            bi = T[q].im;
          } else {
            const R sg = ((-q) & 1) ? R(-1) : R(1);
            br = sg * T[-q].re;
            bi = -sg * T[-q].im;
          }
          // Theta_s^0 is real (its imaginary part is an exact zero), and so is
          // M_k^0 up to rounding residue in cells built by M2M: those terms
          // take the real-factor product (2 FMAs instead of 4).
          if (q == 0) {
            cmac_real(F[hpos(n, m)], br, ar, ai);  // (ar + i ai) * br
          } else if (l == 0) {
            cmac_real(F[hpos(n, m)], ar, br, bi);  // ar * (br + i bi)
          } else {
            cmac(F[hpos(n, m)], ar, ai, br, bi);
          }
        }
      }
    }
#pragma unroll
    for (int q = 0; q <= P; q++) {
      T2[q] = T1[q];
      T1[q] = T[q];
    }
  }
}

// ------------------------------------------------------------------- FP64
// Real-valued layout of an m >= 0 half: (P+1)^2 doubles, degree n at n^2:
// X_n^0 (real), then (re, im) of X_n^m, m = 1..n.
__host__ __device__ constexpr int rre(int n, int m) { return n * n + (m ? 2 * m - 1 : 0); }
__host__ __device__ constexpr int rim(int n, int m) { return n * n + 2 * m; }

// F += M2L of source multipole M at r, both in the real layout, with the
// terms of +l and -l taken together. With M_k^l = a + ib, M_k^{-l} =
// (-1)^l conj(M_k^l) and
//   S = Theta^{m+l} + (-1)^l Theta^{m-l},  D = Theta^{m+l} - (-1)^l Theta^{m-l},
// the two terms of F_n^m are a S - i b D: four multiply-adds instead of
// eight, and S, D depend on n + k, m and l alone, so one set serves every
// (n, k) of a degree, and the set of (m, l) serves (l, m) with the imaginary
// parts exchanged. F_n^0 is real: 2 Re(conj(M_k^l) Theta^l), accumulated
// halved (the caller doubles it). At P = 7: 876 multiply-adds and 112 adds
// for the sums, against 2100 term by term.
// H, NC: only the degrees n of F with n % NC == H (one of the NC waves that share
// a chunk's pairs; NC = 1: all).
// on: whether the lane has a pair (else Theta is 0 and nothing is added).
// load(s) runs before the products of degree s, which read the degrees s - n of
// M; mid() between the degrees s = 0..2 and the others.
template <int P, int H, int NC, class Load, class Mid>
__device__ __forceinline__ void m2l_accumulate64(bool on, double x, double y, double z,
                                                 double soft2, const double* M, double* F,
                                                 Load load, Mid mid) {
  // Softening: the harmonic derivatives of the Plummer kernel are those of
  // 1/r times (r/s)^{2n+1}, s^2 = r^2 + eps^2; in the recursion that is
  // 1/r^2 -> 1/s^2 and the (n-2) term scaled by r^2/s^2 (soft2 = 0: 1).
  const double rr2 = x * x + y * y + z * z;
  const double r2 = rr2 + soft2;
  const double ir = m2l_rsqrt(r2);
  const double ir2 = ir * ir;
  const double kir = soft2 > 0.0 ? rr2 * ir2 * ir2 : ir2;
  const double xs = x * ir2, ys = y * ir2, zs = z * ir2;
  double Tr[P + 1], Ti[P + 1], Ar[P + 1], Ai[P + 1], Br[P + 1], Bi[P + 1];  // Theta_s, _{s-1}, _{s-2}
#pragma unroll
  for (int s = 0; s <= P; s++) {
    // Theta_s^q, q = 0..s (harmonic.rs:91-129 recursion, Dehnen eq. 52/54)
    if (s == 0) {
      Tr[0] = on ? ir : 0.0;
      Ti[0] = 0.0;
    } else {
      const double a = (double)(2 * s - 1) * zs;
#pragma unroll
      for (int q = 0; q <= P; q++) {
        if (q > s) continue;
        if (q + 2 <= s) {
          const double bq = (double)((s - 1) * (s - 1) - q * q) * kir;
          Tr[q] = fma(a, Ar[q], -(bq * Br[q]));
          Ti[q] = q == 0 ? 0.0 : fma(a, Ai[q], -(bq * Bi[q]));
        } else if (q == s - 1) {
          Tr[q] = a * Ar[q];
          Ti[q] = q == 0 ? 0.0 : a * Ai[q];
        } else {  // q == s: (2s-1)(x+iy)/r^2 * Theta_{s-1}^{s-1}
          const double wr = (double)(2 * s - 1) * xs, wi = (double)(2 * s - 1) * ys;
          Tr[q] = s == 1 ? wr * Ar[0] : fma(wr, Ar[s - 1], -(wi * Ai[s - 1]));
          Ti[q] = s == 1 ? wi * Ar[0] : fma(wr, Ai[s - 1], wi * Ar[s - 1]);
        }
      }
    }
    load(s);
    // all terms with n + k == s: l = 0, and m = 0
    const double t0 = 0.5 * Tr[0];
#pragma unroll
    for (int n = 0; n <= P; n++) {
      if (n > s) continue;
      if (n % NC != H) continue;
      const int k = s - n;
      F[rre(n, 0)] = fma(M[rre(k, 0)], t0, F[rre(n, 0)]);
#pragma unroll
      for (int l = 1; l <= P; l++) {
        if (l > k) continue;
        F[rre(n, 0)] = fma(M[rre(k, l)], Tr[l], F[rre(n, 0)]);
        F[rre(n, 0)] = fma(M[rim(k, l)], Ti[l], F[rre(n, 0)]);
      }
#pragma unroll
      for (int m = 1; m <= P; m++) {
        if (m > n) continue;
        F[rre(n, m)] = fma(M[rre(k, 0)], Tr[m], F[rre(n, m)]);
        F[rim(n, m)] = fma(M[rre(k, 0)], Ti[m], F[rim(n, m)]);
      }
    }
    // m, l >= 1: one set of sums per unordered {u, v}, u >= v, for (m, l) =
    // (u, v) and (v, u)
#pragma unroll
    for (int u = 1; u <= P; u++) {
#pragma unroll
      for (int v = 1; v <= P; v++) {
        if (v > u || u + v > s) continue;
        const double pr = Tr[u + v], pi = Ti[u + v];
        const double mr = (v & 1) ? -Tr[u - v] : Tr[u - v];
        const double mi = u == v ? 0.0 : ((v & 1) ? -Ti[u - v] : Ti[u - v]);
        const double sr = pr + mr, dr = pr - mr;
        const double si = u == v ? pi : pi + mi, di = u == v ? pi : pi - mi;
#pragma unroll
        for (int w = 0; w < 2; w++) {
          if (w == 1 && u == v) continue;
          const int m = w == 0 ? u : v, l = w == 0 ? v : u;
          const double ssi = w == 0 ? si : di, ddi = w == 0 ? di : si;
#pragma unroll
          for (int n = 0; n <= P; n++) {
            const int k = s - n;
            if (n < m || k < l) continue;
            if (n % NC != H) continue;
            const double a = M[rre(k, l)], b = M[rim(k, l)];
            F[rre(n, m)] = fma(a, sr, F[rre(n, m)]);
            F[rim(n, m)] = fma(a, ssi, F[rim(n, m)]);
            F[rre(n, m)] = fma(b, ddi, F[rre(n, m)]);
            F[rim(n, m)] = fma(-b, dr, F[rim(n, m)]);
          }
        }
      }
    }
#pragma unroll
    for (int q = 0; q <= P; q++) {
      if (q > s) continue;
      Br[q] = Ar[q];
      Bi[q] = Ai[q];
      Ar[q] = Tr[q];
      Ai[q] = Ti[q];
    }
    if (s == (P < 2 ? P : 2)) mid();
  }
}

// Source rows: the cells' multipoles in the real layout with the cell centre,
// one contiguous row per cell (k_m2l_rows). The tail of the multipole is
// staged through LDS in 64-byte segments (SEG of them); the first NDIR
// doubles and the centre are read by each lane itself. Lanes reading whole
// rows by themselves touch 64 cache lines per load and made the kernel wait
// on the address unit (P = 7: 36 loads x 64 lines per source against 9600
// cycles of arithmetic, with one wave a SIMD and so no overlap). Four lanes
// now read a segment of one row, and the copy to LDS runs without registers
// while the wave computes. Measured (kernel alone): P = 7, 8.4M bodies, 152M
// directed pairs 20.7 -> 10.4 ms; P = 8, 1M bodies, 38.8M pairs 10.0 -> 4.6 ms;
// P = 6, 250k bodies 0.66 -> 0.35 ms. The rows' traffic (88 GB at P = 7, 8.4
// TB/s, mostly from the memory-side cache) and FP64 issue now bound it
// together. P = 8 keeps its first degrees out of LDS so that
// four waves fit a CU; from P = 9 on four waves share the staged rows.
template <int P>
struct M2lRow {
  static constexpr int NM = (P + 1) * (P + 1);
  static constexpr int NDIR = m2l_row_direct(P);
  static constexpr int SEG = m2l_row_segs(P);
  static constexpr int DIR = m2l_row_tail(P);      // centre + direct part
  static constexpr int WORDS = m2l_row_words(P);  // staged part first, 64-byte rows
};

// Blocks of the row kernels for `words` words in all, one a thread up to 2^30:
// a launch holds fewer than 2^32 threads, and 34M cells at p = 10 have as many
// words, so past that the threads take several.
inline dim3 m2l_row_blocks(size_t words) {
  const size_t most = (size_t)1 << 22, b = (words + 255) / 256;
  return dim3((unsigned)(b < most ? b : most));
}

template <int P>
__device__ __forceinline__ void m2l_row_word(size_t g, const cplx* __restrict__ moments,
                                             const double* __restrict__ ccx,
                                             const double* __restrict__ ccy,
                                             const double* __restrict__ ccz,
                                             double* __restrict__ rows) {
  using R = M2lRow<P>;
  const uint32_t c = (uint32_t)(g / R::WORDS);
  const int i = (int)(g - (size_t)c * R::WORDS);
  // position i -> multipole entry e (-1: none) or centre coordinate
  const int d = i - R::SEG * 8;
  const int e = d < 0 ? (i + R::NDIR < R::NM ? i + R::NDIR : -1) : (d >= 3 && d - 3 < R::NDIR ? d - 3 : -1);
  double v = 0.0;
  if (e >= 0) {
    int n = 0;
    while ((n + 1) * (n + 1) <= e) n++;
    const int r = e - n * n;  // 0: m = 0; 2m-1: re, 2m: im
    const cplx q = moments[(size_t)c * hdim(P) + hidx(n, (r + 1) / 2)];
    v = r > 0 && (r & 1) == 0 ? q.im : q.re;
  } else if (d >= 0 && d < 3) {
    v = d == 0 ? ccx[c] : d == 1 ? ccy[c] : ccz[c];
  }
  rows[g] = v;
}

template <int P>
__global__ void __launch_bounds__(256) k_m2l_rows(uint32_t nc, const cplx* __restrict__ moments,
                                                 const double* __restrict__ ccx,
                                                 const double* __restrict__ ccy,
                                                 const double* __restrict__ ccz,
                                                 double* __restrict__ rows) {
  const size_t words = (size_t)nc * M2lRow<P>::WORDS;
  for (size_t g = (size_t)blockIdx.x * 256 + threadIdx.x; g < words; g += (size_t)gridDim.x * 256)
    m2l_row_word<P>(g, moments, ccx, ccy, ccz, rows);
}

typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(1))) const char gbl_char;

// Piece I of a row group's segments to LDS. The instruction adds its offset
// (64 I) to both addresses, so the LDS side is passed less that much.
template <int SEG, int I = 0>
__device__ __forceinline__ void m2l_copy_segments(gbl_char* from, lds_char* to) {
  if constexpr (I < SEG) {
    __builtin_amdgcn_global_load_lds(from, to + I * (1024 - 64), 16, 64 * I, 0);
    m2l_copy_segments<SEG, I + 1>(from, to);
  }
}

// What the kernels of 64 lanes, one chunk each, share: trips, sources, rows.
template <int P>
struct M2lLane {
  using R = M2lRow<P>;
  const M2lChunk ck;
  const uint64_t* skeys;
  const uint64_t smask;
  const double* rows;
  const int lane;
  uint32_t cnt, trips;
  double dir[R::DIR];  // the source's centre and direct part

  __device__ __forceinline__ M2lLane(bool live, const M2lChunk c, const uint64_t* k, uint64_t sm,
                                     const double* r)
      : ck(c), skeys(k), smask(sm), rows(r), lane((int)(threadIdx.x & 63)) {
    cnt = live ? ck.end - ck.begin : 0u;
    trips = cnt;  // the wave runs its longest chunk's trip count
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) trips = max(trips, (uint32_t)__shfl_xor((int)trips, o, 64));
    trips = (uint32_t)wave_uniform((int)trips);
  }
  // a lane past its chunk's end goes on reading the chunk's last source (a
  // dead lane cell 0), so every row address stays valid
  __device__ __forceinline__ uint32_t source(uint32_t j) const {
    return cnt ? (uint32_t)(skeys[ck.begin + min(j, cnt - 1)] & smask) : 0u;
  }
  // copy of the staged part of the rows of 16 lanes' sources (16 g ..) into LDS,
  // [16-row group][segment][row][4] of 16 bytes, the four pieces of a row rotated
  // by its number so that 16 lanes reading one piece of 16 rows hit all banks
  __device__ __forceinline__ void copy(uint32_t src, int g, lds_char* stage) const {
    const uint32_t rs = (uint32_t)__shfl((int)src, g * 16 + (lane >> 2), 64);
    m2l_copy_segments<R::SEG>(
        (gbl_char*)(rows + (size_t)rs * R::WORDS) + ((lane & 3) ^ ((lane >> 4) & 3)) * 16,
        stage + g * R::SEG * 1024);
  }
  // piece e (two doubles) of the lane's own row
  __device__ __forceinline__ double2 piece(const double2* stage, int e) const {
    const double2* mine = stage + (lane >> 4) * R::SEG * 64 + (lane & 15) * 4;
    return mine[(e >> 2) * 64 + ((e & 3) ^ ((lane >> 2) & 3))];
  }
  __device__ __forceinline__ void direct(uint32_t sc) {
    const double2* d2 = (const double2*)(rows + (size_t)sc * R::WORDS + R::SEG * 8);
#pragma unroll
    for (int i = 0; i < (3 + R::NDIR + 1) / 2; i++) {
      const double2 v = d2[i];
      dir[2 * i] = v.x;
      dir[2 * i + 1] = v.y;
    }
  }
};

// The degrees n % NC == H of a chunk's partial.
template <int P, int H, int NC>
__device__ __forceinline__ void m2l_store64(const double* F, double* __restrict__ out) {
#pragma unroll
  for (int n = 0; n <= P; n++) {
    if (n % NC != H) continue;
    out[rre(n, 0)] = 2.0 * F[rre(n, 0)];
#pragma unroll
    for (int m = 1; m <= P; m++) {
      if (m > n) continue;
      out[rre(n, m)] = F[rre(n, m)];
      out[rim(n, m)] = F[rim(n, m)];
    }
  }
}

template <int P>
__global__ void __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(1))) k_m2l(const M2lChunk* __restrict__ chunks,
                                              uint32_t nchunks, const uint64_t* __restrict__ skeys,
                                              uint64_t smask, const double* __restrict__ rows,
                                              double soft2, double* __restrict__ part) {
  using R = M2lRow<P>;
  __shared__ double2 stage[R::SEG * 256];
  const uint32_t ci = xcd_block(blockIdx.x, gridDim.x) * 64 + threadIdx.x;
  const bool live = ci < nchunks;
  M2lChunk ck{0, 0, 0};
  if (live) ck = chunks[ci];
  M2lLane<P> ln(live, ck, skeys, smask, rows);
  if (ln.trips == 0) return;
  lds_char* stage3 = (lds_char*)stage;
  double F[R::NM];
#pragma unroll
  for (int i = 0; i < R::NM; i++) F[i] = 0.0;
  auto fetch = [&](uint32_t src) {
    ln.direct(src);
#pragma unroll
    for (int g = 0; g < 4; g++) ln.copy(src, g, stage3);
  };
  fetch(ln.source(0));
  const double* t = rows + (size_t)ck.target * R::WORDS + R::SEG * 8;
  const double tx = t[0], ty = t[1], tz = t[2];
  uint32_t src_n = ln.source(1);
  for (uint32_t j = 0; j < ln.trips; j++) {
    double M[R::NM];
    const double x = tx - ln.dir[0], y = ty - ln.dir[1], z = tz - ln.dir[2];
#pragma unroll
    for (int i = 0; i < R::NDIR; i++) M[i] = ln.dir[3 + i];
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the copy has landed
#pragma unroll
    for (int e = 0; e < R::SEG * 4; e++) {
      const double2 v = ln.piece(stage, e);
      if (R::NDIR + 2 * e < R::NM) M[R::NDIR + 2 * e] = v.x;
      if (R::NDIR + 2 * e + 1 < R::NM) M[R::NDIR + 2 * e + 1] = v.y;
    }
    // the next source's copy starts once this one's row has been read (while
    // the first degrees are computed) and runs under the rest
    m2l_accumulate64<P, 0, 1>(j < ln.cnt, x, y, z, soft2, M, F, [](int) {}, [&] {
      if (j + 1 < ln.trips) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        const uint32_t cur = src_n;
        src_n = ln.source(j + 2);
        fetch(cur);
      }
    });
  }
  if (live) m2l_store64<P, 0, 1>(F, part + (size_t)ci * R::NM);
}

// P = 9 and 10: the accumulators and the row need more registers than a wave has
// (a wave for each half of the degrees, rows read into registers: 227 and 617 of
// them spilled). Four waves share the pairs of 64 chunks and one staged copy of
// their rows; wave H takes the degrees n % 4 == H (of about equal work, 22 to 39
// accumulators) and reads, for the products of degree s, the degrees s - n of the
// row from LDS, a quarter of it on average, so that 256 registers do and two blocks
// fit a CU. Each wave runs the recursion and makes the sums S and D for itself, on
// top of its quarter of the products. M2L of 1M bodies at eps 1e-5, theta
// 0.5 and leaf 96: P = 9, 34.0M directed pairs 18.0 -> 7.0 ms, 18.4M 9.3 -> 3.5;
// P = 10, 29.8M 31.6 -> 8.0, 18.4M 18.2 -> 4.5 (term by term on two waves before
// that: 13.5, 7.3, 14.7 and 9.1).
constexpr int M2L_SHARED_FROM = 9, M2L_NC = 4;

template <int P, int H>
__device__ __forceinline__ void m2l_shared(uint32_t ci, bool live, const M2lChunk ck,
                                           const uint64_t* __restrict__ skeys, uint64_t smask,
                                           const double* __restrict__ rows, double soft2,
                                           const double2* stage, double* __restrict__ part) {
  using R = M2lRow<P>;
  static_assert(R::NDIR == 1, "entry 2 e + 1 starts piece e");
  M2lLane<P> ln(live, ck, skeys, smask, rows);
  if (ln.trips == 0) return;  // of the block: its waves have the same chunks
  lds_char* stage3 = (lds_char*)stage;
  double F[R::NM];
#pragma unroll
  for (int i = 0; i < R::NM; i++) F[i] = 0.0;
  uint32_t src = ln.source(0);
  ln.direct(src);
  ln.copy(src, H, stage3);
  const double* t = rows + (size_t)ck.target * R::WORDS + R::SEG * 8;
  const double tx = t[0], ty = t[1], tz = t[2];
  src = ln.source(1);
  for (uint32_t j = 0; j < ln.trips; j++) {
    double M[R::NM];
    const double x = tx - ln.dir[0], y = ty - ln.dir[1], z = tz - ln.dir[2];
    M[0] = ln.dir[3];
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the wave's copy has landed ...
    __syncthreads();                                  // ... and the block's
    m2l_accumulate64<P, H, M2L_NC>(
        j < ln.cnt, x, y, z, soft2, M, F,
        [&](int s) {
          // the products of the degrees before come first (nothing else keeps the
          // compiler from reading all of the row here and multiplying later)
#pragma unroll
          for (int n = 0; n < P; n++) {
            if (n >= s || n % M2L_NC != H) continue;
#pragma unroll
            for (int i = n * n; i <= n * n + 2 * n; i++) asm volatile("" : "+v"(F[i]));
          }
          asm volatile("" ::: "memory");
#pragma unroll
          for (int k = 1; k <= P; k++) {
            if (k > s || (s - k) % M2L_NC != H) continue;
#pragma unroll
            for (int e = (k * k - 1) / 2; e <= (k * k + 2 * k - 1) / 2; e++) {
              const double2 v = ln.piece(stage, e);
              if (2 * e + 1 >= k * k) M[2 * e + 1] = v.x;
              if (2 * e + 2 <= k * k + 2 * k) M[2 * e + 2] = v.y;
            }
          }
          if (s != P) return;
          // the last of the rows has been read by every wave: the next ones' copy
          // runs under the products of degree P
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          __syncthreads();
          if (j + 1 < ln.trips) {
            ln.direct(src);
            ln.copy(src, H, stage3);
            src = ln.source(j + 2);
          }
        },
        [] {});
  }
  if (live) m2l_store64<P, H, M2L_NC>(F, part + (size_t)ci * R::NM);
}

template <int P>
__global__ void __launch_bounds__(64 * M2L_NC) __attribute__((amdgpu_waves_per_eu(2)))
k_m2l_shared(const M2lChunk* __restrict__ chunks, uint32_t nchunks,
             const uint64_t* __restrict__ skeys, uint64_t smask, const double* __restrict__ rows,
             double soft2, double* __restrict__ part) {
  __shared__ double2 stage[M2lRow<P>::SEG * 256];
  const uint32_t ci = xcd_block(blockIdx.x, gridDim.x) * 64 + (threadIdx.x & 63);
  const bool live = ci < nchunks;
  M2lChunk ck{0, 0, 0};
  if (live) ck = chunks[ci];
  const int h = wave_uniform((int)(threadIdx.x >> 6));
  if (h == 0)
    m2l_shared<P, 0>(ci, live, ck, skeys, smask, rows, soft2, stage, part);
  else if (h == 1)
    m2l_shared<P, 1>(ci, live, ck, skeys, smask, rows, soft2, stage, part);
  else if (h == 2)
    m2l_shared<P, 2>(ci, live, ck, skeys, smask, rows, soft2, stage, part);
  else
    m2l_shared<P, 3>(ci, live, ck, skeys, smask, rows, soft2, stage, part);
}

template <int P>
void m2l_t(const M2lChunk* chunks, uint32_t nchunks, const uint64_t* skeys, uint64_t smask,
           uint32_t nc, DevCells c, const cplx* moments, double soft2, double* rows, double* part,
           hipStream_t s) {
  if (!nchunks) return;
  hipLaunchKernelGGL(k_m2l_rows<P>, m2l_row_blocks((size_t)nc * M2lRow<P>::WORDS), dim3(256), 0, s,
                     nc, moments, c.cx, c.cy, c.cz, rows);
  const dim3 nb((nchunks + 63) / 64);
  if constexpr (P < M2L_SHARED_FROM)
    hipLaunchKernelGGL(k_m2l<P>, nb, dim3(64), 0, s, chunks, nchunks, skeys, smask,
                       (const double*)rows, soft2, part);
  else
    hipLaunchKernelGGL(k_m2l_shared<P>, nb, dim3(64 * M2L_NC), 0, s, chunks, nchunks, skeys, smask,
                       (const double*)rows, soft2, part);
}

// ------------------------------------------------------- FP32 (mixed form)
// The same chunked M2L on radius-scaled FP32 operands. Per target t a scale
// lam_t (its radius, floored at a quarter of its octant edge) gives
// dimensionless offsets v = r / lam_t, and by homogeneity
// Theta_s(r) = lam_t^-(s+1) Theta_s(v) (softened: eps -> eps / lam_t), so
//   F_n = lam_t^-(n+1) sum_k (M_k lam_t^-k) Theta_{n+k}(v).
// Moments are stored pre-scaled per source cell, Mt_k = M_k lam_s^-k (FP32),
// and M_k lam_t^-k = Mt_k kappa^k with kappa = lam_s / lam_t. Every operand
// is then O(1) up to the MAC's (rho / r)^k decay; the recursion, products and
// the chunk's sums run in FP32. Chunks write their scaled F in FP32; the
// reduce adds a target's chunks in FP64 and applies lam_t^-(n+1).
template <int P, int H>
__device__ __forceinline__ void m2l_chunk32(const M2lChunk ck, uint32_t ci,
                                            const uint64_t* __restrict__ skeys, uint64_t smask,
                                            const double* __restrict__ ccx,
                                            const double* __restrict__ ccy,
                                            const double* __restrict__ ccz,
                                            const double* __restrict__ lam,
                                            const cplxf* __restrict__ m32, double soft2,
                                            cplxf* __restrict__ part) {
  constexpr int NF = hnpos(P);
  const double tx = ccx[ck.target], ty = ccy[ck.target], tz = ccz[ck.target];
  const double ilt = 1.0 / lam[ck.target];
  const float s2s = (float)(soft2 * ilt * ilt);
  cplxf F[NF];
#pragma unroll
  for (int i = 0; i < NF; i++) F[i] = cplxf{0.f, 0.f};
  for (uint32_t j = ck.begin; j < ck.end; j++) {
    const uint32_t src = (uint32_t)(skeys[j] & smask);
    const cplxf* ms = m32 + (size_t)src * NF;
    const float kap = (float)(lam[src] * ilt);
    cplxf M[NF];
    float kk = 1.f;
#pragma unroll
    for (int k = 0; k <= P; k++) {
#pragma unroll
      for (int l = 0; l <= k; l++) {
        const cplxf v = ms[hpos(k, l)];
        M[hpos(k, l)] = cplxf{v.re * kk, v.im * kk};
      }
      kk *= kap;
    }
    m2l_accumulate<P, H, P, float, cplxf>(true, (float)((tx - ccx[src]) * ilt),
                                          (float)((ty - ccy[src]) * ilt),
                                          (float)((tz - ccz[src]) * ilt), s2s, M, F, [](float&) {});
  }
  cplxf* out = part + (size_t)ci * NF;
#pragma unroll
  for (int n = 0; n <= P; n++) {
    if (H != 2 && (n & 1) != H) continue;
#pragma unroll
    for (int m = 0; m <= n; m++) out[hpos(n, m)] = F[hpos(n, m)];
  }
}

// Source rows of the staged orders 3..8: SEG 64-byte segments of the scaled
// moments (from the NDIR-th on) that go through LDS, then centre, scale and the
// first NDIR moments, which each lane reads itself. As in the FP64 form, rows
// read lane by lane kept the address unit busy as long as the arithmetic (P =
// 7: 18 loads of 64 lines a source), and the loads were waited for at the top
// of each source, with two waves a SIMD; the copy now runs under the products of
// the last degree, before which the row must be in registers anyway (earlier
// it costs registers that P = 8 does not have: 2.44 ms there, 2.68 - 2.83 before
// an earlier degree). Two waves a SIMD of 20 KB each fill the LDS. Kernel alone:
// P = 8, 1M bodies 2.94 -> 2.44 ms; P = 7, 16.8M bodies 17.3 -> 15.2; P = 3 .. 6,
// 250k bodies 198 / 244 / 380 / 446 -> 128 / 179 / 222 / 298 us, and 4 - 16 us (83
// at 16.8M) for the rows. FP32 issue bounds it now (3.1 cycles an instruction).
// P = 1, 2 have less than a segment, and P = 9, 10 no registers left: read
// directly.
template <int P>
struct M2lRow32 {
  static constexpr int NF = hnpos(P);
  static constexpr bool STAGED = m2l32_staged(P);
  static constexpr int SEG = m2l32_row_segs(P);
  static constexpr int NDIR = m2l32_row_direct(P);
  static constexpr int WORDS = m2l32_row_words(P);  // of 8 bytes
};

template <int P>
__device__ __forceinline__ void m2l_row_word32(size_t g, const cplxf* __restrict__ m32,
                                               const double* __restrict__ ccx,
                                               const double* __restrict__ ccy,
                                               const double* __restrict__ ccz,
                                               const double* __restrict__ lam,
                                               double* __restrict__ rows) {
  using R = M2lRow32<P>;
  const uint32_t c = (uint32_t)(g / R::WORDS);
  const int i = (int)(g - (size_t)c * R::WORDS), d = i - R::SEG * 8;
  const int e = d < 0 ? i + R::NDIR : d >= 4 && d - 4 < R::NDIR ? d - 4 : -1;
  double v = 0.0;
  if (e >= 0)
    v = __builtin_bit_cast(double, m32[(size_t)c * R::NF + e]);
  else if (d < 4)
    v = d == 0 ? ccx[c] : d == 1 ? ccy[c] : d == 2 ? ccz[c] : lam[c];
  rows[g] = v;
}

template <int P>
__global__ void __launch_bounds__(256) k_m2l_rows32(uint32_t nc, const cplxf* __restrict__ m32,
                                                   const double* __restrict__ ccx,
                                                   const double* __restrict__ ccy,
                                                   const double* __restrict__ ccz,
                                                   const double* __restrict__ lam,
                                                   double* __restrict__ rows) {
  const size_t words = (size_t)nc * M2lRow32<P>::WORDS;
  for (size_t g = (size_t)blockIdx.x * 256 + threadIdx.x; g < words; g += (size_t)gridDim.x * 256)
    m2l_row_word32<P>(g, m32, ccx, ccy, ccz, lam, rows);
}

// The chunks of 64 lanes, rows staged as in m2l_chunks64 (same layout in LDS).
template <int P>
__device__ __forceinline__ void m2l_chunks32(uint32_t ci, bool live, const M2lChunk ck,
                                             const uint64_t* __restrict__ skeys, uint64_t smask,
                                             const double* __restrict__ rows, double soft2,
                                             float4* stage, cplxf* __restrict__ part) {
  using R = M2lRow32<P>;
  const int lane = threadIdx.x;
  lds_char* stage3 = (lds_char*)stage;
  const uint32_t cnt = live ? ck.end - ck.begin : 0u;
  uint32_t trips = cnt;  // the wave runs its longest chunk's trip count
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) trips = max(trips, (uint32_t)__shfl_xor((int)trips, o, 64));
  trips = (uint32_t)wave_uniform((int)trips);
  if (trips == 0) return;
  cplxf F[R::NF];
#pragma unroll
  for (int i = 0; i < R::NF; i++) F[i] = cplxf{0.f, 0.f};
  // past the end: the last one; a dead lane: the first key's
  auto source = [&](uint32_t j) -> uint32_t {
    return (uint32_t)(skeys[ck.begin + min(j, max(cnt, 1u) - 1)] & smask);
  };
  auto copy = [&](uint32_t src) {
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const uint32_t rs = (uint32_t)__shfl((int)src, g * 16 + (lane >> 2), 64);
      m2l_copy_segments<R::SEG>(
          (gbl_char*)(rows + (size_t)rs * R::WORDS) + ((lane & 3) ^ ((lane >> 4) & 3)) * 16,
          stage3 + g * R::SEG * 1024);
    }
  };
  const int swz = (lane >> 2) & 3;
  const float4* mine = stage + (lane >> 4) * R::SEG * 64 + (lane & 15) * 4;
  double cl[4];  // the source's centre and scale
  cplxf dir[R::NDIR];
  auto direct = [&](uint32_t sc) {
    const double* d = rows + (size_t)sc * R::WORDS + R::SEG * 8;
    const double2 a = *(const double2*)d, b = *(const double2*)(d + 2);
    cl[0] = a.x;
    cl[1] = a.y;
    cl[2] = b.x;
    cl[3] = b.y;
    const float4* q = (const float4*)(d + 4);
#pragma unroll
    for (int i = 0; i < (R::NDIR + 1) / 2; i++) {
      const float4 v = q[i];
      dir[2 * i] = cplxf{v.x, v.y};
      if (2 * i + 1 < R::NDIR) dir[2 * i + 1] = cplxf{v.z, v.w};
    }
  };
  uint32_t src = source(0);
  direct(src);
  copy(src);
  const double* t = rows + (size_t)ck.target * R::WORDS + R::SEG * 8;
  const double tx = t[0], ty = t[1], tz = t[2], ilt = 1.0 / t[3];
  const float s2s = (float)(soft2 * ilt * ilt);
  src = source(1);
  for (uint32_t j = 0; j < trips; j++) {
    const float x = (float)((tx - cl[0]) * ilt), y = (float)((ty - cl[1]) * ilt),
                z = (float)((tz - cl[2]) * ilt);
    const float kap = (float)(cl[3] * ilt);
    float kk[P + 1];
    kk[0] = 1.f;
#pragma unroll
    for (int k = 1; k <= P; k++) kk[k] = kk[k - 1] * kap;
    cplxf M[R::NF];
#pragma unroll
    for (int i = 0; i < R::NDIR; i++) M[i] = dir[i];
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the copy has landed
#pragma unroll
    for (int e = 0; e < R::SEG * 4; e++) {
      const float4 v = mine[(e >> 2) * 64 + ((e & 3) ^ swz)];
      M[R::NDIR + 2 * e] = cplxf{v.x, v.y};
      M[R::NDIR + 2 * e + 1] = cplxf{v.z, v.w};
    }
#pragma unroll
    for (int k = 0; k <= P; k++)
#pragma unroll
      for (int l = 0; l <= k; l++) {
        M[hpos(k, l)].re *= kk[k];
        M[hpos(k, l)].im *= kk[k];
      }
    m2l_accumulate<P, 2, P, float, cplxf>(j < cnt, x, y, z, s2s, M, F, [&](float& tq) {
      // the row has been read; tq ties the point to the degrees (a branch or a
      // free wait would move to the top of the loop, and the row's registers
      // with it)
      asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(tq)::"memory");
      direct(src);
      copy(src);
      src = source(j + 2);
    });
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the last copy, into a wave's LDS
  if (!live) return;
  cplxf* out = part + (size_t)ci * R::NF;
#pragma unroll
  for (int i = 0; i < R::NF; i++) out[i] = F[i];
}

template <int P>
__global__ void __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(2))) k_m2l32_staged(const M2lChunk* __restrict__ chunks,
                                                       uint32_t nchunks,
                                                       const uint64_t* __restrict__ skeys,
                                                       uint64_t smask,
                                                       const double* __restrict__ rows,
                                                       double soft2, cplxf* __restrict__ part) {
  __shared__ float4 stage[M2lRow32<P>::SEG * 256];
  const uint32_t ci = xcd_block(blockIdx.x, gridDim.x) * 64 + threadIdx.x;
  const bool live = ci < nchunks;
  M2lChunk ck{0, 0, 0};
  if (live) ck = chunks[ci];
  m2l_chunks32<P>(ci, live, ck, skeys, smask, rows, soft2, stage, part);
}

template <int P, bool SPLIT>
__global__ void __launch_bounds__(64) k_m2l32(const M2lChunk* __restrict__ chunks,
                                             uint32_t nchunks, const uint64_t* __restrict__ skeys,
                                             uint64_t smask, const double* __restrict__ ccx,
                                             const double* __restrict__ ccy,
                                             const double* __restrict__ ccz,
                                             const double* __restrict__ lam,
                                             const cplxf* __restrict__ m32, double soft2,
                                             cplxf* __restrict__ part) {
  const uint32_t lb = xcd_block(blockIdx.x, gridDim.x);
  if constexpr (SPLIT) {
    const uint32_t ci = (lb >> 1) * blockDim.x + threadIdx.x;
    if (ci >= nchunks) return;
    if (lb & 1)
      m2l_chunk32<P, 1>(chunks[ci], ci, skeys, smask, ccx, ccy, ccz, lam, m32, soft2, part);
    else
      m2l_chunk32<P, 0>(chunks[ci], ci, skeys, smask, ccx, ccy, ccz, lam, m32, soft2, part);
  } else {
    const uint32_t ci = lb * blockDim.x + threadIdx.x;
    if (ci >= nchunks) return;
    m2l_chunk32<P, 2>(chunks[ci], ci, skeys, smask, ccx, ccy, ccz, lam, m32, soft2, part);
  }
}

// Orders whose FP32 accumulators are split over two waves.
#ifndef FMMH_M2L32_SPLIT_FROM
#define FMMH_M2L32_SPLIT_FROM 9
#endif

template <int P>
void m2l32_t(const M2lChunk* chunks, uint32_t nchunks, const uint64_t* skeys, uint64_t smask,
             uint32_t nc, DevCells c, const double* lam, const cplxf* m32, double soft2,
             double* rows, cplxf* part, hipStream_t s) {
  if (!nchunks) return;
  if constexpr (M2lRow32<P>::STAGED) {
    hipLaunchKernelGGL(k_m2l_rows32<P>, m2l_row_blocks((size_t)nc * M2lRow32<P>::WORDS), dim3(256),
                       0, s, nc, m32, c.cx, c.cy, c.cz, lam, rows);
    hipLaunchKernelGGL(k_m2l32_staged<P>, dim3((nchunks + 63) / 64), dim3(64), 0, s, chunks,
                       nchunks, skeys, smask, (const double*)rows, soft2, part);
  } else {
    constexpr bool split = P >= FMMH_M2L32_SPLIT_FROM;
    const uint32_t nb = (nchunks + 63) / 64 * (split ? 2 : 1);
    hipLaunchKernelGGL((k_m2l32<P, split>), dim3(nb), dim3(64), 0, s, chunks, nchunks, skeys,
                       smask, c.cx, c.cy, c.cz, lam, m32, soft2, part);
  }
}

// One translation unit per range of orders instantiates the launches.
#define FMMH_M2L_INSTANTIATE(P)                                                             \
  template void m2l_t<P>(const M2lChunk*, uint32_t, const uint64_t*, uint64_t, uint32_t,    \
                         DevCells, const cplx*, double, double*, double*, hipStream_t);     \
  template void m2l32_t<P>(const M2lChunk*, uint32_t, const uint64_t*, uint64_t, uint32_t,  \
                           DevCells, const double*, const cplxf*, double, double*, cplxf*,  \
                           hipStream_t);

}  // namespace fmmh
