// upward.hip — upward pass on gfx950 (compiled -ffp-contract=off):
// P2M and M2M on Dehnen solid harmonics, multipole power, the p=0 f pre-pass
// and per-cell fmin. These feed the error-controlled MAC, whose decisions
// must match the reference's exactly, so every sum runs in the reference's
// order (crates/fmm moments.rs:30-168, mac.rs:99-186) and no product is fused.
#include "common.h"
#include "internal.h"

namespace fmmh {

// Column m of Upsilon(r) (harmonic.rs:141-173) for one body, with the
// diagonal seed chained exactly as the table recursion does, accumulated
// as mass * Upsilon into acc[n] (m) and accn[n] (-m). P compile-time keeps
// the column in registers.
template <int P>
__device__ __forceinline__ void upsilon_column_acc(double x, double y, double z, double r2, int m,
                                                   double ms, cplx* acc, cplx* accn) {
  cplx u = cplx{1.0, 0.0};
#pragma unroll
  for (int j = 1; j <= P; j++)
    if (j <= m) u = cmul(cscale(cplx{x, y}, 1.0 / (double)(2 * j)), u);
  const double sgn = (m % 2 == 0) ? 1.0 : -1.0;
  cplx u1 = u, u2 = cz();
#pragma unroll
  for (int n = 0; n <= P; n++) {
    if (n < m) continue;
    cplx un;
    if (n == m) {
      un = u;
    } else {
      double a = (double)(2 * n - 1) * z;
      double c = (double)(n * n - m * m);
      // n == m+1 reads the ZERO seed: 0*r2 = +0 and x - (+0) = x.
      cplx p2 = (n >= m + 2) ? u2 : cz();
      un = cscale(csub(cscale(u1, a), cscale(p2, r2)), 1.0 / c);
      u2 = u1;
      u1 = un;
    }
    acc[n] = cadd(acc[n], cscale(un, ms));
    if (m > 0) {
      cplx neg = cscale(cconj(un), sgn);
      accn[n] = cadd(accn[n], cscale(neg, ms));
    }
  }
}

// P2M (moments.rs:30-53) of column M of one leaf; bodies in slot order.
template <int P, int M>
__device__ __forceinline__ void p2m_column(uint32_t id, DevCells c, DevBodies b,
                                           cplx* __restrict__ moments) {
  constexpr int D = hdim(P);
  const double zx = c.cx[id], zy = c.cy[id], zz = c.cz[id];
  cplx acc[P + 1], accn[P + 1];
#pragma unroll
  for (int n = 0; n <= P; n++) acc[n] = accn[n] = cz();
  const uint32_t f = c.first[id], e = f + c.count[id];
  for (uint32_t k = f; k < e; k++) {
    const double4 q = b.xyzm[k];  // one 32-byte load (a lane's leaf differs from its neighbours')
    double x = q.x - zx, y = q.y - zy, z = q.z - zz;
    double r2 = x * x + y * y + z * z;
    upsilon_column_acc<P>(x, y, z, r2, M, q.w, acc, accn);
  }
  cplx* out = moments + (size_t)id * D;
#pragma unroll
  for (int n = M; n <= P; n++) {
    out[hidx(n, M)] = acc[n];
    if (M > 0) out[hidx(n, -M)] = accn[n];
  }
}

template <int P, int M = 0>
__device__ __forceinline__ void p2m_dispatch(int m, uint32_t id, DevCells c, DevBodies b,
                                             cplx* __restrict__ moments) {
  if constexpr (M <= P) {
    if (m == M)
      p2m_column<P, M>(id, c, b, moments);
    else
      p2m_dispatch<P, M + 1>(m, id, c, b, moments);
  }
}

// One block per 64 leaves, wave m computing column m of each: a wave runs
// one column's exact work, and the leaves come in body-count order, so its
// lanes loop over nearly equal numbers of bodies.
template <int P>
__global__ void __launch_bounds__(64 * (P + 1)) k_p2m(const uint32_t* __restrict__ leaf_ids,
                                                     uint32_t nleaves, DevCells c, DevBodies b,
                                                     cplx* __restrict__ moments) {
  const int m = (int)(threadIdx.x >> 6);
  const uint32_t li = blockIdx.x * 64 + (threadIdx.x & 63);
  if (li >= nleaves) return;
  p2m_dispatch<P>(m, leaf_ids[li], c, b, moments);
}

// Full Upsilon column m (both signs) written into a table (for M2M's
// per-child tables in LDS).
template <int P>
__device__ __forceinline__ void upsilon_column_store(double x, double y, double z, int m,
                                                     cplx* tab) {
  double r2 = x * x + y * y + z * z;
  cplx u = cplx{1.0, 0.0};
#pragma unroll
  for (int j = 1; j <= P; j++)
    if (j <= m) u = cmul(cscale(cplx{x, y}, 1.0 / (double)(2 * j)), u);
  const double sgn = (m % 2 == 0) ? 1.0 : -1.0;
  cplx u1 = u, u2 = cz();
#pragma unroll
  for (int n = 0; n <= P; n++) {
    if (n < m) continue;
    cplx un;
    if (n == m) {
      un = u;
    } else {
      double a = (double)(2 * n - 1) * z;
      double c = (double)(n * n - m * m);
      cplx p2 = (n >= m + 2) ? u2 : cz();
      un = cscale(csub(cscale(u1, a), cscale(p2, r2)), 1.0 / c);
      u2 = u1;
      u1 = un;
    }
    tab[hidx(n, m)] = un;
    if (m > 0) tab[hidx(n, -m)] = cscale(cconj(un), sgn);
  }
}

// M2M work schedule. Output coefficient e = (n, m) of a parent is the sum,
// child by child, of its terms (k, l): Upsilon_k^l(child offset) times the
// child's M_{n-k}^{m-l}, in the reference's order (k ascending, then l).
// The schedule lists every output's terms as LDS byte offsets
// (Upsilon index * 16 | moment index * 16 << 16) and orders the outputs
// ("slots") by term count, longest first, so that the eight outputs a wave
// works on at a time have nearly equal trip counts.
constexpr int m2m_terms(int n, int m) {
  int t = 0;
  for (int k = 0; k <= n; k++) {
    const int nk = n - k;
    const int lo = -k > m - nk ? -k : m - nk, hi = k < m + nk ? k : m + nk;
    if (hi >= lo) t += hi - lo + 1;
  }
  return t;
}
constexpr int m2m_total_terms(int p) {
  int t = 0;
  for (int n = 0; n <= p; n++)
    for (int m = -n; m <= n; m++) t += m2m_terms(n, m);
  return t;
}

template <int P>
struct M2mSched {
  static constexpr int D = hdim(P);
  static constexpr int T = m2m_total_terms(P);
  uint32_t code[T];
  uint16_t e_of[D], base[D], nt[D];
};

template <int P>
constexpr M2mSched<P> make_m2m_sched() {
  M2mSched<P> s{};
  constexpr int D = M2mSched<P>::D;
  int cnt[D] = {};
  int ord[D] = {};
  for (int e = 0; e < D; e++) {
    int n = 0;
    while ((n + 1) * (n + 1) <= e) n++;
    cnt[e] = m2m_terms(n, e - n * (n + 1));
    ord[e] = e;
  }
  for (int i = 1; i < D; i++) {  // stable insertion sort, longest first
    const int v = ord[i];
    int j = i;
    while (j > 0 && cnt[ord[j - 1]] < cnt[v]) {
      ord[j] = ord[j - 1];
      j--;
    }
    ord[j] = v;
  }
  int at = 0;
  for (int slot = 0; slot < D; slot++) {
    const int e = ord[slot];
    int n = 0;
    while ((n + 1) * (n + 1) <= e) n++;
    const int m = e - n * (n + 1);
    s.e_of[slot] = (uint16_t)e;
    s.base[slot] = (uint16_t)at;
    s.nt[slot] = (uint16_t)cnt[e];
    for (int k = 0; k <= n; k++) {
      const int nk = n - k;
      const int lo = -k > m - nk ? -k : m - nk, hi = k < m + nk ? k : m + nk;
      for (int l = lo; l <= hi; l++)
        s.code[at++] = (uint32_t)(hidx(k, l) * 16) | ((uint32_t)(hidx(nk, m - l) * 16) << 16);
    }
  }
  return s;
}

template <int P>
__device__ constexpr M2mSched<P> kM2mSched = make_m2m_sched<P>();

constexpr int M2M_T = 256;

// M2M (moments.rs:56-90): one block per internal cell of a level. The
// children's Upsilon tables and moments are staged in LDS; thread (slot
// group g, child o) computes child o's partial sum of the outputs in slots
// g, g + 32, g + 64, ... (each from zero, terms in the reference's order),
// then each output adds its children's partials in octant order. Every
// output is therefore the reference's sum, bit for bit.
template <int P>
__global__ void __launch_bounds__(M2M_T) k_m2m(const uint32_t* __restrict__ cells, uint32_t cnt,
                                              DevCells c, cplx* __restrict__ moments) {
  using S = M2mSched<P>;
  constexpr int D = S::D;
  __shared__ cplx u[8][D];
  __shared__ cplx mo[8][D];
  __shared__ cplx part[8][D];
  __shared__ uint32_t code[S::T];
  const uint32_t id = cells[blockIdx.x];
  if (c.leaf[id]) return;  // block-uniform
  const double zx = c.cx[id], zy = c.cy[id], zz = c.cz[id];
  const int32_t* ch = c.children + (size_t)id * 8;
  for (int t = threadIdx.x; t < 8 * (P + 1); t += M2M_T) {
    const int o = t / (P + 1), m = t % (P + 1);
    const int q = ch[o];
    if (q < 0) continue;
    upsilon_column_store<P>(c.cx[q] - zx, c.cy[q] - zy, c.cz[q] - zz, m, u[o]);
  }
  for (int t = threadIdx.x; t < 8 * D; t += M2M_T) {
    const int o = t / D, e = t - o * D;
    const int q = ch[o];
    if (q >= 0) mo[o][e] = moments[(size_t)q * D + e];
  }
  for (int t = threadIdx.x; t < S::T; t += M2M_T) code[t] = kM2mSched<P>.code[t];
  __syncthreads();
  const int o = threadIdx.x & 7;
  const bool has = ch[o] >= 0;
  const char* ub = (const char*)&u[o][0];
  const char* mb = (const char*)&mo[o][0];
  for (int slot = threadIdx.x >> 3; slot < D; slot += M2M_T / 8) {
    const int e = kM2mSched<P>.e_of[slot], b = kM2mSched<P>.base[slot];
    const int nt = has ? (int)kM2mSched<P>.nt[slot] : 0;
    cplx acc = cz();
    // the terms' LDS reads overlap; the additions stay in order
#pragma unroll 4
    for (int t = 0; t < nt; t++) {
      const uint32_t cd = code[b + t];
      const cplx uv = *(const cplx*)(ub + (cd & 0xFFFFu));
      const cplx mv = *(const cplx*)(mb + (cd >> 16));
      acc = cadd(acc, cmul(uv, mv));
    }
    part[o][e] = acc;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < D; e += M2M_T) {
    cplx acc = cz();
    for (int q = 0; q < 8; q++)
      if (ch[q] >= 0) acc = cadd(acc, part[q][e]);
    moments[(size_t)id * D + e] = acc;
  }
}

template <int P>
static void p2m_t(const uint32_t* leaf_ids, uint32_t nleaves, DevCells c, DevBodies b,
                  cplx* moments, hipStream_t s) {
  hipLaunchKernelGGL(k_p2m<P>, dim3((nleaves + 63) / 64), dim3(64 * (P + 1)), 0, s, leaf_ids,
                     nleaves, c, b, moments);
}

template <int P>
static void m2m_t(const uint32_t* cells, uint32_t cnt, DevCells c, cplx* moments, hipStream_t s) {
  hipLaunchKernelGGL(k_m2m<P>, dim3(cnt), dim3(M2M_T), 0, s, cells, cnt, c, moments);
}

#define FMMH_P_SWITCH(p, CALL) \
  switch (p) {                 \
    case 1: CALL(1); break;    \
    case 2: CALL(2); break;    \
    case 3: CALL(3); break;    \
    case 4: CALL(4); break;    \
    case 5: CALL(5); break;    \
    case 6: CALL(6); break;    \
    case 7: CALL(7); break;    \
    case 8: CALL(8); break;    \
    case 9: CALL(9); break;    \
    case 10: CALL(10); break;  \
    default: return false;     \
  }

bool launch_p2m(int p, const uint32_t* leaf_ids, uint32_t nleaves, DevCells c, DevBodies b,
                cplx* moments, hipStream_t s) {
  if (nleaves == 0) return true;
#define CALL(P) p2m_t<P>(leaf_ids, nleaves, c, b, moments, s)
  FMMH_P_SWITCH(p, CALL)
#undef CALL
  return true;
}

bool launch_m2m(int p, const uint32_t* cells, uint32_t cnt, DevCells c, cplx* moments,
                hipStream_t s) {
  if (cnt == 0) return true;
#define CALL(P) m2m_t<P>(cells, cnt, c, moments, s)
  FMMH_P_SWITCH(p, CALL)
#undef CALL
  return true;
}

// Multipole power (moments.rs:150-168): one thread per (cell, n).
__global__ void __launch_bounds__(256) k_pows(int p, uint32_t nc, const cplx* __restrict__ moments,
                                             const double* __restrict__ fact,
                                             double* __restrict__ pows) {
  size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= (size_t)nc * (p + 1)) return;
  size_t cell = t / (p + 1);
  int n = (int)(t % (p + 1));
  const cplx* mc = moments + cell * (size_t)hdim(p);
  double s = 0.0;
  for (int m = -n; m <= n; m++) {
    int am = m < 0 ? -m : m;
    cplx v = mc[hidx(n, m)];
    double w = fact[n - am] * fact[n + am];
    s += w * (v.re * v.re + v.im * v.im);
  }
  pows[t] = sqrt(s);
}

void launch_pows(int p, uint32_t nc, const cplx* moments, const double* fact, double* pows,
                 hipStream_t s) {
  size_t threads = (size_t)nc * (p + 1);
  hipLaunchKernelGGL(k_pows, dim3((threads + 255) / 256), dim3(256), 0, s, p, nc, moments, fact,
                     pows);
}

// f pre-pass (mac.rs:99-147) as a wave-coherent stackless walk. The lanes
// of a wave (64 / SUB consecutive slots, SUB lanes each) share one traversal
// pointer over the mirrored DFS (children 7..0, exactly the reference
// stack's pop order); a body that accepts a cell's monopole sleeps until the
// wave reaches that cell's rope, so each accumulates precisely its own
// reference sequence of terms, in order.
// Ensembles (vlev > 0): a body walks only its own system's subtree. A
// virtual cell (level < vlev) is opened by the bodies whose system it holds
// and skipped by the others; a real cell of another system is skipped; so
// every body meets its system's cells in the standalone order.
//
// A step is bound by the latency of the cell it moves to, so a cell is one
// 64-byte record (one scalar load; nine arrays before) and both candidates
// for the next step, the rope and the last child, are loaded before the
// current cell is computed. SUB = 4: four lanes take four consecutive bodies
// of a leaf and divide, then each adds the four terms in slot order (read
// from its neighbours by lane permutation), so the sequence is unchanged
// while the division, most of the arithmetic, is done once per four bodies,
// and there are four times as many, smaller waves.
// Measured: 1M bodies 3.93 -> 1.77 ms, 250k 1.12 -> 0.71, 16k 0.65 -> 0.24,
// 1k 0.235 -> 0.10.
struct __align__(64) FpRec {
  double cx, cy, cz, rho2, mass;
  int32_t rope, last;  // last: -1 in a leaf
  uint32_t first, count, level, pad;
};

__global__ void __launch_bounds__(256) k_pack_fp(uint32_t nc, DevCells c, FpRec* __restrict__ rec) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= nc) return;
  FpRec r;
  r.cx = c.cx[i];
  r.cy = c.cy[i];
  r.cz = c.cz[i];
  r.rho2 = c.rho[i] * c.rho[i];
  r.mass = c.mass[i];
  r.rope = c.rope[i];
  r.last = c.last_child[i];
  r.first = c.first[i];
  r.count = c.count[i];
  r.level = c.level[i];
  r.pad = 0;
  rec[i] = r;
}

// Value of lane (4 q + J) in every lane of quad q.
template <int J>
__device__ __forceinline__ double quad_read(double v) {
  const uint64_t u = (uint64_t)__double_as_longlong(v);
  constexpr int ctl = J * 0x55;  // quad_perm [J, J, J, J]
  const uint32_t lo =
      (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)u, ctl, 0xf, 0xf, true);
  const uint32_t hi =
      (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(u >> 32), ctl, 0xf, 0xf, true);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

template <int SUB>
__global__ void __launch_bounds__(64) k_fprepass(uint32_t n, uint32_t max_steps,
                                                const FpRec* __restrict__ rec,
                                                const double4* __restrict__ body,
                                                const uint64_t* __restrict__ keys_sorted, int vlev,
                                                double* __restrict__ f) {
  const int ACTIVE = -2, NEVER = -3;
  const uint32_t i = blockIdx.x * (64 / SUB) + threadIdx.x / SUB;
  const uint32_t sub = threadIdx.x % SUB;
  const bool valid = i < n;
  const int sh = 63 - 3 * vlev;
  const uint32_t mysys = (valid && vlev) ? (uint32_t)(keys_sorted[i] >> sh) : 0u;
  const double4 me = body[valid ? i : 0];
  const double px = me.x, py = me.y, pz = me.z;
  double fi = 0.0;
  int resume = valid ? ACTIVE : NEVER;
  int cur = 0;
  FpRec r = rec[0];
  // The mirrored DFS visits each cell at most once, so a wave needs at most
  // ncells steps; the cap only guards against a corrupt tree.
  for (uint32_t step = 0; step < max_steps; step++) {
    const int rope = wave_uniform(r.rope), last = wave_uniform(r.last);
    // both candidates for the next step, in flight while this one is computed
    const FpRec r_rope = rec[rope >= 0 ? rope : 0];
    const FpRec r_last = rec[last >= 0 ? last : 0];
    if (resume == cur) resume = ACTIVE;
    bool act = resume == ACTIVE;
    bool virt = false;
    if (vlev) {
      const uint32_t slo = (uint32_t)(keys_sorted[r.first] >> sh);
      virt = (int)r.level < vlev;
      if (act) {
        const uint32_t shi = virt ? (uint32_t)(keys_sorted[r.first + r.count - 1] >> sh) : slo;
        if (mysys < slo || mysys > shi) {  // not this body's system
          resume = rope;
          act = false;
        }
      }
    }
    bool open = false;
    if (last < 0) {
      const uint32_t f0 = r.first, e = f0 + r.count;
      if (SUB == 1) {
#pragma unroll 4
        for (uint32_t k = f0; k < e; k++) {
          const double4 q = body[k];
          const double dx = px - q.x, dy = py - q.y, dz = pz - q.z;
          const double r2 = dx * dx + dy * dy + dz * dz;
          if (act && k != i && r2 > 0.0) fi += q.w / r2;
        }
      } else {
        for (uint32_t k0 = f0; k0 < e; k0 += SUB) {
          const uint32_t k = k0 + sub;
          const double4 q = body[min(k, e - 1)];
          const double dx = px - q.x, dy = py - q.y, dz = pz - q.z;
          const double r2 = dx * dx + dy * dy + dz * dz;
          // an absent term is +0: fi + 0 is fi
          const double t = (act && k < e && k != i && r2 > 0.0) ? q.w / r2 : 0.0;
          fi += quad_read<0>(t);
          fi += quad_read<1>(t);
          fi += quad_read<2>(t);
          fi += quad_read<3>(t);
        }
      }
    } else if (act && virt) {
      open = true;  // a virtual cell on the way to the body's system root
    } else if (act) {
      const double dx = px - r.cx, dy = py - r.cy, dz = pz - r.cz;
      const double d2 = dx * dx + dy * dy + dz * dz;
      if (d2 > r.rho2) {
        fi += r.mass / d2;
        resume = rope;
      } else {
        open = true;
      }
    }
    const bool down = __ballot(open) != 0;
    cur = down ? last : rope;
    if (cur < 0) break;
    if (down)
      r = r_last;
    else
      r = r_rope;
  }
  if (valid && sub == 0) f[i] = fi;
}

// Four lanes per body while all those waves are resident at once (8192: 256
// CUs x 32); past that the extra waves only queue. SUB = 4 against 1: 1k 0.10
// and 0.21 ms, 16k 0.24 and 0.50, 250k 0.76 and 0.71, 1M 3.40 and 1.77.
constexpr uint32_t FP_SUB4_N = 8192 * 16;

size_t fp_rec_bytes() { return sizeof(FpRec); }

void launch_pack_fp(uint32_t nc, DevCells c, void* rec, hipStream_t s) {
  if (nc == 0) return;
  hipLaunchKernelGGL(k_pack_fp, dim3((nc + 255) / 256), dim3(256), 0, s, nc, c, (FpRec*)rec);
}

void launch_fprepass(uint32_t n, uint32_t nc, const void* rec, const double4* body,
                     const uint64_t* keys_sorted, int vlev, double* f, hipStream_t s) {
  if (n <= FP_SUB4_N)
    hipLaunchKernelGGL(k_fprepass<4>, dim3((n + 15) / 16), dim3(64), 0, s, n, nc + 1,
                       (const FpRec*)rec, body, keys_sorted, vlev, f);
  else
    hipLaunchKernelGGL(k_fprepass<1>, dim3((n + 63) / 64), dim3(64), 0, s, n, nc + 1,
                       (const FpRec*)rec, body, keys_sorted, vlev, f);
}

// fmin (mac.rs:151-173): the smallest f of a cell's bodies, which are one range
// of slots: minima of 64 and of 4096 slots first, then every cell from the ends
// of its range and the blocks between, in two launches for all levels (from the
// children's minima, it took one launch a level: 1M bodies 12 launches, 82 us,
// now 26; 1k bodies 7 launches, 32 us, now 10).
constexpr uint32_t FM = 64, FM2 = FM * FM;
size_t fmin_blocks_words(size_t n) { return (n + FM - 1) / FM + (n + FM2 - 1) / FM2; }

__global__ void __launch_bounds__(256) k_fmin_blocks(uint32_t n, const double* __restrict__ f,
                                                    double* __restrict__ b1,
                                                    double* __restrict__ b2) {
  __shared__ double sh[FM];
  const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  double v[FM / 4];
#pragma unroll
  for (uint32_t g = 0; g < FM / 4; g++) {
    const uint32_t i = blockIdx.x * FM2 + (w * (FM / 4) + g) * FM + lane;
    v[g] = i < n ? f[i] : INFINITY;
  }
#pragma unroll
  for (uint32_t g = 0; g < FM / 4; g++) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v[g] = fmin(v[g], __shfl_xor(v[g], o, 64));
    if (lane == 0) sh[w * (FM / 4) + g] = v[g];
  }
  __syncthreads();
  if (w != 0) return;
  double m = sh[lane];
  const uint32_t g = blockIdx.x * FM + lane;
  if ((size_t)g * FM < n) b1[g] = m;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmin(m, __shfl_xor(m, o, 64));
  if (lane == 0) b2[blockIdx.x] = m;
}

constexpr uint32_t FML = 16;  // lanes per cell
__global__ void __launch_bounds__(256) k_fmin(uint32_t nc, const uint32_t* __restrict__ first,
                                             const uint32_t* __restrict__ count,
                                             const double* __restrict__ f,
                                             const double* __restrict__ b1,
                                             const double* __restrict__ b2,
                                             double* __restrict__ fmin_out) {
  const uint32_t id = blockIdx.x * (256 / FML) + threadIdx.x / FML, l = threadIdx.x % FML;
  if (id >= nc) return;
  double m = INFINITY;
  auto range = [&](const double* v, uint32_t b, uint32_t e) {
#pragma unroll 4
    for (uint32_t k = b + l; k < e; k += FML) m = fmin(m, v[k]);
  };
  // [b, e) of a level: its ends, and the whole blocks between on the next
  auto ends = [&](const double* v, uint32_t& b, uint32_t& e) {
    const uint32_t bb = (b + FM - 1) / FM, be = e / FM;
    if (bb >= be) {
      range(v, b, e);
      b = e = 0;
      return;
    }
    range(v, b, bb * FM);
    range(v, be * FM, e);
    b = bb;
    e = be;
  };
  uint32_t b = first[id], e = b + count[id];
  ends(f, b, e);
  ends(b1, b, e);
  range(b2, b, e);
#pragma unroll
  for (int o = FML / 2; o > 0; o >>= 1) m = fmin(m, __shfl_xor(m, o, FML));
  if (l == 0) fmin_out[id] = m;
}

// blocks: scratch of fmin_blocks_words(n) doubles.
void launch_fmin(uint32_t n, uint32_t nc, DevCells c, const double* f, double* blocks, double* fmin,
                 hipStream_t s) {
  if (nc == 0) return;
  double* b2 = blocks + (n + FM - 1) / FM;
  hipLaunchKernelGGL(k_fmin_blocks, dim3((n + FM2 - 1) / FM2), dim3(256), 0, s, n, f, blocks, b2);
  hipLaunchKernelGGL(k_fmin, dim3((nc + 256 / FML - 1) / (256 / FML)), dim3(256), 0, s, nc, c.first,
                     c.count, f, (const double*)blocks, (const double*)b2, fmin);
}

}  // namespace fmmh
