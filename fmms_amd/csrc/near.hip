// near.hip — P2P near field on gfx950 (FP64 and mixed forms), fused with the
// final near + far sum and the slot -> particle-id scatter.
//
// Reference: crates/fmm p2p.rs:13-88 (mutual a_i += m_j d/r^3, a_j -= m_i
// d/r^3, pot += m/r) and translate.rs:339-342 (accel[id] += near + far).
// Here each target leaf owns its sums: one wave per work item (a leaf, or a
// slice of a heavy leaf's neighbour list) streams the item's source bodies
// (its own leaf included, self excluded by slot) through LDS in tiles of 64.
// The leaf's targets run as power-of-two chunks of n bodies with 64/n lanes
// per body, each lane on a strided share of every tile, combined by
// xor-shuffles at the end.
// Softening (an extension; 0 = the reference): r^2 += eps^2.
#include <algorithm>

#include "common.h"
#include "internal.h"
#include "m2l_chunk.h"

namespace fmmh {

constexpr uint32_t P2P_RMAX = 256;  // source ranges staged in LDS per pass

// P2P work items (uint4): x = target leaf | P2P_OWN when the item holds the
// leaf's own bodies as sources, [y, z) = its slice of the leaf's neighbour
// list, w = P2P_DIRECT (the item is the whole leaf: results go straight to
// accel / pot) or the offset of its partial sums (one double4 per target).
constexpr uint32_t P2P_OWN = 0x80000000u;
constexpr uint32_t P2P_FIRST = 0x40000000u;  // launched among the first blocks (longs)
constexpr uint32_t P2P_LEAF_MASK = 0x3fffffffu;
constexpr uint32_t P2P_DIRECT = 0xffffffffu;

// The source stream of one segment: the item's nonempty source ranges back to
// back, each as {stream position after it, slot - stream position in it}.
// A tile is 64 consecutive stream positions. Its lanes find their ranges
// together: 64 lanes look at the next 64 range ends and mark the lanes they
// fall on (a forward lane permutation), and a lane's range is the tile's first
// plus the marks up to it. The cost does not depend on the number of ranges;
// walking them one by one took 13 dependent steps a tile at 5 bodies a leaf
// (P2P of 1k bodies 44 us walked, 31 marked; of 1M at leaf capacity 16, 810
// and 660 us) and was no faster at 30 bodies a leaf.
struct StreamCursor {
  uint32_t at;   // range holding the next tile's first position
  uint32_t end;  // the lane's range end, ranges[at + lane].x
};

// The lane's body of the tile at `pos` (loaded, not waited on; past the
// stream's end any body: the caller pads).
__device__ __forceinline__ double4 gather_tile(const uint2* ranges, uint32_t nr, uint32_t total,
                                               uint32_t pos, StreamCursor& c, uint32_t lane,
                                               const double4* __restrict__ body) {
  const uint32_t e = c.at + lane < nr ? c.end - pos : 0xFFFFFFFFu;  // > 0: `at` holds pos
  // ends past the tile are sent to lane 0, where no range can end
  const int got = __builtin_amdgcn_ds_permute((int)(e < 64u ? e : 0u) * 4, 1);
  const uint64_t marks = __ballot(got == 1) & ~1ull;
  const uint32_t r = c.at + (uint32_t)__popcll(marks & (lanemask_lt() | (1ull << lane)));
  const uint32_t d = ranges[min(r, nr - 1)].y;
  c.at += (uint32_t)__popcll(__ballot(e <= 64u));
  c.end = ranges[min(c.at + lane, nr - 1)].x;  // for the next tile
  return body[pos + lane < total ? pos + lane + d : 0u];
}

// The two forms of the pairwise terms. FP64: absolute positions, the
// Newton-refined rsqrt. Mixed: float4 positions relative to the target
// leaf's centre (the subtraction done in FP64), the hardware FP32 rsqrt, and
// each tile's FP32 partial sums added into FP64 accumulators.
template <bool F32> struct P2PForm;
template <> struct P2PForm<false> {
  using T = double;
  using T4 = double4;
  static __device__ __forceinline__ double rsq(double x) { return rsqrt_pos(x); }
  static __device__ __forceinline__ double fmat(double a, double b, double c) {
    return __builtin_fma(a, b, c);
  }
  static __device__ __forceinline__ double4 stage(double4 v, double, double, double) { return v; }
};
template <> struct P2PForm<true> {
  using T = float;
  using T4 = float4;
  static __device__ __forceinline__ float rsq(float x) { return __builtin_amdgcn_rsqf(x); }
  static __device__ __forceinline__ float fmat(float a, float b, float c) {
    return __builtin_fmaf(a, b, c);
  }
  static __device__ __forceinline__ float4 stage(double4 v, double cx, double cy, double cz) {
    return make_float4((float)(v.x - cx), (float)(v.y - cy), (float)(v.z - cz), (float)v.w);
  }
};

// Bodies of a 64-entry LDS tile against the lane's target: the lane takes
// entries sub, sub + K, ... (ts = tile + sub), 64 / K of them. K is a
// template argument, so every lane runs the same trip count (no per-lane
// exit test) and the LDS reads take immediate offsets. Padding entries have
// mass 0 far away and contribute exactly 0. SELF: the entry at offset
// self_i (own slot - tile start - sub) is the target itself and is skipped.
template <bool F32, uint32_t K, bool SELF>
__device__ __forceinline__ void p2p_tile(const typename P2PForm<F32>::T4* __restrict__ ts,
                                         typename P2PForm<F32>::T xi, typename P2PForm<F32>::T yi,
                                         typename P2PForm<F32>::T zi,
                                         typename P2PForm<F32>::T soft2, int self_i,
                                         typename P2PForm<F32>::T& ax,
                                         typename P2PForm<F32>::T& ay,
                                         typename P2PForm<F32>::T& az,
                                         typename P2PForm<F32>::T& ph) {
  using F = P2PForm<F32>;
  using T = typename F::T;
  auto pair = [&](const auto sj, uint32_t i) {
    const T dx = sj.x - xi, dy = sj.y - yi, dz = sj.z - zi;
    T r2 = F::fmat(dx, dx, F::fmat(dy, dy, F::fmat(dz, dz, soft2)));
    T mj = sj.w;
    if (SELF) {
      const bool self = (int)(i * K) == self_i;
      r2 = self ? T(1) : r2;
      mj = self ? T(0) : mj;
    }
    // r2 is finite and > 0 here (softening, or distinct bodies, or padding)
    const T inv = F::rsq(r2);
    const T minv = mj * inv;
    const T s3 = minv * inv * inv;
    ax = F::fmat(s3, dx, ax);
    ay = F::fmat(s3, dy, ay);
    az = F::fmat(s3, dz, az);
    ph += minv;
  };
  if constexpr (F32) {  // 8 reads in flight per lane
#pragma unroll 8
    for (uint32_t i = 0; i < 64 / K; i++) pair(ts[i * K], i);
  } else {
    // four entries (twice the registers each) are read, then computed: the
    // scheduling barrier keeps the compiler from sinking each read to its use,
    // where the wave waits out the LDS latency once per entry (8.4M bodies:
    // 32.0 ms without, 30.6 with; eight entries 32.8)
    constexpr uint32_t N = 64 / K, U = N < 4 ? N : 4;
#pragma unroll 1
    for (uint32_t i0 = 0; i0 < N; i0 += U) {
      typename F::T4 e[U];
#pragma unroll
      for (uint32_t u = 0; u < U; u++) e[u] = ts[(i0 + u) * K];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (uint32_t u = 0; u < U; u++) pair(e[u], i0 + u);
    }
  }
}

// One chunk's pass over a staged tile: n targets (a power of two), 64 / n
// lanes per target, n iterations per lane.
template <bool F32, bool SELF>
__device__ __forceinline__ void p2p_chunk(const typename P2PForm<F32>::T4* __restrict__ tile,
                                          uint32_t n, uint32_t sub, typename P2PForm<F32>::T xi,
                                          typename P2PForm<F32>::T yi,
                                          typename P2PForm<F32>::T zi,
                                          typename P2PForm<F32>::T soft2, int self_i,
                                          typename P2PForm<F32>::T& ax,
                                          typename P2PForm<F32>::T& ay,
                                          typename P2PForm<F32>::T& az,
                                          typename P2PForm<F32>::T& ph) {
  const auto* ts = tile + sub;
  switch (n) {
    case 64: p2p_tile<F32, 1, SELF>(ts, xi, yi, zi, soft2, self_i, ax, ay, az, ph); break;
    case 32: p2p_tile<F32, 2, SELF>(ts, xi, yi, zi, soft2, self_i, ax, ay, az, ph); break;
    case 16: p2p_tile<F32, 4, SELF>(ts, xi, yi, zi, soft2, self_i, ax, ay, az, ph); break;
    case 8: p2p_tile<F32, 8, SELF>(ts, xi, yi, zi, soft2, self_i, ax, ay, az, ph); break;
    case 4: p2p_tile<F32, 16, SELF>(ts, xi, yi, zi, soft2, self_i, ax, ay, az, ph); break;
    case 2: p2p_tile<F32, 32, SELF>(ts, xi, yi, zi, soft2, self_i, ax, ay, az, ph); break;
    default: p2p_tile<F32, 64, SELF>(ts, xi, yi, zi, soft2, self_i, ax, ay, az, ph); break;
  }
}

// A group of r <= 64 targets of one leaf is cut into at most P2P_NQ chunks of
// power-of-two sizes n_q (64 / n_q lanes per target), all run on every
// staged source tile: a tile costs sum(n_q) iterations per lane, so a leaf
// of 37 bodies runs as 32 + 4 + 1 instead of one 64-target chunk with 27
// idle targets. The plan weighs the padding against a fixed cost per chunk
// and tile (its sums and loop set-up), in VALU issues.
constexpr int P2P_NQ = 3;
#ifndef FMMH_P2P_WAVES_F32
#define FMMH_P2P_WAVES_F32 5  // waves per SIMD the mixed-form P2P kernel is built for
#endif

__device__ __forceinline__ uint32_t pow2ceil(uint32_t x) {
  return x <= 1u ? 1u : 1u << (32 - __clz(x - 1u));
}
__device__ __forceinline__ uint32_t pow2floor(uint32_t x) { return 1u << (31 - __clz(x)); }

__device__ __forceinline__ void chunk_plan(uint32_t r, uint32_t (&n)[P2P_NQ]) {
  constexpr uint32_t IT = 14, CH = 12;  // per iteration, per chunk
  n[0] = pow2ceil(r);
  n[1] = n[2] = 0;
  uint32_t best = IT * n[0] + CH;
  const uint32_t a = pow2floor(r), ra = r - a;
  if (ra == 0) return;
  const uint32_t b2 = pow2ceil(ra);
  if (IT * (a + b2) + 2 * CH < best) {
    best = IT * (a + b2) + 2 * CH;
    n[0] = a;
    n[1] = b2;
  }
  const uint32_t b = pow2floor(ra), rb = ra - b;
  if (rb == 0) return;
  const uint32_t c = pow2ceil(rb);
  if (IT * (a + b + c) + 3 * CH < best) {
    n[0] = a;
    n[1] = b;
    n[2] = c;
  }
}

// Compensated FP64 accumulation (Knuth's TwoSum: s + v = t + e exactly, e
// kept in c): the mixed form's final per-body sums.
__device__ __forceinline__ void acc2(double& s, double& c, double v) {
  const double t = s + v;
  const double bp = t - s;
  c += (s - (t - bp)) + (v - bp);
  s = t;
}

// One segment of an item's source stream into LDS: the leaf's own bodies
// first when the stream starts with them, then each directed entry's source
// leaf (its slots), the own leaf's entry left out. Returns the stream length
// and the number of ranges. The barriers keep the previous pass's readers and
// this pass's readers apart.
__device__ __forceinline__ void stage_ranges(uint2* ranges, const uint64_t* __restrict__ skeys,
                                             uint64_t smask, const uint32_t* __restrict__ cfirst,
                                             const uint32_t* __restrict__ ccount, uint32_t ft,
                                             uint32_t nt_all, bool pre, uint32_t seg, uint32_t n,
                                             uint32_t lane, uint32_t* nr, uint32_t* total) {
  __syncthreads();
  uint32_t at = 0, len = 0;
  if (pre) {
    if (lane == 0) ranges[0] = make_uint2(nt_all, ft);
    at = 1;
    len = nt_all;
  }
  for (uint32_t q0 = 0; q0 < n; q0 += 64) {
    const uint32_t q = q0 + lane;
    uint32_t first = 0, c = 0;
    if (q < n) {
      const uint32_t src = (uint32_t)(skeys[seg + q] & smask);
      first = cfirst[src];
      c = first == ft ? 0u : ccount[src];
    }
    uint32_t sum;
    const uint32_t start = len + wave_excl_scan(c, &sum);
    const uint64_t full = __ballot(c > 0u);
    if (c > 0u) {
      const uint32_t k = at + (uint32_t)__popcll(full & lanemask_lt());
      ranges[k] = make_uint2(start + c, first - start);
    }
    at += (uint32_t)__popcll(full);
    len += sum;
  }
  *nr = (uint32_t)wave_uniform((int)at);
  *total = (uint32_t)wave_uniform((int)len);
  __syncthreads();
}

// One wave per work item. The targets of the item's leaf are taken in groups
// of 64, each group cut into chunks (chunk_plan); the item's source stream
// (the leaf's own bodies first when the item holds them, each target
// skipping its own slot there; then the neighbour leaves' ranges with the own
// leaf's entry emptied) is packed back to back into 64-body LDS tiles, and
// every chunk runs on every tile. The next tile's global loads are issued
// before the current one is computed. The mixed form (F32) sums each tile in
// FP32 and compensates the final sums (sub-lane partials, then the far field).
#define FMMH_P2P_PARAMS                                                                     \
  const uint4 *__restrict__ items, uint32_t nlong, const uint32_t *__restrict__ longs, const uint64_t *__restrict__ skeys, uint64_t smask,       \
      const uint32_t *__restrict__ cfirst, const uint32_t *__restrict__ ccount,               \
      const double *__restrict__ ccx, const double *__restrict__ ccy,                         \
      const double *__restrict__ ccz, const double4 *__restrict__ body, double soft2,         \
      const double4 *__restrict__ far, const uint32_t *__restrict__ order,                    \
      double *__restrict__ accel, double *__restrict__ pot, double4 *__restrict__ partial
#define FMMH_P2P_ARGS \
  items, nlong, longs, skeys, smask, cfirst, ccount, ccx, ccy, ccz, body, soft2, far, order,   \
      accel, pot, partial

template <bool F32>
__device__ __forceinline__ void p2p_item(FMMH_P2P_PARAMS) {
  using F = P2PForm<F32>;
  using T = typename F::T;
  __shared__ typename F::T4 tile[64];
  __shared__ uint2 ranges[P2P_RMAX + 1];
  const uint32_t lane = threadIdx.x;
  // the first nlong blocks take the long items, the others every item in
  // leaf order but those
  uint4 it;
  if (blockIdx.x < nlong) {
    it = items[longs[blockIdx.x]];
  } else {
    it = items[xcd_block(blockIdx.x - nlong, gridDim.x - nlong)];
    if (it.x & P2P_FIRST) return;
  }
  const uint32_t leaf = it.x & P2P_LEAF_MASK;
  const bool own = (it.x & P2P_OWN) != 0u;
  const uint32_t ft = cfirst[leaf], nt_all = ccount[leaf];
  const uint32_t jb = it.y, je = it.z;
  // the mixed form works relative to the leaf's centre; FP64 in place
  const double cx = F32 ? ccx[leaf] : 0.0, cy = F32 ? ccy[leaf] : 0.0,
               cz = F32 ? ccz[leaf] : 0.0;
  typename F::T4 pad;  // past the stream's end: far away and massless
  pad.x = pad.y = pad.z = T(1e18);
  pad.w = T(0);
  const T s2 = (T)soft2;
  const uint32_t nseg = (je - jb + P2P_RMAX - 1) / P2P_RMAX;
  uint32_t nr = 0, total = 0;
  for (uint32_t t0 = 0; t0 < nt_all; t0 += 64) {
    const uint32_t r = min(64u, nt_all - t0);
    uint32_t n[P2P_NQ];
    chunk_plan(r, n);
    // lane state per chunk: target index within the leaf (t0 + base + ti)
    // and the lane's strided share sub of each tile (64 / n lanes per target)
    uint32_t tix[P2P_NQ], sub[P2P_NQ];
    bool tval[P2P_NQ];
    T mx[P2P_NQ], my[P2P_NQ], mz[P2P_NQ];
    double ax[P2P_NQ], ay[P2P_NQ], az[P2P_NQ], ph[P2P_NQ];
    uint32_t base = 0;
#pragma unroll
    for (int q = 0; q < P2P_NQ; q++) {
      const uint32_t nq = n[q] ? n[q] : 1u;
      const uint32_t ti = lane & (nq - 1);
      sub[q] = lane / nq;
      tval[q] = n[q] != 0 && base + ti < r;
      tix[q] = t0 + base + ti;
      const auto me = F::stage(body[ft + (tval[q] ? tix[q] : 0)], cx, cy, cz);
      mx[q] = me.x;
      my[q] = me.y;
      mz[q] = me.z;
      ax[q] = ay[q] = az[q] = ph[q] = 0.0;
      base += n[q];
    }
    const uint32_t npass = max(nseg, own ? 1u : 0u);
    for (uint32_t sg = 0; sg < npass; sg++) {
      const uint32_t seg = jb + sg * P2P_RMAX;
      const uint32_t nseq = seg < je ? min(P2P_RMAX, je - seg) : 0u;
      const bool pre = own && sg == 0;  // stream starts with the own leaf
      // an item of one segment stages its ranges once, for every group
      if (nseg > 1 || t0 == 0)
        stage_ranges(ranges, skeys, smask, cfirst, ccount, ft, nt_all, pre, seg, nseq, lane, &nr,
                     &total);
      if (total == 0) continue;
      // the next tile's bodies are on their way while one is computed (padded
      // only when staged: a select on the loaded value would wait for it here)
      StreamCursor cur{0u, ranges[min(lane, nr - 1)].x};
      double4 next = gather_tile(ranges, nr, total, 0u, cur, lane, body);
      for (uint32_t pos = 0; pos < total; pos += 64) {
        tile[lane] = pos + lane < total ? F::stage(next, cx, cy, cz) : pad;
        __syncthreads();
        if (pos + 64 < total) next = gather_tile(ranges, nr, total, pos + 64, cur, lane, body);
        const bool self_tile = pre && pos < nt_all;
#pragma unroll
        for (int q = 0; q < P2P_NQ; q++) {
          if (n[q] == 0) break;
          const int self_i = (int)tix[q] - (int)pos - (int)sub[q];
          if constexpr (F32) {
            float fx = 0.f, fy = 0.f, fz = 0.f, fp = 0.f;
            if (self_tile)
              p2p_chunk<true, true>(tile, n[q], sub[q], mx[q], my[q], mz[q], s2, self_i, fx, fy,
                                    fz, fp);
            else
              p2p_chunk<true, false>(tile, n[q], sub[q], mx[q], my[q], mz[q], s2, 0, fx, fy, fz,
                                     fp);
            ax[q] += fx;
            ay[q] += fy;
            az[q] += fz;
            ph[q] += fp;
          } else {
            if (self_tile)
              p2p_chunk<false, true>(tile, n[q], sub[q], mx[q], my[q], mz[q], s2, self_i, ax[q],
                                     ay[q], az[q], ph[q]);
            else
              p2p_chunk<false, false>(tile, n[q], sub[q], mx[q], my[q], mz[q], s2, 0, ax[q],
                                      ay[q], az[q], ph[q]);
          }
        }
        __syncthreads();
      }
    }
#pragma unroll
    for (int q = 0; q < P2P_NQ; q++) {
      if (n[q] == 0) break;
      double kx = 0.0, ky = 0.0, kz = 0.0, kp = 0.0;
      for (uint32_t o = n[q]; o < 64; o <<= 1) {
        if constexpr (F32) {
          acc2(ax[q], kx, __shfl_xor(ax[q], (int)o, 64));
          acc2(ay[q], ky, __shfl_xor(ay[q], (int)o, 64));
          acc2(az[q], kz, __shfl_xor(az[q], (int)o, 64));
          acc2(ph[q], kp, __shfl_xor(ph[q], (int)o, 64));
          kx += __shfl_xor(kx, (int)o, 64);
          ky += __shfl_xor(ky, (int)o, 64);
          kz += __shfl_xor(kz, (int)o, 64);
          kp += __shfl_xor(kp, (int)o, 64);
        } else {
          ax[q] += __shfl_xor(ax[q], (int)o, 64);
          ay[q] += __shfl_xor(ay[q], (int)o, 64);
          az[q] += __shfl_xor(az[q], (int)o, 64);
          ph[q] += __shfl_xor(ph[q], (int)o, 64);
        }
      }
      if (sub[q] == 0 && tval[q]) {
        const uint32_t si = ft + tix[q];
        if (it.w == P2P_DIRECT) {  // the final near + far sum
          const double4 fv = far[si];
          const uint32_t id = order[si];
          if constexpr (F32) {
            acc2(ax[q], kx, fv.x);
            acc2(ay[q], ky, fv.y);
            acc2(az[q], kz, fv.z);
            acc2(ph[q], kp, fv.w);
          } else {
            ax[q] += fv.x;
            ay[q] += fv.y;
            az[q] += fv.z;
            ph[q] += fv.w;
          }
          accel[3 * (size_t)id] = ax[q] + kx;
          accel[3 * (size_t)id + 1] = ay[q] + ky;
          accel[3 * (size_t)id + 2] = az[q] + kz;
          if (pot) pot[id] = ph[q] + kp;
        } else {
          partial[(size_t)it.w + tix[q]] =
              make_double4(ax[q] + kx, ay[q] + ky, az[q] + kz, ph[q] + kp);
        }
      }
    }
  }
}

// The two forms as kernels of their own, each with the occupancy that
// measured fastest: the mixed form at five waves per SIMD (at most 102 VGPRs:
// the unrolled tile loop keeps fewer reads in flight, and the extra wave
// hides more of the tile staging), FP64 at the compiler's choice.
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(FMMH_P2P_WAVES_F32)))
k_p2p_mixed(FMMH_P2P_PARAMS) {
  p2p_item<true>(FMMH_P2P_ARGS);
}

__global__ void __launch_bounds__(64) k_p2p_fp64(FMMH_P2P_PARAMS) {
  p2p_item<false>(FMMH_P2P_ARGS);
}

// ------------------------------------------------------- the lists' work plan
// M2L: a target's sources in chunks of at most `ch`. P2P: a leaf's work is its
// target count times its source bodies (own leaf plus neighbour leaves). One
// block per leaf leaves the whole device waiting on the few leaves whose
// neighbourhoods are huge (a large sparse leaf beside a dense region), so a
// leaf is cut into m work items (at most one per source unit): m = work / W
// where the work exceeds the context's item bound W (fmmh_tuning.p2p_item_work,
// default 2^18), and in the FP64 form, up to that default, at least one item per
// P2P_CAP sources; a caller who asks for longer items gets them.
// Source units are the own leaf (unit 0) and the neighbour ranges in list
// order; unit u with P_u sources before it goes to item
// min(m - 1, P_u / ceil(S / m)) (items may come out empty). Split items write
// partial sums that k_p2p_reduce adds in item order. The cut depends on the
// leaf's own counts only, so a system evaluates the same alone and in an
// ensemble (unless a memory budget has left the cap out for one of the two).
//
// P2P_CAP: an item is one wave streaming its sources tile by tile, about 1.4
// us per 64 sources however few the targets are, so a leaf of 10 bodies with
// 26000 sources (2^18 pairs, one item) ran for 600 us: all of the near field's
// time at 16k and at 100k bodies. P2P with no cap, 8192, 6144 and 4096 sources:
// 100k bodies 414, 303, 247 and 243 us, 16k 620 (no cap), 182, 124 and 95; at
// 8.4M bodies (4485 sources a leaf) 4096 costs 0.3 of 30.4 ms against no cap.
// The mixed form keeps its items (their tiles are what its FP32 sums are
// grouped by). In both forms the long items (over P2P_LONG64 / P2P_LONG32
// sources), which would otherwise start wherever their leaf comes and end last,
// are launched first, where they are few (by index, in no particular order: an
// item's results do not depend on when it runs): 100k bodies 382 -> 267 us,
// mixed ensemble of 1.5M bodies 4.39 -> 4.13 ms.
constexpr int PLAN_T = 256;
constexpr uint32_t P2P_LONG64 = 2048, P2P_LONG32 = 8192;
constexpr uint32_t PLAN_SHORT = 32;  // a list of so few neighbours is never a long one

__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

struct LeafCut {
  uint32_t leaf, nt, jb, je;
  uint32_t S, m;  // sources (distinct bodies, so below 2^32), items
};

// How a form's leaves are cut: work per item, sources per item, and the
// sources from which an item counts as long.
struct CutRule {
  uint64_t W;
  uint32_t cap, lng;
};

// Source total and item count of a leaf (all lanes get the result).
__device__ __forceinline__ LeafCut leaf_cut(uint32_t leaf, const uint32_t* __restrict__ pptr,
                                            const uint64_t* __restrict__ skeys, uint64_t smask,
                                            const uint32_t* __restrict__ ccount, CutRule cut,
                                            uint32_t lane) {
  LeafCut L;
  L.leaf = leaf;
  L.nt = ccount[leaf];
  L.jb = pptr[leaf];
  L.je = pptr[leaf + 1];
  uint32_t s = 0;
#pragma unroll 4
  for (uint32_t j = L.jb + lane; j < L.je; j += 64) {
    const uint32_t src = (uint32_t)(skeys[j] & smask);
    s += src == leaf ? 0u : ccount[src];
  }
  L.S = L.nt + wave_sum_u32(s);
  const uint64_t work = (uint64_t)L.nt * L.S;
  uint64_t m = work > cut.W ? (work + cut.W - 1) / cut.W : 1;
  if (L.S > cut.cap) m = max(m, (uint64_t)((L.S - 1) / cut.cap + 1));
  const uint64_t units = (uint64_t)(L.je - L.jb) + 1;
  L.m = (uint32_t)min(m, units);
  return L;
}

// Whether a leaf's items are launched first.
__device__ __forceinline__ bool long_items(const LeafCut& L, CutRule cut) {
  return L.je - L.jb > PLAN_SHORT && L.S / L.m > cut.lng;
}

// {M2L chunks, P2P items, partial-sum slots, cut leaves} of cell t in plan[t];
// plan[nc] = 0 closes the scan and plan[nc + 1].x counts the long items. One
// wave per cell at a time, at most PLAN_BLOCKS blocks, each adding its long
// items at once: one addition per long leaf serialised on that word (2.6 ms
// at 280k leaves).
constexpr uint32_t PLAN_BLOCKS = 2048;

__global__ void __launch_bounds__(PLAN_T) k_plan_count(
    uint32_t nc, const uint8_t* __restrict__ leaf, const uint32_t* __restrict__ tptr, uint32_t ch,
    const uint32_t* __restrict__ pptr, const uint64_t* __restrict__ skeys, uint64_t smask,
    const uint32_t* __restrict__ ccount, CutRule cut, uint4* __restrict__ plan) {
  __shared__ uint32_t lng[PLAN_T / 64];
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  uint32_t nl = 0;
  for (uint32_t t = blockIdx.x * (PLAN_T / 64) + wave; t <= nc; t += gridDim.x * (PLAN_T / 64)) {
    uint4 v = make_uint4(0u, 0u, 0u, 0u);
    if (t < nc) {
      v.x = (tptr[t + 1] - tptr[t] + ch - 1) / ch;
      if (leaf[t]) {
        const LeafCut L = leaf_cut(t, pptr, skeys, smask, ccount, cut, lane);
        v.y = L.m;
        v.z = L.m > 1 ? L.m * L.nt : 0u;
        v.w = L.m > 1 ? 1u : 0u;
        if (long_items(L, cut)) nl += L.m;
      }
    }
    if (lane == 0) plan[t] = v;
  }
  if (lane == 0) lng[wave] = nl;
  __syncthreads();
  if (threadIdx.x == 0) {
    nl = 0;
    for (int w = 0; w < PLAN_T / 64; w++) nl += lng[w];
    if (nl) atomicAdd(&plan[nc + 1].x, nl);
  }
}

// Cell t by one wave; plan: the scanned counts. Writes the chunks, the items, the
// records of cut leaves and, unless nlong is null, the indices of the long items
// (their slots counted in *nlong).
__device__ __forceinline__ void plan_emit_cell(
    uint32_t t, uint32_t lane, const uint8_t* __restrict__ leaf, const uint32_t* __restrict__ tptr,
    uint32_t ch, const uint32_t* __restrict__ pptr, const uint64_t* __restrict__ skeys,
    uint64_t smask, const uint32_t* __restrict__ ccount, CutRule cut,
    const uint4* __restrict__ plan, M2lChunk* __restrict__ chunks, uint4* __restrict__ items,
    uint4* __restrict__ reds, uint32_t* __restrict__ nlong, uint32_t* __restrict__ longs) {
  const uint4 at = plan[t];
  {
    const uint32_t b = tptr[t], e = tptr[t + 1];
    for (uint32_t k = lane; b + k * ch < e; k += 64)
      chunks[at.x + k] = M2lChunk{t, b + k * ch, min(e, b + (k + 1) * ch)};
  }
  if (!leaf[t]) return;
  const uint32_t base = at.y;
  const uint32_t m = plan[t + 1].y - base;
  // one item: the whole list, not read again
  if (m == 1 && (!nlong || pptr[t + 1] - pptr[t] <= PLAN_SHORT)) {
    if (lane == 0) items[base] = make_uint4(t | P2P_OWN, pptr[t], pptr[t + 1], P2P_DIRECT);
    return;
  }
  const LeafCut L = leaf_cut(t, pptr, skeys, smask, ccount, cut, lane);
  const bool lng = nlong && long_items(L, cut);
  const uint32_t mark = lng ? P2P_FIRST : 0u;
  if (lng) {
    uint32_t w = 0;
    if (lane == 0) w = atomicAdd(nlong, m);
    w = (uint32_t)__shfl((int)w, 0, 64);
    for (uint32_t k = lane; k < m; k += 64) longs[w + k] = base + k;
  }
  uint32_t* it = (uint32_t*)(items + base);  // [m][4]: leaf|own, begin, end, slot
  for (uint32_t k = lane; k < m; k += 64) {
    it[4 * k] = L.leaf | mark | (k == 0 ? P2P_OWN : 0u);
    it[4 * k + 3] = m > 1 ? at.z + k * L.nt : P2P_DIRECT;
  }
  if (lane == 0) {
    it[1] = L.jb;
    if (m > 1) reds[at.w] = make_uint4(L.leaf, at.z, m, 0u);
  }
  // item boundaries: where the unit's item index steps up
  const uint32_t T = (L.S - 1) / m + 1;
  uint32_t running = L.nt;  // sources before the first neighbour unit
  uint32_t gprev = 0;       // item of unit 0 (the own leaf)
  // PU consecutive units a lane, the following ones' counts loaded ahead: the
  // longest leaf's chain of such steps bounds the launch (100k bodies, one unit a
  // lane 102 us, four 66)
  constexpr uint32_t PU = 4;
  auto units = [&](uint32_t j0, uint32_t* cnt) {
    uint32_t src[PU];
#pragma unroll
    for (uint32_t u = 0; u < PU; u++)
      src[u] = j0 + u < L.je ? (uint32_t)(skeys[j0 + u] & smask) : L.leaf;
#pragma unroll
    for (uint32_t u = 0; u < PU; u++) cnt[u] = src[u] == L.leaf ? 0u : ccount[src[u]];
  };
  uint32_t next[PU];
  units(L.jb + PU * lane, next);
  for (uint32_t c0 = L.jb; m > 1 && c0 < L.je; c0 += 64 * PU) {
    const uint32_t j = c0 + PU * lane;
    uint32_t cnt[PU], own = 0u;
#pragma unroll
    for (uint32_t u = 0; u < PU; u++) {
      cnt[u] = next[u];
      own += cnt[u];
    }
    units(j + 64 * PU, next);
    uint32_t incl = own;  // inclusive wave scan
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t v = __shfl_up(incl, o, 64);
      if ((int)lane >= o) incl += v;
    }
    uint32_t P = running + incl - own;
    uint32_t g[PU], glast = 0u;  // of the lane's last valid unit
#pragma unroll
    for (uint32_t u = 0; u < PU; u++) {
      g[u] = min(P / T, m - 1);
      if (j + u < L.je) glast = g[u];
      P += cnt[u];
    }
    const uint32_t gl = (uint32_t)__shfl_up(glast, 1, 64);
    uint32_t before = lane == 0 ? gprev : gl;
#pragma unroll
    for (uint32_t u = 0; u < PU; u++) {
      if (j + u >= L.je) break;
      for (uint32_t k = before + 1; k <= g[u]; k++) {
        it[4 * k + 1] = j + u;
        it[4 * (k - 1) + 2] = j + u;
      }
      before = g[u];
    }
    const uint32_t last = min(63u, (L.je - 1 - c0) / PU);  // last lane with a unit
    gprev = (uint32_t)__shfl(glast, (int)last, 64);
    running += __shfl(incl, 63, 64);
  }
  // items after the last unit's item are empty; the last item ends the list
  for (uint32_t k = gprev + lane; k < m; k += 64) {
    if (k > gprev) it[4 * k + 1] = L.je;
    it[4 * k + 2] = L.je;
  }
}

__global__ void __launch_bounds__(PLAN_T) k_plan_emit(
    uint32_t nc, const uint8_t* __restrict__ leaf, const uint32_t* __restrict__ tptr, uint32_t ch,
    const uint32_t* __restrict__ pptr, const uint64_t* __restrict__ skeys, uint64_t smask,
    const uint32_t* __restrict__ ccount, CutRule cut, const uint4* __restrict__ plan,
    M2lChunk* __restrict__ chunks, uint4* __restrict__ items, uint4* __restrict__ reds,
    uint32_t* __restrict__ nlong, uint32_t* __restrict__ longs) {
  const uint32_t lane = threadIdx.x & 63;
  for (uint32_t t = blockIdx.x * (PLAN_T / 64) + (threadIdx.x >> 6); t < nc;
       t += gridDim.x * (PLAN_T / 64))
    plan_emit_cell(t, lane, leaf, tptr, ch, pptr, skeys, smask, ccount, cut, plan, chunks, items, reds,
                   nlong, longs);
}

// Split leaves: far field + the items' partial sums in item order, scattered
// to particle-id order.
// COMP (the mixed form): the item sums and the far field are added with
// compensated (TwoSum) accumulation.
template <bool COMP>
__global__ void __launch_bounds__(64) k_p2p_reduce(const uint4* __restrict__ reds,
                                                  const uint32_t* __restrict__ cfirst,
                                                  const uint32_t* __restrict__ ccount,
                                                  const double4* __restrict__ partial,
                                                  const double4* __restrict__ far,
                                                  const uint32_t* __restrict__ order,
                                                  double* __restrict__ accel,
                                                  double* __restrict__ pot) {
  const uint4 r = reds[blockIdx.x];
  const uint32_t ft = cfirst[r.x], nt = ccount[r.x];
  for (uint32_t t = threadIdx.x; t < nt; t += 64) {
    double ax = 0.0, ay = 0.0, az = 0.0, ph = 0.0;
    double kx = 0.0, ky = 0.0, kz = 0.0, kp = 0.0;
    for (uint32_t k = 0; k <= r.z; k++) {  // the items in order, then the far field
      const double4 v = k < r.z ? partial[(size_t)r.y + (size_t)k * nt + t] : far[ft + t];
      if (COMP) {
        acc2(ax, kx, v.x);
        acc2(ay, ky, v.y);
        acc2(az, kz, v.z);
        acc2(ph, kp, v.w);
      } else {
        ax += v.x;
        ay += v.y;
        az += v.z;
        ph += v.w;
      }
    }
    const uint32_t id = order[ft + t];
    accel[3 * (size_t)id] = ax + kx;
    accel[3 * (size_t)id + 1] = ay + ky;
    accel[3 * (size_t)id + 2] = az + kz;
    if (pot) pot[id] = ph + kp;
  }
}

static CutRule cut_rule(uint64_t item_work, uint32_t cap, bool fp32) {
  return CutRule{item_work, cap, fp32 ? P2P_LONG32 : P2P_LONG64};
}

// plan: nc + 2 entries, zeroed at [nc + 1] by the caller; scanned by the
// caller between the two.
void plan_count(uint32_t nc, DevCells c, const uint32_t* tptr, uint32_t ch, const uint32_t* pptr,
                const uint64_t* skeys, int sbits, uint64_t item_work, uint32_t cap, bool fp32,
                uint4* plan, hipStream_t s) {
  const uint32_t nb = std::min(PLAN_BLOCKS, (nc + 1 + PLAN_T / 64 - 1) / (PLAN_T / 64));
  hipLaunchKernelGGL(k_plan_count, dim3(nb), dim3(PLAN_T), 0, s, nc, c.leaf, tptr, ch, pptr, skeys, (1ull << sbits) - 1ull, c.count,
                     cut_rule(item_work, cap, fp32), plan);
}

void plan_emit(uint32_t nc, DevCells c, const uint32_t* tptr, uint32_t ch, const uint32_t* pptr,
               const uint64_t* skeys, int sbits, uint64_t item_work, uint32_t cap, bool fp32,
               const uint4* plan, void* chunks, uint4* items, uint4* reds, uint32_t* nlong,
               uint32_t* longs, hipStream_t s) {
  // a launch holds fewer than 2^32 threads: past 2^23 blocks (34M cells) a wave
  // takes several cells
  const uint32_t nb = std::min(1u << 23, (nc + PLAN_T / 64 - 1) / (PLAN_T / 64));
  hipLaunchKernelGGL(k_plan_emit, dim3(nb), dim3(PLAN_T), 0, s,
                     nc, c.leaf, tptr, ch, pptr, skeys, (1ull << sbits) - 1ull, c.count,
                     cut_rule(item_work, cap, fp32), plan, (M2lChunk*)chunks, items, reds, nlong, longs);
}

void launch_p2p_f32(const P2PPlan& pl, DevCells c, const double4* body, const uint64_t* skeys,
                    int sbits, double soft2, const double4* far, const uint32_t* order,
                    double* accel, double* pot, hipStream_t s) {
  if (pl.nitems == 0) return;
  const uint64_t smask = (1ull << sbits) - 1ull;
  hipLaunchKernelGGL(k_p2p_mixed, dim3(pl.nitems + pl.nlong),
                     dim3(64), 0, s, pl.items, pl.nlong, pl.longs, skeys, smask, c.first,
                     c.count, c.cx, c.cy, c.cz, body, soft2, far, order, accel, pot, pl.partial);
}

void launch_p2p_reduce(const P2PPlan& pl, DevCells c, const double4* far, const uint32_t* order,
                       double* accel, double* pot, bool compensated, hipStream_t s) {
  if (pl.nitems == 0 || pl.nsplit == 0) return;
  if (compensated)
    hipLaunchKernelGGL(k_p2p_reduce<true>, dim3(pl.nsplit), dim3(64), 0, s, pl.reds, c.first,
                       c.count, pl.partial, far, order, accel, pot);
  else
    hipLaunchKernelGGL(k_p2p_reduce<false>, dim3(pl.nsplit), dim3(64), 0, s, pl.reds, c.first,
                       c.count, pl.partial, far, order, accel, pot);
}

void launch_p2p(const P2PPlan& pl, DevCells c, const double4* body, const uint64_t* skeys,
                int sbits, double soft2, const double4* far, const uint32_t* order, double* accel,
                double* pot, hipStream_t s) {
  if (pl.nitems == 0) return;
  const uint64_t smask = (1ull << sbits) - 1ull;
  hipLaunchKernelGGL(k_p2p_fp64, dim3(pl.nitems + pl.nlong),
                     dim3(64), 0, s, pl.items, pl.nlong, pl.longs, skeys, smask, c.first,
                     c.count, c.cx, c.cy, c.cz, body, soft2, far, order, accel, pot, pl.partial);
}

__global__ void __launch_bounds__(256) k_p2p_count(const uint2* __restrict__ pairs, uint32_t np,
                                                  const uint32_t* __restrict__ count,
                                                  unsigned long long* __restrict__ part) {
  __shared__ unsigned long long sh[4];
  uint32_t i = blockIdx.x * 256 + threadIdx.x;
  unsigned long long v = 0;
  if (i < np) {
    uint2 pr = pairs[i];
    unsigned long long ca = count[pr.x], cb = count[pr.y];
    v = pr.x == pr.y ? ca * (ca - 1) : 2 * ca * cb;
  }
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
}

__global__ void __launch_bounds__(256) k_sum_u64(const unsigned long long* __restrict__ part,
                                                uint32_t np, unsigned long long* __restrict__ out) {
  __shared__ unsigned long long sh[4];
  unsigned long long v = 0;
  for (uint32_t i = threadIdx.x; i < np; i += 256) v += part[i];
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) *out = sh[0] + sh[1] + sh[2] + sh[3];
}

size_t p2p_count_scratch(uint32_t np) { return ((size_t)np + 255) / 256 + 1; }

// out[0] = total; out[1..] scratch of p2p_count_scratch(np) words.
void launch_p2p_count(const uint2* pairs, uint32_t np, const uint32_t* count,
                      unsigned long long* out, hipStream_t s) {
  uint32_t nb = (np + 255) / 256;
  if (nb)
    hipLaunchKernelGGL(k_p2p_count, dim3(nb), dim3(256), 0, s, pairs, np, count, out + 1);
  hipLaunchKernelGGL(k_sum_u64, dim3(1), dim3(256), 0, s, out + 1, nb, out);
}

}  // namespace fmmh
