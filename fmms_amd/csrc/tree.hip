// tree.hip — Morton-key octree build on gfx950 (compiled -ffp-contract=off).
//
// Follows crates/fmm tree.rs:94-227 and reproduces its output bit for bit:
//   bbox (min/max, order-free) -> 63-bit Morton keys with the reference's
//   quantiser (every axis measured from the x minimum, tree.rs:37-46) ->
//   stable LSD radix sort (prims.hip) -> cells straight from the sorted keys
//   -> geometry in the reference's arithmetic order.
//
// The cells need no recursion and no level-by-level pass. A cell is a run of
// slots sharing a key prefix, and the cells starting at one slot are a
// parent -> first-child chain over consecutive levels, from the level at
// which the slot parts from its predecessor to the first level that is not
// split; a cell splits when it holds more than n_leaf bodies, which for the
// chain is a comparison with the key n_leaf slots on. DFS preorder sorts
// cells by (first slot, level), so a cell's id is the number of cells whose
// range starts before its slot (an exclusive scan of the chain lengths) plus
// its position in the chain. One host read (the counts per level) replaces
// one per level: 100k bodies 36 launches and 10 reads -> 7 and 1.
#include <algorithm>

#include "common.h"
#include "internal.h"

namespace fmmh {

constexpr int BITS = 21;  // tree.rs:16
constexpr int TB = 256;
constexpr uint32_t BBOX_BLOCKS = 1024;

// Minima and maxima of the block's threads; thread 0 returns them.
__device__ __forceinline__ void bbox_block(double lo[3], double hi[3]) {
  __shared__ double sh[6][TB];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    sh[d][threadIdx.x] = lo[d];
    sh[3 + d][threadIdx.x] = hi[d];
  }
  __syncthreads();
  for (int st = TB / 2; st > 0; st >>= 1) {
    if (threadIdx.x < st) {
#pragma unroll
      for (int d = 0; d < 3; d++) {
        sh[d][threadIdx.x] = fmin(sh[d][threadIdx.x], sh[d][threadIdx.x + st]);
        sh[3 + d][threadIdx.x] = fmax(sh[3 + d][threadIdx.x], sh[3 + d][threadIdx.x + st]);
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int d = 0; d < 3; d++) {
    lo[d] = sh[d][0];
    hi[d] = sh[3 + d][0];
  }
}

// tree.rs:99-111: side = max extent (at least f64::MIN_POSITIVE), inv = 1/side.
__device__ __forceinline__ void bbox_write(const double lo[3], const double hi[3], BBox* out) {
  double side = fmax(fmax(fmax(hi[0] - lo[0], hi[1] - lo[1]), hi[2] - lo[2]), 2.2250738585072014e-308);
  for (int d = 0; d < 3; d++) {
    out->lo[d] = lo[d];
    out->hi[d] = hi[d];
  }
  out->side = side;
  out->inv_side = 1.0 / side;
}

// nb blocks per system reduce its body range [off[s], off[s+1]) (one system: off
// null, [0, n)); a system's only block writes its box.
__global__ void __launch_bounds__(TB) k_bbox_partial(const double* __restrict__ pos, size_t n,
                                                    const uint64_t* __restrict__ off, uint32_t nb,
                                                    double* __restrict__ partial,
                                                    BBox* __restrict__ out) {
  const uint32_t sys = blockIdx.x / nb, k = blockIdx.x - sys * nb;
  const size_t b = off ? off[sys] : 0, e = off ? off[sys + 1] : n;
  double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (size_t i = b + (size_t)k * TB + threadIdx.x; i < e; i += (size_t)nb * TB) {
#pragma unroll
    for (int d = 0; d < 3; d++) {
      double v = pos[3 * i + d];
      lo[d] = fmin(lo[d], v);
      hi[d] = fmax(hi[d], v);
    }
  }
  bbox_block(lo, hi);
  if (threadIdx.x != 0) return;
  if (nb == 1) {
    bbox_write(lo, hi, out + sys);
    return;
  }
  double* o = partial + (size_t)blockIdx.x * 6;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    o[d] = lo[d];
    o[3 + d] = hi[d];
  }
}

__global__ void __launch_bounds__(TB) k_bbox_final(const double* __restrict__ partial, uint32_t nb,
                                                  BBox* __restrict__ out) {
  const double* pt = partial + (size_t)blockIdx.x * nb * 6;
  double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (uint32_t b = threadIdx.x; b < nb; b += TB)
    for (int d = 0; d < 3; d++) {
      lo[d] = fmin(lo[d], pt[6 * b + d]);
      hi[d] = fmax(hi[d], pt[6 * b + 3 + d]);
    }
  bbox_block(lo, hi);
  if (threadIdx.x == 0) bbox_write(lo, hi, out + blockIdx.x);
}

// Blocks per system: BBOX_BLOCKS in all, each with a body a thread at least on
// average. One block per system left most of the chip idle: 48 systems of 31k
// bodies 291 -> 21 + 5 us. Minima and maxima do not depend on the split.
static uint32_t bbox_blocks(size_t n, uint32_t nsys) {
  const size_t most = std::max<size_t>(1, BBOX_BLOCKS / nsys);
  return (uint32_t)std::min(most, std::max<size_t>(1, (n / nsys + TB - 1) / TB));
}

size_t bbox_partial_bytes(size_t n, uint32_t nsys) {
  const uint32_t nb = bbox_blocks(n, nsys);
  return nb > 1 ? (size_t)6 * nsys * nb * sizeof(double) : 0;  // a system's only block keeps none
}

void launch_bbox(const double* pos, size_t n, const uint64_t* off, uint32_t nsys, double* partial,
                 BBox* out, hipStream_t s) {
  const uint32_t nb = bbox_blocks(n, nsys);
  hipLaunchKernelGGL(k_bbox_partial, dim3(nsys * nb), dim3(TB), 0, s, pos, n, off, nb, partial, out);
  if (nb > 1) hipLaunchKernelGGL(k_bbox_final, dim3(nsys), dim3(TB), 0, s, partial, nb, out);
}

// Spread the low 21 bits of x to every third bit (tree.rs:28-35).
__device__ __forceinline__ uint64_t dilate21(uint64_t x) {
  x &= (1ull << BITS) - 1;
  x = (x | (x << 32)) & 0x001f00000000ffffull;
  x = (x | (x << 16)) & 0x001f0000ff0000ffull;
  x = (x | (x << 8)) & 0x100f00f00f00f00full;
  x = (x | (x << 4)) & 0x10c30c30c30c30c3ull;
  return (x | (x << 2)) & 0x1249249249249249ull;
}

// tree.rs:37-46: clamp((c - lo[0]) * inv_side, 0, 1) * (2^21-1), truncated;
// NaN keeps through the clamp and converts to 0.
__device__ __forceinline__ uint64_t quantise(double c, double lo0, double inv_side) {
  double v = (c - lo0) * inv_side;
  if (v < 0.0) v = 0.0;
  if (v > 1.0) v = 1.0;
  double w = v * 2097151.0;
  if (!(w == w)) return 0;
  return (uint64_t)w;
}

__global__ void __launch_bounds__(TB) k_keys(const double* __restrict__ pos,
                                            const double* __restrict__ mass, size_t n,
                                            const BBox* __restrict__ bb,
                                            uint64_t* __restrict__ keys,
                                            uint32_t* __restrict__ vals,
                                            uint32_t* __restrict__ flags,
                                            double4* __restrict__ pk) {
  size_t i = (size_t)blockIdx.x * TB + threadIdx.x;
  if (i >= n) return;
  const double lo0 = bb->lo[0], inv = bb->inv_side;
  double x = pos[3 * i], y = pos[3 * i + 1], z = pos[3 * i + 2], m = mass[i];
  uint64_t key = dilate21(quantise(z, lo0, inv));
  key |= dilate21(quantise(y, lo0, inv)) << 1;
  key |= dilate21(quantise(x, lo0, inv)) << 2;
  keys[i] = key;
  vals[i] = (uint32_t)i;
  pk[i] = make_double4(x, y, z, m);
  if (!(isfinite(x) && isfinite(y) && isfinite(z) && isfinite(m))) atomicOr(flags, 1u);
}

__device__ __forceinline__ uint32_t system_of(const uint64_t* __restrict__ off, uint32_t nsys,
                                              uint64_t i) {
  uint32_t lo = 0, hi = nsys;  // off[lo] <= i < off[lo + 1]
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (off[mid] <= i)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

// Ensemble keys, first half: the body's Morton key within its own system's
// box (its standalone key). The bodies are sorted by these keys first, so
// bodies whose keys agree above the low 3V bits keep their standalone order.
__global__ void __launch_bounds__(TB) k_keys_sys(const double* __restrict__ pos,
                                                const double* __restrict__ mass, size_t n,
                                                const uint64_t* __restrict__ off, uint32_t nsys,
                                                int vlev, const BBox* __restrict__ bbs,
                                                uint64_t* __restrict__ keys,
                                                uint32_t* __restrict__ vals,
                                                uint32_t* __restrict__ flags,
                                                double4* __restrict__ pk) {
  size_t i = (size_t)blockIdx.x * TB + threadIdx.x;
  if (i >= n) return;
  const BBox* bb = bbs + system_of(off, nsys, i);
  const double lo0 = bb->lo[0], inv = bb->inv_side;
  double x = pos[3 * i], y = pos[3 * i + 1], z = pos[3 * i + 2], m = mass[i];
  uint64_t key = dilate21(quantise(z, lo0, inv));
  key |= dilate21(quantise(y, lo0, inv)) << 1;
  key |= dilate21(quantise(x, lo0, inv)) << 2;
  keys[i] = key;
  vals[i] = (uint32_t)i;
  pk[i] = make_double4(x, y, z, m);
  if (!(isfinite(x) && isfinite(y) && isfinite(z) && isfinite(m))) atomicOr(flags, 1u);
}

// Ensemble keys, second half (on the bodies sorted by standalone key): the
// standalone key with its low 3V bits dropped, under a 3V-bit system prefix
// (V virtual levels, nsys <= 8^V). A stable sort on the prefix bits then
// orders the bodies by (system, standalone key), and below level V the
// forest splits exactly like each system's standalone tree.
__global__ void __launch_bounds__(TB) k_keys_prefix(uint64_t* __restrict__ keys,
                                                   const uint32_t* __restrict__ ids, size_t n,
                                                   const uint64_t* __restrict__ off, uint32_t nsys,
                                                   int vlev) {
  size_t k = (size_t)blockIdx.x * TB + threadIdx.x;
  if (k >= n) return;
  const uint32_t sys = system_of(off, nsys, ids[k]);
  keys[k] = ((uint64_t)sys << (63 - 3 * vlev)) | (keys[k] >> (3 * vlev));
}

void launch_keys_prefix(uint64_t* keys, const uint32_t* ids, size_t n, const uint64_t* off,
                        uint32_t nsys, int vlev, hipStream_t s) {
  hipLaunchKernelGGL(k_keys_prefix, dim3((n + TB - 1) / TB), dim3(TB), 0, s, keys, ids, n, off,
                     nsys, vlev);
}

void launch_keys_sys(const double* pos, const double* mass, size_t n, const uint64_t* off,
                     uint32_t nsys, int vlev, const BBox* bbs, uint64_t* keys, uint32_t* vals,
                     uint32_t* flags, double4* pk, hipStream_t s) {
  hipLaunchKernelGGL(k_keys_sys, dim3((n + TB - 1) / TB), dim3(TB), 0, s, pos, mass, n, off, nsys,
                     vlev, bbs, keys, vals, flags, pk);
}

void launch_keys(const double* pos, const double* mass, size_t n, const BBox* bb, uint64_t* keys,
                 uint32_t* vals, uint32_t* flags, double4* pk, hipStream_t s) {
  hipLaunchKernelGGL(k_keys, dim3((n + TB - 1) / TB), dim3(TB), 0, s, pos, mass, n, bb, keys, vals,
                     flags, pk);
}

// Bodies::from_parts (bodies.rs:27-47): id order AoS -> slot order SoA.
__global__ void __launch_bounds__(TB) k_gather(const double* __restrict__ pos,
                                              const double* __restrict__ mass,
                                              const uint32_t* __restrict__ order, size_t n,
                                              DevBodies b) {
  size_t k = (size_t)blockIdx.x * TB + threadIdx.x;
  if (k >= n) return;
  size_t id = order[k];
  const double x = pos[3 * id], y = pos[3 * id + 1], z = pos[3 * id + 2], m = mass[id];
  b.x[k] = x;
  b.y[k] = y;
  b.z[k] = z;
  b.m[k] = m;
  b.xyzm[k] = make_double4(x, y, z, m);
}

void launch_gather(const double* pos, const double* mass, const uint32_t* order, size_t n,
                   DevBodies b, hipStream_t s) {
  hipLaunchKernelGGL(k_gather, dim3((n + TB - 1) / TB), dim3(TB), 0, s, pos, mass, order, n, b);
}

// The same gather from the keys kernel's packed copy (x, y, z, m in id
// order, 32 bytes per body): one aligned 32-byte read per body instead of
// the position triple and the mass from two arrays.
__global__ void __launch_bounds__(TB) k_gather_packed(const double4* __restrict__ pk,
                                                     const uint32_t* __restrict__ order, size_t n,
                                                     DevBodies b) {
  size_t k = (size_t)blockIdx.x * TB + threadIdx.x;
  if (k >= n) return;
  const double4 v = pk[order[k]];
  b.x[k] = v.x;
  b.y[k] = v.y;
  b.z[k] = v.z;
  b.m[k] = v.w;
  b.xyzm[k] = v;
}

void launch_gather_packed(const double4* pk, const uint32_t* order, size_t n, DevBodies b,
                          hipStream_t s) {
  hipLaunchKernelGGL(k_gather_packed, dim3((n + TB - 1) / TB), dim3(TB), 0, s, pk, order, n, b);
}

// Leading octal digits (levels) in which two 63-bit keys agree, 0..21.
__device__ __forceinline__ int common_levels(uint64_t a, uint64_t b) {
  const uint64_t x = a ^ b;
  return x == 0 ? BITS : ((int)__clzll((long long)x) - 1) / 3;
}
__device__ __forceinline__ bool same_cell(uint64_t a, uint64_t b, int level) {
  return ((a ^ b) >> (3 * (BITS - level))) == 0;
}

// Levels [top, bottom] of the cells starting at slot i (tree.rs:414: a cell
// splits when it has more than n_leaf bodies and its level is below 21; the
// virtual levels of an ensemble, level < vlev, always split). top > bottom:
// none.
__device__ __forceinline__ void slot_chain(const uint64_t* __restrict__ keys, uint32_t n,
                                           uint32_t i, uint32_t n_leaf, int vlev, int* top,
                                           int* bottom) {
  const uint64_t k = keys[i];
  int t = 0;
  if (i > 0) {
    // the slot starts cells below level q, if the cell of level q that holds
    // it and its predecessor splits
    const int q = common_levels(keys[i - 1], k);
    *top = 1;
    *bottom = 0;
    if (q == BITS) return;
    if (q >= vlev) {
      // more than n_leaf bodies around slots i - 1 and i: half as many on one
      // side at least (rejects nearly every slot inside a leaf) ...
      const uint32_t h = n_leaf - n_leaf / 2;
      const bool hi = (uint64_t)i + h < n && same_cell(keys[i + h], k, q);
      const bool lo = i >= h && same_cell(keys[i - h], k, q);
      if (!hi && !lo) return;
      // ... and n_leaf slots past the cell's start still in it
      uint32_t a = i > n_leaf ? i - n_leaf : 0u, b = i;  // start in [a, b] unless before a
      while (a < b) {
        const uint32_t mid = a + (b - a) / 2;
        if (same_cell(keys[mid], k, q))
          b = mid;
        else
          a = mid + 1;
      }
      if (!((uint64_t)a + n_leaf < n && same_cell(keys[a + n_leaf], k, q))) return;
    }
    t = q + 1;
  }
  const int g = (uint64_t)i + n_leaf < n ? common_levels(k, keys[i + n_leaf]) : -1;
  *top = t;
  *bottom = max(max(t, vlev), min(g, BITS - 1) + 1);
}

// Per slot the cells that start there (count << 32 | 1 if any: each chain
// ends in exactly one leaf) and per level the internal cells and leaves
// (hist[2 level + leaf]).
__global__ void __launch_bounds__(TB) k_chain(const uint64_t* __restrict__ keys, uint32_t n,
                                             uint32_t n_leaf, int vlev,
                                             uint64_t* __restrict__ chain,
                                             uint32_t* __restrict__ hist) {
  __shared__ uint32_t h[TREE_HIST];
  for (int q = threadIdx.x; q < TREE_HIST; q += TB) h[q] = 0;
  __syncthreads();
  for (uint64_t i = (uint64_t)blockIdx.x * TB + threadIdx.x; i < n; i += (uint64_t)gridDim.x * TB) {
    int top, bot;
    slot_chain(keys, n, (uint32_t)i, n_leaf, vlev, &top, &bot);
    chain[i] = top <= bot ? ((uint64_t)(bot - top + 1) << 32) | 1ull : 0ull;
    for (int l = top; l <= bot; l++) atomicAdd(&h[2 * l + (l == bot ? 1 : 0)], 1u);
  }
  __syncthreads();
  for (int q = threadIdx.x; q < TREE_HIST; q += TB)
    if (h[q]) atomicAdd(&hist[q], h[q]);
}

void launch_chain(const uint64_t* keys, size_t n, uint32_t n_leaf, int vlev, uint64_t* chain,
                  uint32_t* hist, hipStream_t s) {
  const size_t nb = std::min<size_t>((n + TB - 1) / TB, 2048);
  hipLaunchKernelGGL(k_chain, dim3(nb), dim3(TB), 0, s, keys, (uint32_t)n, n_leaf, vlev, chain,
                     hist);
}

// Writes each slot's chain of cells (start = exclusive scan of chain: cells
// << 32 | leaves before the slot): first slot, level, leaf flag, the links
// inside the chain, and the leaf list. The chain's top cell gets its parent
// from k_cell_links.
__global__ void __launch_bounds__(TB) k_cell_emit(const uint64_t* __restrict__ keys, uint32_t n,
                                                 const uint64_t* __restrict__ chain,
                                                 const uint64_t* __restrict__ start, DevCells c,
                                                 uint32_t* __restrict__ leaf_ids) {
  const uint32_t i = blockIdx.x * TB + threadIdx.x;
  if (i >= n) return;
  const int m = (int)(chain[i] >> 32);
  if (m == 0) return;
  const uint64_t k = keys[i];
  const int top = i == 0 ? 0 : common_levels(keys[i - 1], k) + 1;
  const uint32_t id0 = (uint32_t)(start[i] >> 32);
  for (int q = 0; q < m; q++) {
    const uint32_t id = id0 + (uint32_t)q;
    c.first[id] = i;
    c.level[id] = (uint8_t)(top + q);
    c.leaf[id] = q == m - 1 ? 1 : 0;
    if (q > 0) c.parent[id] = (int32_t)(id - 1);
    const int32_t next = q == m - 1 ? -1 : (int32_t)(id + 1);
    // the octant of the next cell of the chain (a leaf has none, and at level 21
    // the key has no digit left to shift to)
    const int oct = next < 0 ? -1 : (int)((k >> (3 * (BITS - (top + q + 1)))) & 7u);
    int32_t* ch = c.children + (size_t)id * 8;
#pragma unroll
    for (int o = 0; o < 8; o++) ch[o] = o == oct ? next : -1;
  }
  leaf_ids[(uint32_t)start[i]] = id0 + (uint32_t)(m - 1);
}

// Per cell: body count (the end of its prefix run, found by galloping) and,
// for the top cell of a chain, the link to its parent, the cell one level up
// whose run holds the slot before. Leaves also mark their slots.
__global__ void __launch_bounds__(TB) k_cell_links(const uint64_t* __restrict__ keys, uint32_t n,
                                                  const uint64_t* __restrict__ start, uint32_t nc,
                                                  DevCells c, uint32_t* __restrict__ leaf_of_slot) {
  const uint32_t id = blockIdx.x * TB + threadIdx.x;
  if (id >= nc) return;
  const uint32_t f = c.first[id];
  const int lev = c.level[id];
  const uint64_t k = keys[f];
  // end: the last slot known inside is f + in, the first known outside f + out
  uint64_t in = 0, out = 1;
  while (f + out < n && same_cell(keys[f + out], k, lev)) {
    in = out;
    out *= 2;
  }
  out = min(out, (uint64_t)(n - f));
  while (out - in > 1) {
    const uint64_t mid = in + (out - in) / 2;
    if (same_cell(keys[f + mid], k, lev))
      in = mid;
    else
      out = mid;
  }
  c.count[id] = (uint32_t)out;
  if (c.leaf[id])
    for (uint32_t j = 0; j < (uint32_t)out; j++) leaf_of_slot[f + j] = id;
  if (id == 0) {
    c.parent[0] = -1;
    return;
  }
  if ((uint32_t)(start[f] >> 32) != id) return;  // not the chain's top
  uint64_t back = 0, past = 1;  // f - back is in the parent's run, f - past is not
  while (past <= f && same_cell(keys[f - past], k, lev - 1)) {
    back = past;
    past *= 2;
  }
  past = min(past, (uint64_t)f + 1);
  while (past - back > 1) {
    const uint64_t mid = back + (past - back) / 2;
    if (same_cell(keys[f - mid], k, lev - 1))
      back = mid;
    else
      past = mid;
  }
  const uint32_t head = (uint32_t)(start[f - back] >> 32);
  const uint32_t pa = head + (uint32_t)(lev - 1) - (uint32_t)c.level[head];
  c.parent[id] = (int32_t)pa;
  c.children[(size_t)pa * 8 + ((k >> (3 * (BITS - lev))) & 7u)] = (int32_t)id;
}

void launch_cells(const uint64_t* keys, size_t n, const uint64_t* chain, const uint64_t* start,
                  uint32_t nc, DevCells c, uint32_t* leaf_ids, uint32_t* leaf_of_slot,
                  hipStream_t s) {
  hipLaunchKernelGGL(k_cell_emit, dim3((n + TB - 1) / TB), dim3(TB), 0, s, keys, (uint32_t)n, chain,
                     start, c, leaf_ids);
  hipLaunchKernelGGL(k_cell_links, dim3((nc + TB - 1) / TB), dim3(TB), 0, s, keys, (uint32_t)n,
                     start, nc, c, leaf_of_slot);
}

// ---------------------------------------------------------------- geometry
__device__ __forceinline__ double dist3(double ax, double ay, double az, double bx, double by,
                                        double bz) {  // tree.rs:392-402
  double dx = ax - bx, dy = ay - by, dz = az - bz;
  return sqrt(dx * dx + dy * dy + dz * dz);
}

// Ritter grow/enclose sphere with the bbox-centred fallback, tree.rs:290-389.
// `get(i, c, r)` yields item i's centre and radius.
template <class Get>
__device__ void ritter(int nitems, Get get, double out[3]) {
  const double MINP = 2.2250738585072014e-308;
  double c0[3], r0;
  int a = 0, b = 0;
  double best = -1.0;
  double ca[3], ra;
  get(0, ca, &ra);
  for (int i = 0; i < nitems; i++) {
    double ci[3], ri;
    get(i, ci, &ri);
    double dx = ci[0] - ca[0], dy = ci[1] - ca[1], dz = ci[2] - ca[2];
    double d2 = dx * dx + dy * dy + dz * dz;
    if (d2 > best) {
      best = d2;
      b = i;
    }
  }
  a = b;
  best = -1.0;
  get(a, ca, &ra);
  for (int i = 0; i < nitems; i++) {
    double ci[3], ri;
    get(i, ci, &ri);
    double dx = ci[0] - ca[0], dy = ci[1] - ca[1], dz = ci[2] - ca[2];
    double d2 = dx * dx + dy * dy + dz * dz;
    if (d2 > best) {
      best = d2;
      b = i;
    }
  }
  double pa[3], pb[3], rad_a, rad_b;
  get(a, pa, &rad_a);
  get(b, pb, &rad_b);
  double dir[3];
  {
    double dx = pb[0] - pa[0], dy = pb[1] - pa[1], dz = pb[2] - pa[2];
    double d = fmax(sqrt(dx * dx + dy * dy + dz * dz), MINP);
    dir[0] = dx / d;
    dir[1] = dy / d;
    dir[2] = dz / d;
  }
  double fa[3] = {pa[0] + rad_a * dir[0], pa[1] + rad_a * dir[1], pa[2] + rad_a * dir[2]};
  double fb[3] = {pb[0] - rad_b * dir[0], pb[1] - rad_b * dir[1], pb[2] - rad_b * dir[2]};
  c0[0] = (fa[0] + fb[0]) * 0.5;
  c0[1] = (fa[1] + fb[1]) * 0.5;
  c0[2] = (fa[2] + fb[2]) * 0.5;
  r0 = dist3(fa[0], fa[1], fa[2], fb[0], fb[1], fb[2]) * 0.5;
  for (int pass = 0; pass < 2; pass++) {
    for (int i = 0; i < nitems; i++) {
      double q[3], rad;
      get(i, q, &rad);
      double d = dist3(q[0], q[1], q[2], c0[0], c0[1], c0[2]);
      if (d + rad > r0) {
        double dd = fmax(d, MINP);
        double dr[3] = {(q[0] - c0[0]) / dd, (q[1] - c0[1]) / dd, (q[2] - c0[2]) / dd};
        double pnt[3] = {q[0] + rad * dr[0], q[1] + rad * dr[1], q[2] + rad * dr[2]};
        double d_far = d + rad;
        double t = (d_far - r0) / (2.0 * d_far);
        for (int k = 0; k < 3; k++) c0[k] += t * (pnt[k] - c0[k]);
        r0 = (d_far + r0) * 0.5;
      }
    }
  }
  double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (int i = 0; i < nitems; i++) {
    double q[3], rad;
    get(i, q, &rad);
    for (int d = 0; d < 3; d++) {
      lo[d] = fmin(lo[d], q[d] - rad);
      hi[d] = fmax(hi[d], q[d] + rad);
    }
  }
  double cb[3] = {(lo[0] + hi[0]) * 0.5, (lo[1] + hi[1]) * 0.5, (lo[2] + hi[2]) * 0.5};
  double rb = 0.0;
  for (int i = 0; i < nitems; i++) {
    double q[3], rad;
    get(i, q, &rad);
    rb = fmax(rb, dist3(q[0], q[1], q[2], cb[0], cb[1], cb[2]) + rad);
  }
  if (rb < r0) {
    out[0] = cb[0];
    out[1] = cb[1];
    out[2] = cb[2];
  } else {
    out[0] = c0[0];
    out[1] = c0[1];
    out[2] = c0[2];
  }
}

// tree.rs:152-227, one thread per internal cell of a level (children done
// first). The children's data is gathered before any of it is used, so the
// cell costs two dependent loads instead of two per child.
__global__ void __launch_bounds__(TB) k_geometry(const uint32_t* __restrict__ cells, uint32_t cnt,
                                                DevCells c, int mode) {
  const uint32_t i = blockIdx.x * TB + threadIdx.x;
  if (i >= cnt) return;
  const uint32_t id = cells[i];
  int q[8];
  double qm[8], qx[8], qy[8], qz[8], qr[8];
  const int32_t* ch = c.children + (size_t)id * 8;
#pragma unroll
  for (int o = 0; o < 8; o++) q[o] = ch[o];
#pragma unroll
  for (int o = 0; o < 8; o++) {
    const int a = q[o] >= 0 ? q[o] : (int)id;  // absent: read, not used
    qm[o] = c.mass[a];
    qx[o] = c.cx[a];
    qy[o] = c.cy[a];
    qz[o] = c.cz[a];
    qr[o] = c.rho[a];
  }
  double ms = 0.0;
  double cen[3];
#pragma unroll
  for (int o = 0; o < 8; o++)
    if (q[o] >= 0) ms += qm[o];
  if (mode == 0) {
    double com[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int o = 0; o < 8; o++) {
      if (q[o] < 0) continue;
      com[0] += qm[o] * qx[o];
      com[1] += qm[o] * qy[o];
      com[2] += qm[o] * qz[o];
    }
    cen[0] = com[0] / ms;
    cen[1] = com[1] / ms;
    cen[2] = com[2] / ms;
  } else {
    int list[8];
    int nl = 0;
    for (int o = 0; o < 8; o++)
      if (ch[o] >= 0) list[nl++] = ch[o];
    ritter(
        nl,
        [&](int e, double* ec, double* er) {
          const int cc = list[e];
          ec[0] = c.cx[cc];
          ec[1] = c.cy[cc];
          ec[2] = c.cz[cc];
          *er = c.rho[cc];
        },
        cen);
  }
  double rho = 0.0;
#pragma unroll
  for (int o = 0; o < 8; o++) {
    if (q[o] < 0) continue;
    rho = fmax(rho, qr[o] + dist3(qx[o], qy[o], qz[o], cen[0], cen[1], cen[2]));
  }
  c.mass[id] = ms;
  c.cx[id] = cen[0];
  c.cy[id] = cen[1];
  c.cz[id] = cen[2];
  c.rho[id] = rho;
}

// Leaf geometry with one wave per leaf (tree.rs:152-227, 257-275, 290-389). Order-dependent sums
// (mass, centre of mass) run in slot order over bodies read from the lanes
// that hold them; the farthest-point searches, the box and the radius and
// rho maxima spread over the lanes (a maximum, ties to the lowest slot, does
// not depend on the order); the grow passes test a chunk of bodies against
// the current sphere at once and apply the first failing body's update, then
// test the bodies after it again, which is exactly the sequential pass.
constexpr int GEO_WAVES = 4;

__device__ __forceinline__ double wave_max_pos(double v) {  // v >= +0 in every lane
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return v;
}

// Farthest body from slot a (first slot on ties), over the leaf's bodies.
__device__ __forceinline__ uint32_t wave_farthest(DevBodies b, uint32_t f, uint32_t n, uint32_t a,
                                                  int lane) {
  const double ax = b.x[f + a], ay = b.y[f + a], az = b.z[f + a];
  double best = -1.0;
  uint32_t bi = 0;
  for (uint32_t i = (uint32_t)lane; i < n; i += 64) {
    const double dx = b.x[f + i] - ax, dy = b.y[f + i] - ay, dz = b.z[f + i] - az;
    const double d2 = dx * dx + dy * dy + dz * dz;
    if (d2 > best) {
      best = d2;
      bi = i;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double ob = __shfl_xor(best, o, 64);
    const uint32_t oi = (uint32_t)__shfl_xor((int)bi, o, 64);
    if (ob > best || (ob == best && oi < bi)) {
      best = ob;
      bi = oi;
    }
  }
  return bi;
}

__global__ void __launch_bounds__(64 * GEO_WAVES) k_geometry_leaf(
    const uint32_t* __restrict__ leaf_ids, uint32_t nleaves, DevCells c, DevBodies b, int mode) {
  // per wave: one chunk of the leaf's bodies (mass, x, y, z) for the serial sums
  __shared__ double chunk[GEO_WAVES][4][64];
  const uint32_t wv = threadIdx.x >> 6;
  const uint32_t li = blockIdx.x * GEO_WAVES + wv;
  const int lane = threadIdx.x & 63;
  if (li >= nleaves) return;
  const uint32_t id = leaf_ids[li];
  const uint32_t f = c.first[id], n = c.count[id];
  // Slot-ordered sums over chunks of 64 bodies: the lanes stage the chunk in
  // LDS, then lane 0 sums the masses (m * 1) and lanes 1-3 the mass-weighted
  // coordinates, each in slot order (the wave's LDS operations run in program
  // order; the wave barrier keeps the compiler from reordering them).
  double sum = 0.0;  // lane 0: mass; lanes 1-3: sum of m x, m y, m z
  for (uint32_t base = 0; base < n; base += 64) {
    const uint32_t i = base + (uint32_t)lane;
    const bool have = i < n;
    const uint32_t cnt = min(64u, n - base);
    chunk[wv][0][lane] = have ? b.m[f + i] : 0.0;
    if (mode == 0) {  // com_of_slots, tree.rs:257-275
      chunk[wv][1][lane] = have ? b.x[f + i] : 0.0;
      chunk[wv][2][lane] = have ? b.y[f + i] : 0.0;
      chunk[wv][3][lane] = have ? b.z[f + i] : 0.0;
    }
    __builtin_amdgcn_wave_barrier();
    if (lane < (mode == 0 ? 4 : 1)) {
      for (uint32_t k = 0; k < cnt; k++) {
        const double m = chunk[wv][0][k];
        sum += m * (lane == 0 ? 1.0 : chunk[wv][lane][k]);
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  const double ms = lane_read(sum, 0);
  double cen[3];
  if (mode == 0) {
    cen[0] = lane_read(sum, 1) / ms;
    cen[1] = lane_read(sum, 2) / ms;
    cen[2] = lane_read(sum, 3) / ms;
  } else {  // Ritter sphere, tree.rs:290-389 (bodies have radius 0)
    const double MINP = 2.2250738585072014e-308;
    const double rad = 0.0;
    const uint32_t a = wave_farthest(b, f, n, 0, lane);
    const uint32_t bb = wave_farthest(b, f, n, a, lane);
    const double pa[3] = {b.x[f + a], b.y[f + a], b.z[f + a]};
    const double pb[3] = {b.x[f + bb], b.y[f + bb], b.z[f + bb]};
    double dir[3];
    {
      const double dx = pb[0] - pa[0], dy = pb[1] - pa[1], dz = pb[2] - pa[2];
      const double d = fmax(sqrt(dx * dx + dy * dy + dz * dz), MINP);
      dir[0] = dx / d;
      dir[1] = dy / d;
      dir[2] = dz / d;
    }
    const double fa[3] = {pa[0] + rad * dir[0], pa[1] + rad * dir[1], pa[2] + rad * dir[2]};
    const double fb[3] = {pb[0] - rad * dir[0], pb[1] - rad * dir[1], pb[2] - rad * dir[2]};
    double c0[3] = {(fa[0] + fb[0]) * 0.5, (fa[1] + fb[1]) * 0.5, (fa[2] + fb[2]) * 0.5};
    double r0 = dist3(fa[0], fa[1], fa[2], fb[0], fb[1], fb[2]) * 0.5;
    for (int pass = 0; pass < 2; pass++) {
      for (uint32_t base = 0; base < n; base += 64) {
        const uint32_t i = base + (uint32_t)lane;
        const bool have = i < n;
        const double qx = have ? b.x[f + i] : 0.0, qy = have ? b.y[f + i] : 0.0,
                     qz = have ? b.z[f + i] : 0.0;
        int start = 0;
        // each round either ends the chunk or moves start past one lane
        while (start < 64) {
          double d = 0.0;
          bool out = false;
          if (have && lane >= start) {
            d = dist3(qx, qy, qz, c0[0], c0[1], c0[2]);
            out = d + rad > r0;
          }
          const uint64_t m = __ballot(out);
          if (m == 0) break;
          const int j = __ffsll((long long)m) - 1;
          const double q[3] = {__shfl(qx, j, 64), __shfl(qy, j, 64), __shfl(qz, j, 64)};
          const double dj = __shfl(d, j, 64);
          const double dd = fmax(dj, MINP);
          const double dr[3] = {(q[0] - c0[0]) / dd, (q[1] - c0[1]) / dd, (q[2] - c0[2]) / dd};
          const double pnt[3] = {q[0] + rad * dr[0], q[1] + rad * dr[1], q[2] + rad * dr[2]};
          const double d_far = dj + rad;
          const double t = (d_far - r0) / (2.0 * d_far);
          for (int k = 0; k < 3; k++) c0[k] += t * (pnt[k] - c0[k]);
          r0 = (d_far + r0) * 0.5;
          start = j + 1;
        }
      }
    }
    // the box: a min/max does not depend on the order (up to the sign of a
    // zero extreme, which changes no centre unless both extremes are zero)
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (uint32_t i = (uint32_t)lane; i < n; i += 64) {
      const double q[3] = {b.x[f + i], b.y[f + i], b.z[f + i]};
      for (int d = 0; d < 3; d++) {
        lo[d] = fmin(lo[d], q[d] - rad);
        hi[d] = fmax(hi[d], q[d] + rad);
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
      for (int d = 0; d < 3; d++) {
        lo[d] = fmin(lo[d], __shfl_xor(lo[d], o, 64));
        hi[d] = fmax(hi[d], __shfl_xor(hi[d], o, 64));
      }
    const double cb[3] = {(lo[0] + hi[0]) * 0.5, (lo[1] + hi[1]) * 0.5, (lo[2] + hi[2]) * 0.5};
    double rb = 0.0;
    for (uint32_t i = (uint32_t)lane; i < n; i += 64)
      rb = fmax(rb, dist3(b.x[f + i], b.y[f + i], b.z[f + i], cb[0], cb[1], cb[2]) + rad);
    rb = wave_max_pos(rb);
    for (int k = 0; k < 3; k++) cen[k] = rb < r0 ? cb[k] : c0[k];
  }
  double rho = 0.0;
  for (uint32_t i = (uint32_t)lane; i < n; i += 64)
    rho = fmax(rho, dist3(b.x[f + i], b.y[f + i], b.z[f + i], cen[0], cen[1], cen[2]));
  rho = wave_max_pos(rho);
  if (lane == 0) {
    c.mass[id] = ms;
    c.cx[id] = cen[0];
    c.cy[id] = cen[1];
    c.cz[id] = cen[2];
    c.rho[id] = rho;
  }
}

void launch_geometry_leaves(const uint32_t* leaf_ids, uint32_t nleaves, DevCells c, DevBodies b,
                            int center_mode, hipStream_t s) {
  if (nleaves == 0) return;
  hipLaunchKernelGGL(k_geometry_leaf, dim3((nleaves + GEO_WAVES - 1) / GEO_WAVES),
                     dim3(64 * GEO_WAVES), 0, s, leaf_ids, nleaves, c, b, center_mode);
}

void launch_geometry(const uint32_t* cells, uint32_t cnt, DevCells c, int center_mode,
                     hipStream_t s) {
  if (cnt == 0) return;
  hipLaunchKernelGGL(k_geometry, dim3((cnt + TB - 1) / TB), dim3(TB), 0, s, cells, cnt, c,
                     center_mode);
}

// Ropes of the mirrored DFS (children visited 7..0): the cell visited after
// a cell's subtree is its next lower existing sibling, else its parent's
// rope. Each cell climbs to the first ancestor with a lower sibling (one
// launch for all levels; a pass per level before).
__global__ void __launch_bounds__(TB) k_ropes(uint32_t nc, DevCells c) {
  const uint32_t i = blockIdx.x * TB + threadIdx.x;
  if (i >= nc) return;
  int32_t last = -1;
  const int32_t* ch = c.children + (size_t)i * 8;
#pragma unroll
  for (int o = 0; o < 8; o++)
    if (ch[o] >= 0) last = ch[o];
  c.last_child[i] = last;
  int32_t rope = -1;
  int32_t cur = (int32_t)i;
  for (int l = 0; l <= BITS && rope < 0; l++) {
    const int32_t pa = c.parent[cur];
    if (pa < 0) break;
    const int32_t* sib = c.children + (size_t)pa * 8;
#pragma unroll
    for (int o = 0; o < 8; o++)  // ids rise with the octant: the highest one below cur
      if (sib[o] >= 0 && sib[o] < cur) rope = sib[o];
    cur = pa;
  }
  c.rope[i] = rope;
}

void launch_ropes(uint32_t nc, DevCells c, hipStream_t s) {
  hipLaunchKernelGGL(k_ropes, dim3((nc + TB - 1) / TB), dim3(TB), 0, s, nc, c);
}

}  // namespace fmmh
