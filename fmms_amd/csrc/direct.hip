// direct.hip — FP64 direct sum at sampled targets (the checker of the force
// error: direct.rs:6-31 semantics with optional Plummer softening, the
// sampled error of crates/bench/src/main.rs:34-78), and its allocation-free
// entry point.
//
// Each target's sources are cut into nsplit contiguous ranges, one 256-thread
// block per (group of targets, range): a few sampled targets still fill the device.
// Every block writes its five partial sums (ax, ay, az, pot, f) and a second
// kernel adds them in range order, so the result does not depend on timing; the
// only range of a small system is the result, in one launch.
#include <cmath>
#include <mutex>

#include "internal.h"

namespace fmmh {

constexpr int DT = 256;
constexpr int DN = 4;  // targets per block of k_direct_part at the larger sizes
// Scratch of the allocation-free entry point: partial sums, 5 doubles per
// (target, range). 8 MiB per device.
constexpr size_t DIRECT_SCRATCH_WORDS = (size_t)1 << 20;
static_assert(5 * (size_t)FMMH_DIRECT_NOALLOC_MAX_TARGETS <= DIRECT_SCRATCH_WORDS,
              "one range per target must fit the scratch");

// Sums of 2 H values (a power of two) over the wave, by halving: as long as a lane
// holds more than one of them, it hands half to the lane opposite and keeps the
// other, so a block of four targets makes 32 exchanges instead of 120 (most of the
// time of a small system's sums: 12 sources and 4414 targets 16.9 -> 7.5 us, 712 and
// 17961 52.9 -> 27.4; with one target a block 10.6 and 37.7). v[0] of a lane is the sum of the value whose number is
// returned, -1 in the lanes that hold a copy.
template <int H, int O = 32>
__device__ __forceinline__ int scatter_sums(double* v, int lane) {
  if constexpr (H > 0) {
    const bool up = (lane & O) != 0;
#pragma unroll
    for (int i = 0; i < H; i++) {
      const double keep = up ? v[i + H] : v[i], send = up ? v[i] : v[i + H];
      v[i] = keep + __shfl_xor(send, O, 64);
    }
    const int slot = scatter_sums<H / 2, O / 2>(v, lane);
    return slot < 0 ? slot : slot + (up ? H : 0);
  } else {  // lanes that differ in the bits left hold parts of one sum
#pragma unroll
    for (int o = O; o > 0; o >>= 1) v[0] += __shfl_xor(v[0], o, 64);
    return (lane & (2 * O - 1)) == 0 ? 0 : -1;
  }
}

// NT targets per block, in scalar registers: a thread reads a source once and
// evaluates it against all of them. One target per block read 32 bytes from
// the cache for every pair and divided by a square root: 4096 targets x 1M
// sources 8.4 ms, now 3.4 - 3.5 one launch after another (19 FP64 instructions and
// a rsqrt a pair are 3.3 ms at the FP64 issue rate) and 4.1 for a launch by itself,
// which the clock is still rising under.
template <int NT>
__global__ void __launch_bounds__(DT) k_direct_part(const double* __restrict__ pos,
                                                   const double* __restrict__ mass, size_t n,
                                                   double soft2, const uint32_t* __restrict__ ids,
                                                   uint32_t nt, uint32_t nsplit, size_t chunk,
                                                   double* __restrict__ part,
                                                   double* __restrict__ acc_out,
                                                   double* __restrict__ pot_out,
                                                   double* __restrict__ f_out) {
  __shared__ double sh[DT / 64][5 * NT];
  const uint32_t t0 = blockIdx.y * NT, k = blockIdx.x;
  uint32_t id[NT];
  double x[NT], y[NT], z[NT];
  double acc[NT][5];
#pragma unroll
  for (int q = 0; q < NT; q++) {
    id[q] = ids[min(t0 + q, nt - 1)];
    const size_t a = id[q] < n ? id[q] : 0;  // out of range: NaN sums below
    x[q] = pos[3 * a];
    y[q] = pos[3 * a + 1];
    z[q] = pos[3 * a + 2];
#pragma unroll
    for (int e = 0; e < 5; e++) acc[q][e] = 0.0;
  }
  const size_t j0 = (size_t)k * chunk, j1 = j0 + chunk < n ? j0 + chunk : n;
  auto pass = [&](size_t j, bool skip) {
    const double px = pos[3 * j], py = pos[3 * j + 1], pz = pos[3 * j + 2], pm = mass[j];
#pragma unroll
    for (int q = 0; q < NT; q++) {
      double dx = px - x[q], dy = py - y[q], dz = pz - z[q];
      const double r2 = fma(dx, dx, fma(dy, dy, fma(dz, dz, soft2)));
      // refined rsqrt; where the estimate is 0 or infinite (r2 infinite or 0)
      // it is the value
      const double e = __builtin_amdgcn_rsq(r2);
      double inv = rsqrt_pos(r2);
      inv = __builtin_amdgcn_class(e, 0x264) ? e : inv;  // +-inf, +-0
      double m = pm;
      if (skip && j == id[q]) {
        inv = 1.0;
        m = dx = dy = dz = 0.0;
      }
      const double mi = m * inv, mi2 = mi * inv, s3 = mi2 * inv;
      acc[q][0] = fma(s3, dx, acc[q][0]);
      acc[q][1] = fma(s3, dy, acc[q][1]);
      acc[q][2] = fma(s3, dz, acc[q][2]);
      acc[q][3] += mi;
      acc[q][4] += mi2;
    }
  };
  if constexpr (NT == 1) {
    for (size_t j = j0 + threadIdx.x; j < j1; j += DT) pass(j, true);
  } else {
    // whole strides of DT sources without a target among them, then the one with
    for (size_t b = j0; b < j1;) {
      size_t e = j1;
#pragma unroll
      for (int q = 0; q < NT; q++)
        if (id[q] >= b && id[q] < e) e = b + (id[q] - b) / DT * DT;
#pragma unroll 1
      for (size_t j = b + threadIdx.x; j < e; j += DT) pass(j, false);
      if (e < j1 && e + threadIdx.x < j1) pass(e + threadIdx.x, true);
      b = e + DT;
    }
  }
  // fixed-order reduction: lanes by halving, then the waves in order
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  constexpr int NV = NT == 1 ? 8 : 32;  // the sums, to a power of two
  static_assert(5 * NT <= NV, "as many sums as are scattered");
  double v[NV];
#pragma unroll
  for (int i = 0; i < NV; i++) v[i] = i < 5 * NT ? acc[i / 5][i % 5] : 0.0;
  const int slot = scatter_sums<NV / 2>(v, lane);
  if (slot >= 0 && slot < 5 * NT) sh[w][slot] = v[0];
  __syncthreads();
  for (int i = threadIdx.x; i < 5 * NT; i += DT) {
    const int q = i / 5;
    if (t0 + q >= nt) continue;
    double sum = 0.0;
    for (int ww = 0; ww < DT / 64; ww++) sum += sh[ww][i];
    if (ids[t0 + q] >= n) sum = __builtin_nan("");  // ids are device data
    const int e = i - 5 * q;
    if (nsplit > 1)
      part[((size_t)(t0 + q) * nsplit + k) * 5 + e] = sum;
    else if (e < 3)  // one range: its sums are the result
      acc_out[3 * (size_t)(t0 + q) + e] = sum;
    else if (e == 3 ? pot_out : f_out)
      (e == 3 ? pot_out : f_out)[t0 + q] = sum;
  }
}

// Sixteen lanes a target, each adding every sixteenth range's sums, then by
// halving: one thread a target waits for one range after another, and its chain
// of roundings is sixteen times as long (one target of 1M sources, 122 ranges:
// 43 -> 24 us with this, 32 targets 165 -> 57).
constexpr int RL = 16;
__global__ void __launch_bounds__(DT) k_direct_reduce(const double* __restrict__ part, uint32_t nt,
                                                     uint32_t nsplit, double* __restrict__ acc,
                                                     double* __restrict__ pot,
                                                     double* __restrict__ f) {
  const uint32_t l = threadIdx.x % RL;
  for (size_t t = (blockIdx.x * DT + threadIdx.x) / RL; t < nt; t += gridDim.x * (DT / RL)) {
    double s[5] = {0, 0, 0, 0, 0};
    const double* pt = part + t * nsplit * 5;
#pragma unroll 4
    for (uint32_t k = l; k < nsplit; k += RL)
#pragma unroll
      for (int q = 0; q < 5; q++) s[q] += pt[5 * k + q];
#pragma unroll
    for (int q = 0; q < 5; q++)
#pragma unroll
      for (int o = RL / 2; o > 0; o >>= 1) s[q] += __shfl_xor(s[q], o, RL);
    if (l != 0) continue;
    acc[3 * t] = s[0];
    acc[3 * t + 1] = s[1];
    acc[3 * t + 2] = s[2];
    if (pot) pot[t] = s[3];
    if (f) f[t] = s[4];
  }
}

// Groups of DN targets once the groups, over the most ranges there can be, give
// two blocks a CU; below, single targets have more blocks (groups against
// singles in us: 10k bodies x 1000 targets, 250 blocks, 29 / 27; 100k x 100, 300
// blocks, 35 / 33; 100k x 200, 600 blocks, 45 / 51; 1M x 32, 976 blocks,
// 99 / 147; 100k x 400, 1200 blocks, 64 / 86). Eight a group are slower up to
// about a thousand targets (1M x 100 202 instead of 177, 1M x 1000 987 instead of
// 912) and faster past that (1M x 4096 3162 instead of 3404): not taken, 0.2 ms of
// a call of 5.4 there.
static bool direct_groups(size_t n, size_t nt) {
  return (nt + DN - 1) / DN * std::min<size_t>(256, std::max<size_t>(1, n / 8192)) >= 512;
}

uint32_t direct_split(size_t n, size_t nt) {
  // about 4096 blocks in all (16 per CU), each block at least 8192 sources
  const size_t g = direct_groups(n, nt) ? (nt + DN - 1) / DN : nt;
  size_t k = (4096 + g - 1) / g;
  k = std::min<size_t>(k, std::max<size_t>(1, n / 8192));
  k = std::min<size_t>(k, 256);
  k = std::min<size_t>(k, std::max<size_t>(1, DIRECT_SCRATCH_WORDS / (5 * nt)));
  return (uint32_t)std::max<size_t>(k, 1);
}

void launch_direct(const double* pos, const double* mass, size_t n, double soft2,
                   const uint32_t* ids, uint32_t nt, uint32_t nsplit, double* part, double* acc,
                   double* pot, double* f, hipStream_t s) {
  if (nt == 0) return;
  const size_t chunk = (n + nsplit - 1) / nsplit;
  if (direct_groups(n, nt))
    hipLaunchKernelGGL(k_direct_part<DN>, dim3(nsplit, (nt + DN - 1) / DN), dim3(DT), 0, s, pos, mass,
                       n, soft2, ids, nt, nsplit, chunk, part, acc, pot, f);
  else
    hipLaunchKernelGGL(k_direct_part<1>, dim3(nsplit, nt), dim3(DT), 0, s, pos, mass, n, soft2, ids,
                       nt, nsplit, chunk, part, acc, pot, f);
  if (nsplit == 1) return;
  const size_t rb = ((size_t)nt * RL + DT - 1) / DT;
  hipLaunchKernelGGL(k_direct_reduce, dim3((unsigned)std::min<size_t>(rb, 1 << 16)), dim3(DT), 0, s,
                     part, nt, nsplit, acc, pot, f);
}

}  // namespace fmmh

using namespace fmmh;

// Partial sums of fmmh_direct_sampled_noalloc. In host code this name is a
// stand-in, not a device address: kernels get the address that
// hipGetSymbolAddress returns for the current device.
static __device__ __align__(256) double scratch[DIRECT_SCRATCH_WORDS];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch[kMaxDevices] = {};

// The current device's copy of `scratch`, looked up once per device.
int scratch_of_current_device(double** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return FMMH_E_HIP;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return FMMH_E_HIP;
    g_scratch[dev] = (double*)p;
  }
  *out = g_scratch[dev];
  return FMMH_OK;
}
}  // namespace

extern "C" int fmmh_direct_sampled_noalloc(size_t n, const double* d_pos, const double* d_mass,
                                           double softening, size_t nt, const uint32_t* d_idx,
                                           double* d_acc, double* d_pot, double* d_f,
                                           void* stream) {
  if (n == 0 || nt == 0) return FMMH_E_EMPTY;
  if (!d_pos || !d_mass || !d_idx || !d_acc) return FMMH_E_PARAM;
  if (nt > FMMH_DIRECT_NOALLOC_MAX_TARGETS || n >= 0xFFFFFFFFull) return FMMH_E_PARAM;
  if (!(softening >= 0.0) || !std::isfinite(softening)) return FMMH_E_PARAM;
  double* part = nullptr;
  if (int rc = scratch_of_current_device(&part)) return rc;
  const uint32_t nsplit = direct_split(n, nt);
  launch_direct(d_pos, d_mass, n, softening * softening, d_idx, (uint32_t)nt, nsplit, part, d_acc,
                d_pot, d_f, (hipStream_t)stream);
  return hipGetLastError() == hipSuccess ? FMMH_OK : FMMH_E_HIP;
}
