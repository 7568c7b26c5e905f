// Exclusive scan of values that a loader computes on the fly (a count array, a flag derived from a byte), with the total
// written where the host reads it. Included by the translation units that scan their own loaders.
//
// Reduce-then-scan over 2048-element tiles (256 threads x 8 items, one u64 running sum per thread); inputs of up to
// 16384 elements are scanned by one block in one launch (a request's small scans cost one launch, not three).
#pragma once
#include "engine.h"

namespace gsj {

namespace {

constexpr int SCAN_T = 256, SCAN_ITEMS = 8, SCAN_TILE = SCAN_T * SCAN_ITEMS;

__device__ __forceinline__ uint64_t wave_incl_scan(uint64_t v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    uint64_t t = __shfl_up(v, o, 64);
    if (lane >= o) v += t;
  }
  return v;
}

// block-wide exclusive scan of one value per thread (blockDim == SCAN_T); returns exclusive prefix, *total = sum
__device__ __forceinline__ uint64_t block_excl_scan(uint64_t v, uint64_t* total) {
  __shared__ uint64_t wsum[SCAN_T / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint64_t inc = wave_incl_scan(v);
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  uint64_t base = 0, tot = 0;
#pragma unroll
  for (int k = 0; k < SCAN_T / 64; k++) {
    if (k < w) base += wsum[k];
    tot += wsum[k];
  }
  __syncthreads();
  *total = tot;
  return base + inc - v;
}

// loader of a plain count or flag array
template <class T>
struct LoadArray {
  static constexpr bool PACKED = false;
  const T* p;
  __device__ __forceinline__ uint64_t operator()(uint64_t i) const { return (uint64_t)p[i]; }
};

// Where the total goes: words[0] (device memory, or pinned host memory that the kernel writes directly), and with `over`
// a counter that the caller's earlier kernel incremented: its value goes to words[1] and it starts at 0 again; dev (or
// null) takes the total for a later kernel.
struct ScanTotal {
  uint64_t* words = nullptr;
  uint32_t* over = nullptr;
  uint64_t* dev = nullptr;
  __device__ __forceinline__ void put(uint64_t total) const {
    if (words) words[0] = total;
    if (dev) *dev = total;
    if (over) { words[1] = *over; *over = 0; }
  }
};

template <class Ld>
__global__ void __launch_bounds__(SCAN_T) k_tile_sums(const Ld in, uint64_t n, uint64_t* sums) {
  const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE;
  uint64_t s = 0;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; k++) {
    uint64_t i = base + (uint64_t)k * SCAN_T + threadIdx.x;
    if (i < n) s += in(i);
  }
  uint64_t tot;
  (void)block_excl_scan(s, &tot);
  if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

// single block: exclusive scan of nb tile sums in place; grand total out
__global__ void __launch_bounds__(SCAN_T) k_scan_sums(uint64_t* sums, uint64_t nb, ScanTotal total) {
  uint64_t carry = 0;
  for (uint64_t base = 0; base < nb; base += SCAN_T) {
    uint64_t i = base + threadIdx.x;
    uint64_t v = i < nb ? sums[i] : 0;
    uint64_t tot;
    uint64_t ex = block_excl_scan(v, &tot);
    if (i < nb) sums[i] = carry + ex;
    carry += tot;
  }
  if (threadIdx.x == 0) total.put(carry);
}

template <class Ld, class TO>
__global__ void __launch_bounds__(SCAN_T) k_tile_scan(const Ld in, TO* out, uint64_t n, const uint64_t* offs) {
  const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_ITEMS;   // contiguous per thread
  uint64_t v[SCAN_ITEMS];
  uint64_t s = 0;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; k++) {
    uint64_t i = base + k;
    v[k] = i < n ? in(i) : 0;
    s += v[k];
  }
  uint64_t tot;
  uint64_t ex = block_excl_scan(s, &tot) + offs[blockIdx.x];
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; k++) {
    uint64_t i = base + k;
    if (i < n) out[i] = (TO)ex;
    ex += v[k];
  }
}

// one block: exclusive scan of n <= SS_MAX elements; thread t scans elements [per t, per (t + 1)). They are read and
// written in order, 64 lanes side by side, and pass through LDS between (each thread reading its own run from memory
// touched a line per element: 10.6k probe counts 8.3 -> 5.9 us). An odd `per` spreads the threads' runs over the banks. A total of
// 2^32 or more (prefixes that do not fit the LDS words) is written from the registers. A PACKED loader counts two kinds in
// the halves of a word, at most one each: they pass through LDS as 16-bit halves, and so do their prefixes. Every element is read before
// the first is written, so in and out may be the same array.
constexpr int SS_T = 1024, SS_ITEMS = 17, SS_MAX = 16384;
template <bool PACKED> __device__ __forceinline__ uint32_t ss_pack(uint64_t v) { return PACKED ? (uint32_t)v | (uint32_t)(v >> 16) : (uint32_t)v; }
template <bool PACKED> __device__ __forceinline__ uint64_t ss_unpack(uint32_t v) { return PACKED ? (uint64_t)(v & 0xFFFFu) | (uint64_t)(v >> 16) << 32 : v; }
template <class Ld, class TO>
__global__ void __launch_bounds__(SS_T) k_scan_small(const Ld in, TO* out, uint64_t n64, ScanTotal total) {
  __shared__ uint64_t wsum[SS_T / 64];
  __shared__ uint32_t buf[SS_MAX];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const uint32_t n = (uint32_t)n64, per = (n + SS_T - 1) / SS_T | 1u;
  uint32_t v[SS_ITEMS];
#pragma unroll
  for (int k = 0; k < SS_MAX / SS_T; k++) v[k] = t + (uint32_t)k * SS_T < n ? ss_pack<Ld::PACKED>(in(t + (uint32_t)k * SS_T)) : 0u;   // all loads in flight
#pragma unroll
  for (int k = 0; k < SS_MAX / SS_T; k++)
    if (t + (uint32_t)k * SS_T < n) buf[t + k * SS_T] = v[k];
  __syncthreads();
  uint64_t s = 0;
  const uint32_t base = (uint32_t)t * per;
#pragma unroll
  for (int k = 0; k < SS_ITEMS; k++) {
    v[k] = k < (int)per && base + k < n ? buf[base + k] : 0u;
    s += ss_unpack<Ld::PACKED>(v[k]);
  }
  const uint64_t inc = wave_incl_scan(s);
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  uint64_t ex = inc - s, tot = 0;
#pragma unroll
  for (int k = 0; k < SS_T / 64; k++) {
    if (k < w) ex += wsum[k];
    tot += wsum[k];
  }
  if (!Ld::PACKED && (tot >> 32)) {
#pragma unroll
    for (int k = 0; k < SS_ITEMS; k++) {
      if (k < (int)per && base + k < n) out[base + k] = (TO)ex;
      ex += v[k];
    }
  } else {
    uint32_t e = ss_pack<Ld::PACKED>(ex);   // (halves of at most SS_MAX = 2^14)
#pragma unroll
    for (int k = 0; k < SS_ITEMS; k++) {
      if (k < (int)per && base + k < n) buf[base + k] = e;
      e += v[k];
    }
    __syncthreads();
    for (uint32_t i = t; i < n; i += SS_T) out[i] = (TO)ss_unpack<Ld::PACKED>(buf[i]);
  }
  if (t == 0) total.put(tot);
}

__global__ void k_scan_none(ScanTotal total) { total.put(0); }

// out[0 .. n) = exclusive sums of in(0 .. n); asynchronous
template <class TO, class Ld>
void scan_loaded(Context& c, const Ld& in, TO* out, uint64_t n, const ScanTotal& total) {
  if (n == 0) {
    if (total.words || total.over) {
      hipLaunchKernelGGL(k_scan_none, dim3(1), dim3(1), 0, c.stream, total);
      GSJ_LAUNCHED();
    }
    return;
  }
  if (n <= (uint64_t)SS_MAX) {
    hipLaunchKernelGGL((k_scan_small<Ld, TO>), dim3(1), dim3(SS_T), 0, c.stream, in, out, n, total);
    GSJ_LAUNCHED();
    return;
  }
  const uint64_t nb = (n + SCAN_TILE - 1) / SCAN_TILE;
  uint64_t* sums = c.s_scal.as<uint64_t>(nb + 8);
  hipLaunchKernelGGL(k_tile_sums<Ld>, dim3((uint32_t)nb), dim3(SCAN_T), 0, c.stream, in, n, sums);
  GSJ_LAUNCHED();
  hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(SCAN_T), 0, c.stream, sums, nb, total);
  GSJ_LAUNCHED();
  hipLaunchKernelGGL((k_tile_scan<Ld, TO>), dim3((uint32_t)nb), dim3(SCAN_T), 0, c.stream, in, out, n, sums);
  GSJ_LAUNCHED();
}

}  // namespace

}  // namespace gsj
