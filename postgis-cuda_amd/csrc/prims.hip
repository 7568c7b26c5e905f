// Device primitives written for CDNA (wave64): exclusive scan and a stable LSD radix sort of (u64 key, u32 value).
//
// Scan: scan.h. A total that the host waits for is written into pinned host memory by the scan itself, so no copy stands
// between the scan and the wait (a copy of 8 bytes takes 3 us of the stream).
// Radix sort: 8-bit digits, 4096-element tiles (256 threads x 16 items). Per pass one histogram kernel, one scan of
// the digit-major histogram, one scatter kernel. Ranks inside a tile come from a wave-level "match" (8 ballots give
// the mask of lanes holding the same digit) plus per-wave digit counts in LDS, so each element's destination is
// computed without per-element LDS atomics and the order of equal keys is preserved. Digits that are identical in
// every key are skipped (found from the OR / AND of all keys).
#include "scan.h"

namespace gsj {

namespace {

// Tiles of 4096 elements; of 1024 up to RS_SMALL elements, where the longer ones would leave most of the chip idle (60k
// elements are 15 blocks of 4096) and the digit counts of the shorter ones still scan in one block
// (a pass over 60k: 27 -> 9 us, its loads sent together as well).
constexpr uint64_t RS_SMALL = 64u << 10;
constexpr int RS_T = 256, RS_ITEMS = 16, RS_ITEMS_SMALL = 4, RS_WAVES = RS_T / 64;

// ------------------------------------------------------------------------------------------- radix sort
__device__ __forceinline__ uint64_t lanemask_lt() {
  const int lane = threadIdx.x & 63;
  return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// lanes whose 8-bit digit equals mine (valid lanes only); `valid` lanes carry d in [0, 256)
__device__ __forceinline__ uint64_t match_digit(uint32_t d, bool valid) {
  uint64_t m = __ballot(valid);
#pragma unroll
  for (int b = 0; b < 8; b++) {
    const bool bit = (d >> b) & 1u;
    const uint64_t bal = __ballot(valid && bit);
    m &= bit ? bal : ~bal;
  }
  return valid ? m : 0ull;
}

template <int ITEMS>
__global__ void __launch_bounds__(RS_T) k_rs_hist(const uint64_t* keys, uint64_t n, int shift, uint32_t ntiles, uint32_t* ghist) {
  __shared__ uint32_t hist[256];
  hist[threadIdx.x] = 0;
  __syncthreads();
  const uint64_t base = (uint64_t)blockIdx.x * (RS_T * ITEMS);
  uint64_t K[ITEMS];
#pragma unroll
  for (int j = 0; j < ITEMS; j++) {
    const uint64_t i = base + (uint64_t)j * RS_T + threadIdx.x;
    K[j] = i < n ? keys[i] : 0;
  }
#pragma unroll
  for (int j = 0; j < ITEMS; j++) {
    const bool valid = base + (uint64_t)j * RS_T + threadIdx.x < n;
    const uint32_t d = valid ? (uint32_t)(K[j] >> shift) & 255u : 0u;
    const uint64_t peers = match_digit(d, valid);
    if (valid && (peers & lanemask_lt()) == 0) atomicAdd(&hist[d], (uint32_t)__popcll(peers));
  }
  __syncthreads();
  ghist[(uint64_t)threadIdx.x * ntiles + blockIdx.x] = hist[threadIdx.x];
}

template <int ITEMS>
__global__ void __launch_bounds__(RS_T) k_rs_scatter(const uint64_t* keys, const uint32_t* vals, uint64_t n, int shift, uint32_t ntiles,
                                                     const uint32_t* goff, uint64_t* keys_out, uint32_t* vals_out) {
  __shared__ uint32_t off[256];
  __shared__ uint32_t wcnt[RS_WAVES][256];
  const int t = threadIdx.x, w = t >> 6;
  off[t] = goff[(uint64_t)t * ntiles + blockIdx.x];
#pragma unroll
  for (int k = 0; k < RS_WAVES; k++) wcnt[k][t] = 0;
  __syncthreads();
  const uint64_t base = (uint64_t)blockIdx.x * (RS_T * ITEMS);
  uint64_t K[ITEMS];   // the tile's loads go out together, ahead of the rounds' barriers
  uint32_t V[ITEMS];
#pragma unroll
  for (int j = 0; j < ITEMS; j++) {
    const uint64_t i = base + (uint64_t)j * RS_T + t;
    K[j] = i < n ? keys[i] : 0;
    V[j] = i < n ? vals[i] : 0;
  }
#pragma unroll
  for (int j = 0; j < ITEMS; j++) {
    const uint64_t i = base + (uint64_t)j * RS_T + t;
    const bool valid = i < n;
    const uint64_t key = K[j];
    const uint32_t val = V[j];
    const uint32_t d = valid ? (uint32_t)(key >> shift) & 255u : 0u;
    const uint64_t peers = match_digit(d, valid);
    const uint32_t rank = (uint32_t)__popcll(peers & lanemask_lt());
    if (valid && rank == 0) wcnt[w][d] = (uint32_t)__popcll(peers);
    __syncthreads();
    if (valid) {
      uint32_t pos = off[d] + rank;
      for (int k = 0; k < w; k++) pos += wcnt[k][d];
      keys_out[pos] = key;
      vals_out[pos] = val;
    }
    __syncthreads();
    uint32_t add = 0;
#pragma unroll
    for (int k = 0; k < RS_WAVES; k++) { add += wcnt[k][t]; wcnt[k][t] = 0; }
    off[t] += add;
    __syncthreads();
  }
}

// or / and of all keys; one pair of atomics per block and at most 256 blocks (a pair per wave of up to 4096 blocks queued
// on two addresses: 23 us of 60k keys, now 7)
__global__ void __launch_bounds__(256) k_key_bits(const uint64_t* keys, uint64_t n, unsigned long long* acc) {
  __shared__ uint64_t po[4], pa[4];
  uint64_t o = 0, a = ~0ull;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) { const uint64_t k = keys[i]; o |= k; a &= k; }
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) { o |= __shfl_xor(o, s, 64); a &= __shfl_xor(a, s, 64); }
  if ((threadIdx.x & 63) == 0) { po[threadIdx.x >> 6] = o; pa[threadIdx.x >> 6] = a; }
  __syncthreads();
  if (threadIdx.x == 0) {
    atomicOr(&acc[0], (unsigned long long)(po[0] | po[1] | po[2] | po[3]));
    atomicAnd(&acc[1], (unsigned long long)(pa[0] & pa[1] & pa[2] & pa[3]));
  }
}

__global__ void k_init_bits(unsigned long long* acc) { acc[0] = 0ull; acc[1] = ~0ull; }

}  // namespace

uint64_t scan_u32_to_u64(Context& c, const uint32_t* in, uint64_t* out, uint64_t n) {
  const HostWords w = host_words(c, 0, 1);
  scan_loaded<uint64_t>(c, LoadArray<uint32_t>{in}, out, n, ScanTotal{w.dev, nullptr});
  w.fetch(c);
  GSJ_HIP(hipStreamSynchronize(c.stream));
  return w.host[0];
}

void scan_u32_to_u64_async(Context& c, const uint32_t* in, uint64_t* out, uint64_t n, uint64_t* d_total) {
  scan_loaded<uint64_t>(c, LoadArray<uint32_t>{in}, out, n, ScanTotal{d_total, nullptr});
}

void key_bits(Context& c, const uint64_t* keys, uint64_t n, uint64_t& or_all, uint64_t& and_all) {
  unsigned long long* acc = c.s_misc.as<unsigned long long>(4);
  hipLaunchKernelGGL(k_init_bits, dim3(1), dim3(1), 0, c.stream, acc);
  GSJ_LAUNCHED();
  if (n) {
    uint32_t g = (uint32_t)std::min<uint64_t>((n + 255) / 256, 256);
    hipLaunchKernelGGL(k_key_bits, dim3(g), dim3(256), 0, c.stream, keys, n, acc);
    GSJ_LAUNCHED();
  }
  uint64_t* h = c.h_scal.as<uint64_t>(4);
  GSJ_HIP(hipMemcpyAsync(h, acc, 16, hipMemcpyDeviceToHost, c.stream));
  GSJ_HIP(hipStreamSynchronize(c.stream));
  or_all = h[0]; and_all = n ? h[1] : 0;
}

void radix_sort_pairs(Context& c, uint64_t*& keys, uint64_t*& keys_alt, uint32_t*& vals, uint32_t*& vals_alt, uint64_t n, int bit0, int bit1,
                      bool probe) {
  if (n <= 1) return;
  GSJ_REQUIRE(n < (1ull << 32), GSJ_E_LIMIT, "radix sort: more than 2^32 elements");
  uint64_t varying = ~0ull;
  if (probe) {
    uint64_t o, a;
    key_bits(c, keys, n, o, a);
    varying = o ^ a;
  }
  const bool small = n <= RS_SMALL;
  const uint32_t ntiles = (uint32_t)div_up(n, RS_T * (small ? RS_ITEMS_SMALL : RS_ITEMS));
  uint32_t* ghist = c.s_tmp2.as<uint32_t>((size_t)256 * ntiles + 8);
  for (int shift = bit0 & ~7; shift < bit1; shift += 8) {
    if (((varying >> shift) & 255u) == 0) continue;
    hipLaunchKernelGGL(small ? k_rs_hist<RS_ITEMS_SMALL> : k_rs_hist<RS_ITEMS>, dim3(ntiles), dim3(RS_T), 0, c.stream, keys, n, shift, ntiles, ghist);
    GSJ_LAUNCHED();
    scan_loaded<uint32_t>(c, LoadArray<uint32_t>{ghist}, ghist, (uint64_t)256 * ntiles, ScanTotal{});
    hipLaunchKernelGGL(small ? k_rs_scatter<RS_ITEMS_SMALL> : k_rs_scatter<RS_ITEMS>, dim3(ntiles), dim3(RS_T), 0, c.stream, keys, vals, n, shift, ntiles,
                       ghist, keys_alt, vals_alt);
    GSJ_LAUNCHED();
    std::swap(keys, keys_alt);
    std::swap(vals, vals_alt);
  }
}

bool deliver_rows(Context& c, const RowPart* parts, int nparts, uint64_t nrows, double& copy_ms,
                  const std::function<int(uint64_t first, uint64_t n)>& give) {
  const uint64_t nchunks = (nrows + DELIVER_ROWS - 1) / DELIVER_ROWS;
  auto rows_of = [&](uint64_t k) { return std::min(DELIVER_ROWS, nrows - k * DELIVER_ROWS); };
  auto send = [&](uint64_t k) {
    for (int p = 0; p < nparts; p++) {
      const size_t off = k * DELIVER_ROWS * parts[p].bytes;
      GSJ_HIP(hipMemcpyAsync(static_cast<char*>(parts[p].host) + off, static_cast<const char*>(parts[p].dev) + off, rows_of(k) * parts[p].bytes,
                             hipMemcpyDeviceToHost, c.stream));
    }
    GSJ_HIP(hipEventRecord(c.ev[17 + (k & 1)], c.stream));
  };
  WallTimer t0;
  if (nchunks) send(0);
  for (uint64_t k = 0; k < nchunks; k++) {
    WallTimer t;
    if (k + 1 < nchunks) send(k + 1);
    GSJ_HIP(hipEventSynchronize(c.ev[17 + (k & 1)]));
    copy_ms += k ? t.ms() : t0.ms();
    if (give(k * DELIVER_ROWS, rows_of(k))) {
      GSJ_HIP(hipStreamSynchronize(c.stream));
      return true;
    }
  }
  return false;
}

}  // namespace gsj
